// p3_sed.hpp -- cloud, rain and ice sedimentation with the surface precipitation,
// and homogeneous freezing with p3_main_part3.
//
// Work decomposition: one column per group of LPC lanes (LPC = 16, 32 or 64,
// aligned inside the 64-lane wavefront); lane j of a group owns the L
// contiguous levels j*L .. j*L+L-1 of its column and keeps their
// sedimentation state in registers for the whole substep loop.  Everything a
// substep needs from other levels goes through cross-lane operations inside
// the group: the CFL maximum and find_top/find_bottom are butterfly
// reductions, and the upwind flux entering a lane's first level is the last
// level's flux of the lane above (one lane shift).  A column therefore runs
// exactly its own number of substeps, without block barriers, and reads its
// state from HBM once per species.
//
// Follows components/eamxx/src/physics/p3/impl/p3_main_impl.hpp:262-312
// (sedimentation, homogeneous freezing, part 3), with
// p3_cloud_sed_impl.hpp:14-147, p3_rain_sed_impl.hpp:14-170,
// p3_ice_sed_impl.hpp:66-270, p3_upwind_impl.hpp:14-151 and
// p3_main_impl_part3.hpp:18-204.
#pragma once

#include "p3_kernel.hpp"

namespace p3d {

// Reductions over aligned groups of LPC lanes, all lanes getting the result,
// entirely in the VALU.  Step o combines each lane with a lane of the other half
// of its 2o-lane block; before the step both halves are uniform, so any pairing of
// the halves does: inside a 16-lane row by DPP (o = 1, 2: quad permutes; 4, 8: the
// half-row and row mirrors), across rows and across the wavefront's halves by
// v_permlane16_swap and v_permlane32_swap, which leave the two halves' values in
// two registers.  A lane reads only lanes of its own group, and every lane of a
// group must be active: the sedimentation code calls these with whole groups.
// (ds_swizzle and ds_bpermute for the last two steps cost an LDS round trip each,
// which a column on 32 or 64 lanes waits for in every substep.)
struct Halves { int a, b; };
template <int O>
__device__ __forceinline__ Halves halves(int v) {
  if constexpr (O == 1) return {v, __builtin_amdgcn_mov_dpp(v, 0xB1, 0xF, 0xF, true)};       // quad_perm:[1,0,3,2]
  else if constexpr (O == 2) return {v, __builtin_amdgcn_mov_dpp(v, 0x4E, 0xF, 0xF, true)};  // quad_perm:[2,3,0,1]
  else if constexpr (O == 4) return {v, __builtin_amdgcn_mov_dpp(v, 0x141, 0xF, 0xF, true)};  // row_half_mirror
  else if constexpr (O == 8) return {v, __builtin_amdgcn_mov_dpp(v, 0x140, 0xF, 0xF, true)};  // row_mirror
  else if constexpr (O == 16) {
    const auto r = __builtin_amdgcn_permlane16_swap(v, v, false, false);
    return {(int)r[0], (int)r[1]};
  } else {
    const auto r = __builtin_amdgcn_permlane32_swap(v, v, false, false);
    return {(int)r[0], (int)r[1]};
  }
}
template <int O>
__device__ __forceinline__ void halves(double v, double& a, double& b) {
  const Halves hi = halves<O>(__double2hiint(v)), lo = halves<O>(__double2loint(v));
  a = __hiloint2double(hi.a, lo.a);
  b = __hiloint2double(hi.b, lo.b);
}

template <int LPC>
__device__ __forceinline__ int grp_min(int v) {
  if constexpr (LPC > 1) {
    const Halves h = halves<LPC / 2>(grp_min<LPC / 2>(v));
    v = min(h.a, h.b);
  }
  return v;
}
template <int LPC>
__device__ __forceinline__ int grp_max(int v) {
  if constexpr (LPC > 1) {
    const Halves h = halves<LPC / 2>(grp_max<LPC / 2>(v));
    v = max(h.a, h.b);
  }
  return v;
}
// (of values that are not NaN)
template <int LPC>
__device__ __forceinline__ double grp_maxd(double v) {
  if constexpr (LPC > 1) {
    double a, b;
    halves<LPC / 2>(grp_maxd<LPC / 2>(v), a, b);
    v = __builtin_fmax(a, b);
  }
  return v;
}
// (Used where one lane of the group holds the value and the others 0, so the
// order of the additions does not matter.)
template <int LPC>
__device__ __forceinline__ double grp_sumd(double v) {
  if constexpr (LPC > 1) {
    double a, b;
    halves<LPC / 2>(grp_sumd<LPC / 2>(v), a, b);
    v = a + b;
  }
  return v;
}
// v of the lane below in the group, 0 in the group's first lane: a DPP shift of
// the row (16 lanes) or of the wavefront.
template <int LPC>
__device__ __forceinline__ double grp_below(double v, int j) {
  constexpr int ctrl = LPC == 16 ? 0x111 : 0x138;  // row_shr:1, wave_shr:1
  const int hi = __builtin_amdgcn_mov_dpp(__double2hiint(v), ctrl, 0xF, 0xF, true);
  const int lo = __builtin_amdgcn_mov_dpp(__double2loint(v), ctrl, 0xF, 0xF, true);
  const double w = __hiloint2double(hi, lo);
  return LPC == 32 && j == 0 ? 0.0 : w;
}

// Sedimentation runs as two kernels, or two halves of one launch, over the same
// column blocks, one per species group: the liquid group (cloud, then rain, with the rain flux and
// the liquid surface precipitation) and the ice group.  The groups touch
// disjoint state fields, so their order does not change a bit; apart, each
// block holds only its own group's field pointers.

// Wavefronts per SIMD the sedimentation kernels are compiled for: up to 5
// levels per lane two fit (256 registers); the FP64 ice group at up to 3
// levels per lane runs at three (167 registers at 3 levels, 138 at 2; at three:
// 736 -> 714 us at 21600 x 72).
template <class R, int G, int L> constexpr int sed_waves_per_simd() {
  return (G == SED_ICE && sizeof(R) == 8 && L <= 3) ? 3 : (L <= 5 ? 2 : 1);
}

// The ice group interpolates its 4 table quantities from an LDS copy of the
// ice-sedimentation records.  Where the blocks the kernel's occupancy puts on
// one CU (blocks of 4 wavefronts) can each hold it in the CU's 160 KB of LDS,
// the copy is of the records that also carry each quantity's difference to
// the next size cell (80 KB in FP64, 32 KB in FP32), which saves the four
// size-direction subtractions per quantity; elsewhere (the FP64 kernels at
// three wavefronts per SIMD) it is of the plain records (48 KB).
constexpr int kIceCells = densize * rimsize * isize;
template <class R, int L> constexpr bool ice_rec_dif() {
  return sed_waves_per_simd<R, SED_ICE, L>() * kIceCells * (sizeof(R) == 8 ? 10 : 8) * (int)sizeof(R) <= 160 * 1024;
}
// Values per cell in LDS.  All lanes read the same 16-byte part of their cells'
// records at a time, so the records' stride decides which of the 16 bank groups
// (16 bytes each) a read can fall on: FP64 records of 64 bytes would use 4 of them
// and those of 32 bytes 8; one part more per record uses all 16 (before, conflicts
// held the LDS 27 % of the kernel's time at 21600 x 72 FP64: sedimentation and part
// 3 635 -> 608 us).  The mixed form's 32-byte records stay: a longer stride would
// cost the fourth block per CU.
template <class R, int L> constexpr int ice_rec_len() { return ice_rec_dif<R, L>() ? 8 : 4; }
template <class R, int L> constexpr int ice_lds_stride() { return ice_rec_len<R, L>() + (sizeof(R) == 8 ? 2 : 0); }
template <class R, int L> constexpr int ice_lds_len() { return kIceCells * ice_lds_stride<R, L>(); }

// An in-cloud value q / cf after the first substep.  In FP64 the reciprocal is formed
// once per level and run (cf does not change over the substeps): five instructions
// instead of a division's thirteen issue slots, for up to four fields per level and
// substep.  So that any cf divides as it should, den is cf times 2^up, up > 0 where cf
// is tiny, and the quotient is scaled back, exactly or to infinity.  (Without the last
// step sedimentation and part 3 take 92.5 us at 2700 x 72 and 266 at 16384 x 128, with it
// 93.3 and 270; with a uniform branch to general divisions instead 95.5 and 270.  A
// second substep loop for such runs spilled: 130 us at 2700 x 72.)
constexpr double kTinyFrac = 0x1p-900;
struct Frac {
  double den, rden;  // rden: p3m_recip(den)
  int up;
  __device__ __forceinline__ void set(double cf) {
    up = m_fabs(cf) < kTinyFrac ? 300 : 0;
    den = __builtin_amdgcn_ldexp(cf, up);
    rden = p3m_recip(den);
  }
};
__device__ __forceinline__ double incloud_div(double q, double, const Frac& f) {
  return __builtin_amdgcn_ldexp(p3m_div_y(q, f.den, f.rden), f.up);
}
__device__ __forceinline__ float incloud_div(float q, float cf, const Frac&) { return q / cf; }

// Per-lane geometry of the owned levels.
template <int L>
struct Geo {
  double rho[L], inv_rho[L], inv_dz[L];
};

// One species' sedimentation over the group's column (SP = 0 cloud, 1 rain,
// 2 ice), with lane j of the group owning the L levels k_top + j*L ..
// k_top + j*L + L-1 from the species' top level k_top down: sedimentation only
// moves mass down, so the levels above k_top take no part, and spreading only
// [k_top, nlev) over the lanes keeps them busy (rain, below the freezing
// level, fills a quarter of a column).  The state of one column's run, held
// in registers: load() reads the species' fields in that mapping, substep()
// is one CFL substep, store() writes the fields back (the rain run also
// stores the rain flux at the interface below each owned level).  Every lane
// of the group calls each of them together (the CFL maximum, find_bottom and
// the upwind flux are cross-lane operations inside the group).  DIF: the ice
// records in ice_tab carry their size-direction differences (the layout the
// kernel staged, chosen by its own levels per lane, not by this run's L).
template <int SP, class R, int LPC, int L, bool DIF, int STRIDE>
struct SedRun {
  static constexpr int NF = SP == 2 ? 4 : 2;  // fields held (cloud always holds nc: its DSD rewrites it)
  Geo<L> g;
  double q[NF][L], cf[L], coef[L], cfl_ice[L], pflux[L];
  Frac frac[L];  // FP64
  int kbase, k_top, k_bot;
  double dt_left, prt_accum;  // prt_accum: mass through the surface, on the lane owning the lowest level
  int nsub;

  __device__ __forceinline__ static void fields(const KParams& p, double* (&fld)[NF]) {
    if constexpr (SP == 0) { fld[0] = p.qc; fld[1] = p.nc; }
    if constexpr (SP == 1) { fld[0] = p.qr; fld[1] = p.nr; }
    if constexpr (SP == 2) { fld[0] = p.qi; fld[1] = p.ni; fld[2] = p.qm; fld[3] = p.bm; }
  }

  __device__ __forceinline__ void load(const KParams& p, int i, int j, int top) {
    const int nlev = p.nlev;
    double* fld[NF];
    fields(p, fld);
    const double* cfp = SP == 0 ? p.cld_frac_l : (SP == 1 ? p.cld_frac_r : p.cld_frac_i);
    const int coef_f = SP == 0 ? SC_ACN : (SP == 1 ? SC_RHOFACR : SC_RHOFACI);
    k_top = top;
    kbase = k_top + j * L;
    int my_bot = -1;
#pragma unroll
    for (int t = 0; t < L; ++t) {
      const int k = kbase + t;
      const bool ok = k < nlev;
      const size_t x = p.at(i, ok ? k : 0);
      const double dz = ok ? p.dz[x] : 1.0;
      const double dp = ok ? p.dpres[x] : 1.0;
      g.rho[t] = air_density(dp, dz);
      g.inv_rho[t] = p3m_div_inf(1.0, g.rho[t]);
      g.inv_dz[t] = p3m_div_inf(1.0, dz);
#pragma unroll
      for (int f = 0; f < NF; ++f) q[f][t] = ok ? fld[f][x] : 0.0;
      cf[t] = ok ? cfp[x] : 1.0;
      if (sizeof(R) == 8) frac[t].set(cf[t]);
      coef[t] = ok ? p.sc(coef_f, i, ok ? k : 0) : 0.0;
      cfl_ice[t] = (SP == 2 && ok) ? p.cld_frac_l[x] : 1.0;
      pflux[t] = 0;
      // find_bottom, P3I/p3_find_impl.hpp:52-92 (find_top gave k_top)
      if (ok && q[0][t] >= QSMALL) my_bot = k;
    }
    k_bot = grp_max<LPC>(my_bot);
    dt_left = p.dt;
    prt_accum = 0;
    nsub = 0;
  }

  // One substep.  FIRST: the first one, which limits the in-cloud mixing ratios (a
  // template parameter, so that neither kind carries the other's branches) but not the
  // numbers, so that its quotients may overflow.
  template <bool FIRST>
  __device__ __forceinline__ void substep(const KParams& p, int j, const R* __restrict__ ice_tab) {
    constexpr bool first = FIRST;
    constexpr Div D = FIRST ? DIV_INF : DIV;
    const int nlev = p.nlev, kbot = nlev - 1;
    const Runtime& rt = p.rt;
    const int nfield = SP == 2 ? 4 : (SP == 1 ? 2 : (p.predictNc ? 2 : 1));
    double V1[L], V2[L];
    double co = 0;
#pragma unroll
    for (int t = 0; t < L; ++t) {
      const int k = kbase + t;
      V1[t] = 0;
      V2[t] = 0;
      if (k >= k_top && k <= k_bot) {  // k_bot < nlev, so k is a real level
        const double rho = g.rho[t];
        if constexpr (SP == 0) {
          // cloud_sedimentation, P3I/p3_cloud_sed_impl.hpp:85-112
          // in-cloud values in the arithmetic type of the form (the state stays FP64)
          const R cfl = R(cf[t]);
          const R qc = R(q[0][t]), nc = R(q[1][t]);
          R qc_incld, nc_incld;
          if (first) {
            const R icfl = m_div<D>(R(1), cfl);
            if (q[0][t] >= QSMALL) { qc_incld = vmin(qc * icfl, R(incloud_limit)); nc_incld = vmax(nc * icfl, R(0)); }
            else { qc_incld = 0; nc_incld = 0; }
          } else {
            qc_incld = incloud_div(qc, cfl, frac[t]);
            nc_incld = incloud_div(nc, cfl, frac[t]);
          }
          if (qc_incld > R(QSMALL)) {
            R ncr = nc_incld, mu_c, lamc;
            get_cloud_dsd2<R, D>(qc_incld, ncr, mu_c, R(rho), lamc);
            q[1][t] = double(ncr) * cf[t];
            const R dum = m_div(R(1), m_pow(lamc, R(bcn)));
            const R acn = R(coef[t]);
            V1[t] = double(m_div(acn * m_tgamma(R(4 + bcn) + mu_c) * dum, m_tgamma(mu_c + R(4))));
            if (p.predictNc) V2[t] = double(m_div(acn * m_tgamma(R(1 + bcn) + mu_c) * dum, m_tgamma(mu_c + R(1))));
          }
        } else if constexpr (SP == 1) {
          // rain_sedimentation + compute_rain_fall_velocity, P3I/p3_rain_sed_impl.hpp:14-34,104-126
          const R cfr = R(cf[t]);
          const R qr = R(q[0][t]), nr = R(q[1][t]);
          R qr_incld, nr_incld;
          if (first) {
            const R icfr = m_div<D>(R(1), cfr);
            if (q[0][t] >= QSMALL) { qr_incld = vmin(qr * icfr, R(precip_limit)); nr_incld = vmax(nr * icfr, R(0)); }
            else { qr_incld = 0; nr_incld = 0; }
          } else {
            qr_incld = incloud_div(qr, cfr, frac[t]);
            nr_incld = incloud_div(nr, cfr, frac[t]);
          }
          if (qr_incld > R(QSMALL)) {
            R nrr = nr_incld, mu_r = 0, lamr;
            get_rain_dsd2<R, D>(rt, qr_incld, nrr, mu_r, lamr);
            const Tab3<R> t3 = lookup3<R>(mu_r, lamr);
            const R rhofacr = R(coef[t]);
            R v[2];  // vm, vn
            apply_table3_v<R>(TabOf<R>::get(p.tab).rain_v, t3, v);
            V1[t] = double(v[0] * rhofacr);
            V2[t] = double(v[1] * rhofacr);
            q[1][t] = double(nrr) * cf[t];
          }
        } else {
          // ice_sedimentation, P3I/p3_ice_sed_impl.hpp:134-166
          const R cfi = R(cf[t]);
          const R qi = R(q[0][t]), ni = R(q[1][t]), qm = R(q[2][t]), bm = R(q[3][t]);
          R qi_incld, ni_incld, qm_incld, bm_incld;
          if (first) {
            const R icfi = m_div<D>(R(1), cfi), icfl = m_div<D>(R(1), R(cfl_ice[t]));
            if (q[0][t] >= QSMALL) { qi_incld = vmin(qi * icfi, R(incloud_limit)); ni_incld = vmax(ni * icfi, R(0)); }
            else { qi_incld = 0; ni_incld = 0; }
            if (q[0][t] >= QSMALL && q[2][t] >= QSMALL) { qm_incld = qm * icfi; bm_incld = vmin(vmax(bm * icfl, R(0)), R(incloud_limit)); }
            else { qm_incld = 0; bm_incld = 0; }
          } else {
            qi_incld = incloud_div(qi, cfi, frac[t]);
            ni_incld = incloud_div(ni, cfi, frac[t]);
            qm_incld = incloud_div(qm, cfi, frac[t]);
            bm_incld = incloud_div(bm, cfi, frac[t]);
          }
          if (qi_incld > R(QSMALL)) {
            R nir = vmax(ni_incld, R(NSMALL));
            R qmr = qm_incld, bmr = bm_incld;
            const R qir = qi_incld;
            const R rhop = calc_bulk_rho_rime<R, D>(rt, qir, qmr, bmr);
            q[2][t] = double(qmr) * cf[t];
            q[3][t] = double(bmr) * cf[t];
            const TabIce<R> ti = lookup_ice<R, D>(qir, nir, qmr, rhop);
            // quantities 0, 1, 6, 7 of the records (in FP64 as two halves, which bounds the registers)
            R v[4];
            if constexpr (sizeof(R) == 4) {
              if constexpr (DIF) apply_table_ice_dif<4, STRIDE, 4, R>(ice_tab, ti, v, 0);
              else apply_table_ice_rec<4, STRIDE, R>(ice_tab, ti, v, 0);
            } else {
              R a[2], b[2];
              if constexpr (DIF) {
                apply_table_ice_dif<2, STRIDE, 4, R>(ice_tab, ti, a, 0);
                apply_table_ice_dif<2, STRIDE, 4, R>(ice_tab, ti, b, 2);
              } else {
                apply_table_ice_rec<2, STRIDE, R>(ice_tab, ti, a, 0);
                apply_table_ice_rec<2, STRIDE, R>(ice_tab, ti, b, 2);
              }
              v[0] = a[0]; v[1] = a[1]; v[2] = b[0]; v[3] = b[1];
            }
            const R t_ni_fall = v[0], t_qi_fall = v[1], t_lammax = v[2], t_lammin = v[3];
            nir = vmin(nir, t_lammax * nir);
            nir = vmax(nir, t_lammin * nir);
            q[1][t] = double(nir) * cf[t];
            const R rhofaci = R(coef[t]);
            V1[t] = double(R(rt.ice_sedimentation_factor) * t_qi_fall * rhofaci);
            V2[t] = double(R(rt.ice_sedimentation_factor) * t_ni_fall * rhofaci);
          }
        }
        const double Co = V1[t] * dt_left * g.inv_dz[t];
        if (Co > co) co = Co;
      }
    }
    const double Co_max = grp_maxd<LPC>(co);

    // generalized_sedimentation + calc_first_order_upwind_step, P3I/p3_upwind_impl.hpp:14-129
    const int tmpint1 = (int)(Co_max + 1);
    const double dt_sub = p3m_div(dt_left, (double)tmpint1);
    const int k_temp = (k_bot == kbot) ? k_bot : k_bot + 1;
    // fluxes F = V r rho.  Only the levels in [k_top, k_temp] update, and
    // they read F of their own level and of the level above, which is in
    // that range too (or is k_top's upper boundary, flux 0): F elsewhere is
    // never read, so it is not masked.
    double F[NF][L];
#pragma unroll
    for (int t = 0; t < L; ++t) {
#pragma unroll
      for (int f = 0; f < NF; ++f) {
        const double V = (SP == 2) ? (f == 1 ? V2[t] : V1[t]) : (f == 0 ? V1[t] : V2[t]);
        F[f][t] = V * q[f][t] * g.rho[t];
      }
    }
    // flux out of the last level of the lane above (lane 0's first level is
    // k_top, whose incoming flux is 0)
    double Fin[NF];
#pragma unroll
    for (int f = 0; f < NF; ++f) Fin[f] = grp_below<LPC>(F[f][L - 1], j);
#pragma unroll
    for (int t = 0; t < L; ++t) {
      const int k = kbase + t;
      if (k >= k_top && k <= k_temp) {
#pragma unroll
        for (int f = 0; f < NF; ++f) {
          if (f < nfield) {
            const double Fa = t == 0 ? Fin[f] : F[f][t > 0 ? t - 1 : 0];
            const double fluxdiv = (Fa - F[f][t]) * g.inv_dz[t];
            q[f][t] = q[f][t] + fluxdiv * dt_sub * g.inv_rho[t];
          }
        }
        if (SP == 1) pflux[t] += F[0][t];  // rain_sed :140-153, interface k+1
        if (k == kbot && k_bot == kbot) prt_accum += F[0][t] * dt_sub;
      }
    }
    if (k_bot != kbot) k_bot += 1;
    dt_left -= dt_sub;
    nsub++;
  }

  // The substeps changed levels k_top .. k_bot only (k_bot has moved down one
  // level after each substep, past the last one's lowest updated level): the
  // levels below keep their loaded values and are not stored again.
  __device__ __forceinline__ void store(const KParams& p, int i) const {
    const int nlev = p.nlev;
    double* fld[NF];
    fields(p, fld);
#pragma unroll
    for (int t = 0; t < L; ++t) {
      const int k = kbase + t;
      if (k < nlev) {
        const size_t x = p.at(i, k);
        if (k <= k_bot) {
          // an empty level is empty in every field (part 3 would zero the others):
          // part 3 then need not read them
          const bool empty = q[0][t] == 0;
#pragma unroll
          for (int f = 0; f < NF; ++f) fld[f][x] = empty ? q[0][t] : q[f][t];
        }
        if (SP == 1) p.precip_liq_flux[p.atf(i, k + 1)] = pflux[t];  // rain_sed :140-153, interface k+1
      }
    }
  }
};

// One species' run over the group's column, whole: load, the substeps (the
// first peeled off the loop, so that neither carries the other's branch),
// store.  prt (every lane) is the mass that left through the surface.
template <int SP, class R, int LPC, int L, bool DIF, int STRIDE>
__device__ __forceinline__ void sediment_run(const KParams& p, int i, int j, int k_top, double& prt,
                                          int& nsub_out, unsigned& err, const R* __restrict__ ice_tab) {
  SedRun<SP, R, LPC, L, DIF, STRIDE> r;
  r.load(p, i, j, k_top);
  if (r.dt_left > dt_left_tol) r.template substep<true>(p, j, ice_tab);
#pragma unroll 1
  while (r.dt_left > dt_left_tol) {
    // The substep count is bounded by the CFL number (a few hundred at most for
    // physical inputs); the cap only guarantees termination for corrupt inputs.
    if (r.nsub >= kMaxSubsteps) { err |= ERR_SUBSTEP_LIMIT; break; }
    r.template substep<false>(p, j, ice_tab);
  }
  r.store(p, i);
  prt = grp_sumd<LPC>(r.prt_accum);  // only the lane owning kbot accumulated
  nsub_out = r.nsub;
}

// find_top (P3I/p3_find_impl.hpp:14-50) of NS species (mixing ratios f[s]) over
// the group's column in the standard mapping (lane j: levels j*L .. j*L+L-1),
// all loads in one pass; top[s] = nlev when species s is absent (or the column
// does not run).  For columns that p3_order_kernel has not listed.
template <int LPC, int L, int NS>
__device__ __forceinline__ void find_tops(const KParams& p, int i, int j, bool run,
                                          const double* const (&f)[NS], int (&top)[NS]) {
  const int nlev = p.nlev;
  int my[NS];
#pragma unroll
  for (int sp = 0; sp < NS; ++sp) my[sp] = nlev;
  if (run) {
    double q[NS][L];
#pragma unroll
    for (int t = 0; t < L; ++t) {
      const int k = j * L + t;
      const size_t x = p.at(i, k < nlev ? k : 0);
#pragma unroll
      for (int sp = 0; sp < NS; ++sp) q[sp][t] = f[sp][x];
    }
#pragma unroll
    for (int t = L - 1; t >= 0; --t) {
      const int k = j * L + t;
#pragma unroll
      for (int sp = 0; sp < NS; ++sp)
        if (k < nlev && q[sp][t] >= QSMALL) my[sp] = k;
    }
  }
#pragma unroll
  for (int sp = 0; sp < NS; ++sp) top[sp] = grp_min<LPC>(my[sp]);
}

// One species' substeps on the fewest levels per lane that cover [k_top, nlev).
// Every lane of the wavefront calls this (k_top = nlev for a lane whose column
// does not run or has none of the species).
template <int SP, class R, int LPC, int L>
__device__ __forceinline__ void sediment(const KParams& p, int i, int j, int k_top, double& prt, int& nsub_out,
                                         unsigned& err, const R* __restrict__ ice_tab = nullptr) {
  const int nlev = p.nlev;
  prt = 0;
  nsub_out = 0;
  // levels per lane for [k_top, nlev), the largest over the wavefront's
  // columns (all its lanes are here), so that the wavefront takes one path
  int lw = k_top < nlev ? (nlev - k_top + LPC - 1) / LPC : 0;
#pragma unroll
  for (int o = 32; o >= LPC; o >>= 1) lw = max(lw, __shfl_xor(lw, o, 64));
  if (k_top >= nlev) return;
  // the ice records' layout is the one the kernel staged for its own L
  constexpr bool dif = ice_rec_dif<R, L>();
  constexpr int str = ice_lds_stride<R, L>();
  if (lw <= 1) sediment_run<SP, R, LPC, 1, dif, str>(p, i, j, k_top, prt, nsub_out, err, ice_tab);
  else if (L > 2 && lw <= 2) sediment_run<SP, R, LPC, (L > 2 ? 2 : L), dif, str>(p, i, j, k_top, prt, nsub_out, err, ice_tab);
  else sediment_run<SP, R, LPC, L, dif, str>(p, i, j, k_top, prt, nsub_out, err, ice_tab);
}

// homogeneous_freezing (P3I/p3_ice_sed_impl.hpp:207-270) + p3_main_part3
// (P3I/p3_main_impl_part3.hpp:60-199, only the fields p3_main outputs) for
// level k of column i, after sedimentation.
template <class R>
__device__ __forceinline__ void part3_level(const KParams& p, int k, int i, bool active, unsigned& err) {
  const int nlev = p.nlev;
  const size_t x = p.at(i, k);
  const double latvap = LatVap, latice = LatIce, inv_cp = INV_CP;
  const Runtime& rt = p.rt;
  p.precip_ice_flux[p.atf(i, k)] = 0;
  if (k == nlev - 1) p.precip_ice_flux[p.atf(i, nlev)] = 0;
  double reff_c = 10.e-6, reff_i = 25.e-6, reff_r = 500.e-6, rho_qi = 0;
  double qc = 0, nc = 0, qr = 0, nr = 0, qi = 0, ni = 0, qm = 0, bm = 0, qv = 0, th = 0;
  // The kernel runs at the HBM rate, so a point reads what it needs: an absent
  // species' other fields are zero (parts 1 and 2 and sedimentation leave them so),
  // and th, qv and the liquid exchange change only where a remainder below QSMALL
  // is given back to the vapour or liquid freezes.
  const bool all = p.amble.on || p.dbg_check;
  double T_part1 = 0, inv_exner = 0, vap_liq = 0, dp = 0, dz = 0, cfl = 0, cfr = 0, cfi = 0;
  bool thermo = false;  // th, qv, inv_exner are loaded
  auto load_thermo = [&] {
    thermo = true;
    qv = p.qv[x]; th = p.th[x];
    inv_exner = p.inv_exner[x];
  };
  bool gives = false;  // cloud or rain gives back a remainder
  if (active || p.amble.on) {
    qc = p.qc[x]; qr = p.qr[x]; qi = p.qi[x];
    const bool cloud = qc >= QSMALL, rain = qr >= QSMALL;
    gives = (qc != 0 && !cloud) || (qr != 0 && !rain);
    if (all || qc != 0) nc = p.nc[x];
    if (all || qr != 0) nr = p.nr[x];
    if (all || qi != 0) { ni = p.ni[x]; qm = p.qm[x]; bm = p.bm[x]; }
    if (all || gives || (qi != 0 && !(qi >= QSMALL))) load_thermo();
    if (cloud || rain) T_part1 = p.sc(SC_T, i, k);
    if (cloud) cfl = p.cld_frac_l[x];
    if (rain) cfr = p.cld_frac_r[x];
    if (cloud || rain || qi >= QSMALL) { dp = p.dpres[x]; dz = p.dz[x]; cfi = p.cld_frac_i[x]; }
    if (gives) vap_liq = p.vap_liq_exchange[x];
  }
  // the state as it is in memory: without the post-amble, a field that part 3
  // leaves bit for bit unchanged is not stored again
  const double in[10] = {qc, nc, qr, nr, qi, ni, qm, bm, qv, th};
  if (active) {
    if (rt.do_ice_production) {
      const bool t_lt = T_part1 < T_homogfrz;  // (0 where there is no liquid)
      const bool qc_ge = t_lt && qc >= QSMALL;
      const bool qr_ge = t_lt && qr >= QSMALL;
      if ((qc_ge || qr_ge) && !thermo) load_thermo();
      const double Qc_nuc = qc, Qr_nuc = qr;
      const double Nc_nuc = vmax(nc, NSMALL), Nr_nuc = vmax(nr, NSMALL);
      if (qc_ge) {
        qm = qm + Qc_nuc; qi = qi + Qc_nuc; bm = bm + Qc_nuc * INV_RHO_RIMEMAX; ni = ni + Nc_nuc;
        th = th + inv_exner * Qc_nuc * latice * inv_cp;
      }
      if (qr_ge) {
        qm = qm + Qr_nuc; qi = qi + Qr_nuc; bm = bm + Qr_nuc * INV_RHO_RIMEMAX; ni = ni + Nr_nuc;
        th = th + inv_exner * Qr_nuc * latice * inv_cp;
      }
      if (qc_ge) { qc = 0; nc = 0; }
      if (qr_ge) { qr = 0; nr = 0; }
    }
    // p3_main_part3, P3I/p3_main_impl_part3.hpp:60-199 (only the fields p3_main outputs)
    const double rho = air_density(dp, dz);
    // cloud
    if (qc >= QSMALL) {
      R ncr = R(p3m_div_any(nc, cfl)), mu_c, lamc;
      get_cloud_dsd2<R>(R(p3m_div_any(qc, cfl)), ncr, mu_c, R(rho), lamc);
      nc = double(ncr) * cfl;
      reff_c = double(m_div<DIV_INF>(R(0.5) * (mu_c + R(3)), lamc));
    } else {
      qv = qv + qc;
      th = th - inv_exner * qc * latvap * inv_cp;
      vap_liq = vap_liq - qc;
      qc = 0; nc = 0;
    }
    // rain
    if (qr >= QSMALL) {
      R nrr = R(p3m_div_any(nr, cfr)), mu_r = 0, lamr;
      get_rain_dsd2<R>(rt, R(p3m_div_any(qr, cfr)), nrr, mu_r, lamr);
      nr = double(nrr) * cfr;
      reff_r = double(m_div(R(1.5), lamr));
    } else {
      qv = qv + qr;
      th = th - inv_exner * qr * latvap * inv_cp;
      vap_liq = vap_liq - qr;
      qr = 0; nr = 0;
    }
    // ice
    if (qi >= QSMALL) {
      const double inv_rho = p3m_div_inf(1.0, rho);
      ni = vmax(ni, NSMALL);
      const double qi_incld = p3m_div_any(qi, cfi);
      double ni_incld = p3m_div_any(ni, cfi);
      double qm_incld = p3m_div_any(qm, cfi), bm_incld = p3m_div_any(bm, cfi);
      R qmr = R(qm_incld), bmr = R(bm_incld);
      const R rhop = calc_bulk_rho_rime<R>(rt, R(qi_incld), qmr, bmr);
      qm_incld = double(qmr); bm_incld = double(bmr);
      qm = qm_incld * cfi;
      bm = bm_incld * cfi;
      impose_max_total_ni<double>(ni_incld, rt.max_total_ni, inv_rho);
      const TabIce<R> ti = lookup_ice<R, DIV_INF, false>(R(qi_incld), R(ni_incld), R(qm_incld), rhop);
      if (p.dbg_ice_idx) p.dbg_ice_idx[x] = ti.dumjj * 10000 + ti.dumii * 100 + ti.dumi;
      R v[4];  // quantities 5, 6, 7, 11
      apply_table_ice_rec<4, 4, R>(TabOf<R>::get(p.tab).ice_p3, ti, v);
      const R t_eff = v[0], t_lammax = v[1], t_lammin = v[2], t_rhomm = v[3];
      ni_incld = vmin(ni_incld, double(t_lammax) * ni_incld);
      ni_incld = vmax(ni_incld, double(t_lammin) * ni_incld);
      reff_i = double(t_eff);
      rho_qi = double(t_rhomm);
      ni = ni_incld * cfi;
      if (qm < QSMALL) { qm = 0; bm = 0; }
    } else {
      if (p.dbg_ice_idx) p.dbg_ice_idx[x] = -1;
      qv = qv + qi;
      th = th - inv_exner * qi * (latvap + latice) * inv_cp;
      qi = 0; ni = 0; qm = 0; bm = 0;
    }
    if (qr < QSMALL) nr = 0;
    if (gives) p.vap_liq_exchange[x] = vap_liq;
    if (p.dbg_check) {
      // check_values (P3I/p3_check_values_impl.hpp:25-79, called after part 3 at
      // P3I/p3_main_impl.hpp:316-324 in debug builds) on T = th exner and qv: T outside
      // (173, 323) K is the trap (ERR_CHECK_VALUES), qv outside (0, 40e-3) only a flag
      const double T = th * (1 / inv_exner);
      const int f = (!(T > 173. && T < 323.) ? 1 : 0) | (!(qv > 0. && qv < 40.e-3) ? 2 : 0);
      if (f) atomicOr(&p.dbg_check[i], f);
      if (f & 1) err |= ERR_CHECK_VALUES;
    }
  } else if (p.dbg_ice_idx) {
    p.dbg_ice_idx[x] = -1;
  }
  if (p.amble.on) {
    // p3_postamble, eamxx_p3_process_interface.hpp:200-241: the temperature change
    // rescaled by dp_dry/dp, dry -> wet mixing ratios, radii in microns
    const Amble& a = p.amble;
    const double dp = a.dp_wet[x], dp_dry = p.dpres[x];
    const double T_before = a.T_mid[x];
    const Ratio wet(dp_dry, dp);
    auto to_wet = [&](double q) { return wet.of(q); };
    double T = to_wet(th * exner_function(a.p_mid[x]) - T_before);
    T += T_before;
    a.T_mid[x] = T;
    a.T_prev[x] = T;
    qv = to_wet(qv);
    p.qc[x] = to_wet(qc); p.nc[x] = to_wet(nc); p.qr[x] = to_wet(qr);
    p.nr[x] = to_wet(nr); p.qi[x] = to_wet(qi); p.ni[x] = to_wet(ni);
    p.qm[x] = to_wet(qm); p.bm[x] = to_wet(bm); p.qv[x] = qv;
    a.qv_prev[x] = qv;
    reff_c *= 1e6;
    reff_i *= 1e6;
    reff_r *= 1e6;
  } else if (active) {
    double* const f[10] = {p.qc, p.nc, p.qr, p.nr, p.qi, p.ni, p.qm, p.bm, p.qv, p.th};
    const double out[10] = {qc, nc, qr, nr, qi, ni, qm, bm, qv, th};
#pragma unroll
    for (int q = 0; q < 10; ++q)
      if (__double_as_longlong(out[q]) != __double_as_longlong(in[q])) f[q][x] = out[q];
  }
  p.diag_eff_radius_qc[x] = reff_c;
  p.diag_eff_radius_qi[x] = reff_i;
  p.diag_eff_radius_qr[x] = reff_r;
  p.rho_qi[x] = rho_qi;
}

// The ice group's per-column outputs once column i's run has ended (any one
// lane of the group writes them): the surface precipitation, its post-amble
// accumulation (eamxx_p3_process_interface.hpp:245-258) and the substep count.
__device__ __forceinline__ void ice_column_out(const KParams& p, int i, bool ran, double prt, int nsub) {
  double ice = 0;
  if (ran) ice += prt * INV_RHO_H2O * (1 / p.dt);
  p.precip_ice_surf[i] = ice;
  if (p.amble.on) p.amble.precip_ice_mass[i] += ice * RHO_H2O * p.dt;
  if (p.dbg_substeps) p.dbg_substeps[(size_t)2 * p.dbg_stride + i] = nsub;
}

// One wavefront's work for group G: the 64/LPC columns starting at column
// col0, with LPC lanes per column.
template <class R, int LPC, int L, int G, class Stage>
__device__ __forceinline__ void sed_wave(const KParams& p, int col0, const R* __restrict__ ice_tab, Stage&& staged) {
  static_assert(64 % LPC == 0, "a column group must divide the wavefront");
  const int lane = threadIdx.x & 63;
  const int j = lane % LPC;
  // the column, in p3_order_kernel's order with its top levels; a position past the
  // end is no column
  int i = col0 + lane / LPC;
  const bool ordered = LPC < 64 && p.ordered();
  uint2 entry = make_uint2((unsigned)i, (unsigned)p.nlev << 16 | (unsigned)p.nlev);
  if (ordered && i < p.ncol) entry = p.order(G)[i];
  i = (int)entry.x;
  const int nlev = p.nlev, kbot = nlev - 1;
  const int kbase = j * L;
  unsigned err = 0;

  // Every lane of the wavefront takes part in sediment() (its wavefront-wide
  // choice of levels per lane); columns past ncol or without a full step only
  // skip the arithmetic.
  const bool live = i < p.ncol;
  // (a column that the reference skips has none of the species: without the
  // status words each species' own top level decides)
  const bool track = p.track();
  const int status = live && track ? p.colstat[i] : 0;
  const bool run = live && (!track || status == kStatusFull);
  const double inv_dt = 1 / p.dt;
  if constexpr (G == SED_LIQ) {
    double prt_c, prt_r;
    int ns_c, ns_r, top[2];
    if (ordered) top[0] = (int)(entry.y & 0xffff), top[1] = (int)(entry.y >> 16);
    else find_tops<LPC, L, 2>(p, i, j, run, {p.qc, p.qr}, top);
    const int top_c = top[0], top_r = top[1];
    sediment<0, R, LPC, L>(p, i, j, top_c, prt_c, ns_c, err);
    sediment<1, R, LPC, L>(p, i, j, top_r, prt_r, ns_r, err);
    if (live) {
#pragma unroll
      for (int t = 0; t < L; ++t) {
        const int k = kbase + t;
        if (k >= nlev) continue;
        // no rain flux above the rain's top level (the rain run stored the rest)
        if (k < top_r) p.precip_liq_flux[p.atf(i, k + 1)] = 0;
        if (k == kbot) {
          double liq = 0;
          if (top_c < nlev) liq = prt_c * INV_RHO_H2O * inv_dt;
          if (top_r < nlev) liq += prt_r * INV_RHO_H2O * inv_dt;
          p.precip_liq_surf[i] = liq;
          // the per-column post-amble, eamxx_p3_process_interface.hpp:245-258 (the
          // boundary fluxes, which need both groups, are written by part 3)
          if (p.amble.on) p.amble.precip_liq_mass[i] += liq * RHO_H2O * p.dt;
        }
      }
      if (j == 0) {
        p.precip_liq_flux[p.atf(i, 0)] = 0;  // the top interface
        // 0 skipped after part 1, 1 skipped after part 2, 2 full step
        if (p.dbg_status) p.dbg_status[i] = status == kStatusFull ? 2 : status;
        if (p.dbg_substeps) {
          p.dbg_substeps[i] = ns_c;
          p.dbg_substeps[(size_t)p.dbg_stride + i] = ns_r;
        }
      }
    }
  } else {
    double prt_i;
    int ns_i, top[1];
    if (ordered) top[0] = (int)(entry.y & 0xffff);
    else find_tops<LPC, L, 1>(p, i, j, run, {p.qi}, top);
    staged();
    const int top_i = top[0];
    sediment<2, R, LPC, L>(p, i, j, top_i, prt_i, ns_i, err, ice_tab);
    if (live && j == 0) ice_column_out(p, i, top_i < nlev, prt_i, ns_i);
  }
  if (err) report_errors(p.err, err);
}

// One block's work for group G: WPB wavefronts of 64/LPC columns each, the
// CB = WPB * 64/LPC columns starting at column bid * CB of the column set p,
// with LPC lanes per column (part 3 follows in p3_part3_lvl_kernel).
// `staged` is called by every wavefront once, when its columns' top levels are
// known and before the ice table is read.
template <class R, int LPC, int L, int WPB, int G, class Stage>
__device__ __forceinline__ void sed_block(const KParams& p, int bid, const R* __restrict__ ice_tab, Stage&& staged) {
  constexpr int CPW = 64 / LPC;  // columns per wavefront
  constexpr int CB = WPB * CPW;  // columns per block
  static_assert((CB & (CB - 1)) == 0, "columns per block must be a power of two");
  const int wave = threadIdx.x >> 6;
  sed_wave<R, LPC, L, G>(p, bid * CB + wave * CPW, ice_tab, staged);
}

// Part 3 as a kernel of its own, one thread per (level, column) on the
// pointwise tiles, after the sedimentation kernel.
//
// Bound by HBM.  Reading all 18 fields at every point it took 70 us at 21600 x 72
// FP64 and 82 us at 16384 x 128 mixed (4.4 TB/s); reading what a point needs
// (part3_level), 54 and 62 us, and with registers for four wavefronts per SIMD
// (128 VGPRs instead of 134), which hide the second round of loads, 51 and 56 us.
// At five it spills (110 us in FP64).
constexpr int kPart3Waves = 4;
template <class R>
__device__ __forceinline__ void part3_tile(const KParams& p, int tile) {
  int i, k;
  if (!pw_point<PW_RUNS>(p, tile, i, k)) return;
  unsigned err = 0;
  // without the status words every column counts as stepped: a level of a
  // skipped one is empty, and part 3 changes nothing there
  const int status = p.track() ? p.colstat[i] : kStatusFull;
  if (!p.exch_zero && (status & kStatusPart1) && p.sc(SC_PEND, i, k) != 0) {
    // a warm clear level of a column that part 2 ran in (front_level)
    const size_t x = p.at(i, k);
    p.vap_ice_exchange[x] = 0;
    p.vap_liq_exchange[x] = 0;
    p.liq_ice_exchange[x] = 0;
  }
  part3_level<R>(p, k, i, status == kStatusFull, err);
  if (k == 0 && p.amble.on && p.amble.water_flux) {
    // the post-amble's boundary fluxes (eamxx_p3_process_interface.hpp:245-258),
    // from the surface precipitation both sedimentation kernels wrote
    const Amble& a = p.amble;
    const double liq = p.precip_liq_surf[i], ice = p.precip_ice_surf[i];
    a.vapor_flux[i] = 0.0;
    a.water_flux[i] = liq + ice;
    a.ice_flux[i] = ice;
    a.heat_flux[i] = 0.0;
  }
  if (err) report_errors(p.err, err);
}

template <class R>
__global__ __launch_bounds__(kTileThreads, kPart3Waves) void p3_part3_lvl_kernel(const KParams p) {
  part3_tile<R>(p, blockIdx.x);
}

// Workgroups go to the 8 XCDs round-robin, and each XCD has its own L2.  A
// block's lanes read a few columns of many levels, so neighbouring blocks share
// every cache line they touch: give each XCD a contiguous range of blocks, so
// that the blocks sharing lines run on one XCD at about the same time.
constexpr int kXcds = 8;
__device__ __forceinline__ int xcd_block(int b, int nb) {
  const int q = nb / kXcds, r = nb % kXcds, x = b % kXcds, n = b / kXcds;
  return x * q + (x < r ? x : r) + n;
}

// The same in runs of kXcdRun blocks per XCD: within each 8 * kXcdRun blocks an
// XCD takes kXcdRun consecutive ones.  For blocks whose work changes along the
// grid: the longest steps first (layout_batch), or the clear columns last
// (p3_order_kernel), which a contiguous range would give to the last XCDs alone.
constexpr int kXcdRun = 16;
__device__ __forceinline__ int run_block(int b, int nb) {
  constexpr int chunk = kXcds * kXcdRun;
  const int c0 = b / chunk * chunk;
  if (c0 + chunk > nb) return b;
  const int r = b - c0;
  return c0 + r % kXcds * kXcdRun + r / kXcds;
}
template <int LPC>
__device__ __forceinline__ int sed_order_block(const KParams& p, int b, int nb) {
  return LPC < 64 && p.ordered() ? run_block(b, nb) : xcd_block(b, nb);
}

// Copies the ice-sedimentation records into the block's LDS copy, in 16-byte
// chunks by the NT threads of the block: requested when the object is made, written
// (and waited for by the whole block) by the call, so that the request travels
// together with whatever the block loads in between: the search for the columns'
// top levels no longer waits for the table (16384 x 128 FP64 sedimentation and part
// 3 288 -> 276 us).
template <class R, int L, int NT>
struct IceTableStage {
  static constexpr int per = ice_rec_len<R, L>() * (int)sizeof(R) / 16;     // chunks per record
  static constexpr int str = ice_lds_stride<R, L>() * (int)sizeof(R) / 16;  // and per record in LDS
  static constexpr int n = kIceCells * per, N = (n + NT - 1) / NT;
  R* s;
  uint4 v[N];
  __device__ __forceinline__ IceTableStage(const R* __restrict__ g, R* lds) : s(lds) {
#pragma unroll
    for (int t = 0; t < N; ++t) {
      const int c = (int)threadIdx.x + t * NT;
      v[t] = reinterpret_cast<const uint4*>(g)[c < n ? c : n - 1];
    }
  }
  __device__ __forceinline__ void operator()() const {
#pragma unroll
    for (int t = 0; t < N; ++t) {
      const int c = (int)threadIdx.x + t * NT;
      if (c < n) reinterpret_cast<uint4*>(s)[c / per * str + c % per] = v[t];
    }
    __syncthreads();
  }
};
struct NoStage {
  __device__ __forceinline__ void operator()() const {}
};

// The ice table's records in the form the ice group of L levels per lane reads.
template <class R, int L>
__device__ __forceinline__ const R* ice_lds_source(const KParams& p) {
  return ice_rec_dif<R, L>() ? TabOf<R>::get(p.tab).ice_sed_d : TabOf<R>::get(p.tab).ice_sed;
}

// The ice group interpolates the ice table from an LDS copy of its records,
// staged once per block, rather than through the L1/L2 caches: 16 gathers per
// level and substep become LDS reads (ice sedimentation 3-13 % faster at
// 21600 x 72 and 16384 x 128 with the plain records).
template <class R, int LPC, int L, int WPB, int G>
__global__ __launch_bounds__(64 * WPB, (sed_waves_per_simd<R, G, L>())) void p3_sed_kernel(const KParams p) {
  if constexpr (G == SED_ICE) {
    static_assert(WPB == 4 || !ice_rec_dif<R, L>(), "the LDS budget assumes blocks of 4 wavefronts");
    __shared__ __align__(16) R s_tab[ice_lds_len<R, L>()];
    const IceTableStage<R, L, 64 * WPB> stage(ice_lds_source<R, L>(p), s_tab);
    sed_block<R, LPC, L, WPB, G>(p, sed_order_block<LPC>(p, blockIdx.x, gridDim.x), s_tab, stage);
  } else {
    sed_block<R, LPC, L, WPB, G>(p, sed_order_block<LPC>(p, blockIdx.x, gridDim.x), nullptr, NoStage{});
  }
}

// Both species groups in one launch, for shapes at which they run on the same
// lanes and levels per lane: blocks
// [0, nb_ice) run the ice group and the blocks after them the liquid group,
// over the same column blocks.  Workgroups are dispatched in order, so the
// short liquid blocks take the CUs that the long ice blocks free at the end of
// the ice work, the longest work first.  Two kernels side by side on two
// streams interleave their blocks from the start instead, and the liquid
// blocks then delay the ice blocks; nor is there a fork or a join between
// streams.  Each block runs the code of the two-kernel form, so the results
// are the same bits.  The kernel is compiled for the ice group's wavefronts
// per SIMD; the shapes it is launched at are those where the liquid group's
// code also fits that register budget without a spill (in FP64 not at 3
// levels per lane, where the ice group runs three wavefronts: the liquid group needed
// 173 VGPRs of 168 when the line was drawn; a kernel of its own now takes 139 to 143).
template <class R, int LPC, int L, int WPB>
__global__ __launch_bounds__(64 * WPB, (sed_waves_per_simd<R, SED_ICE, L>())) void p3_sed_fused_kernel(
    const KParams p, int nb_ice) {
  static_assert(WPB == 4 || !ice_rec_dif<R, L>(), "the LDS budget assumes blocks of 4 wavefronts");
  __shared__ __align__(16) R s_tab[ice_lds_len<R, L>()];
  const int b = blockIdx.x;  // uniform over the block: the whole block takes one branch
  if (b < nb_ice) {
    const IceTableStage<R, L, 64 * WPB> stage(ice_lds_source<R, L>(p), s_tab);
    sed_block<R, LPC, L, WPB, SED_ICE>(p, sed_order_block<LPC>(p, b, nb_ice), s_tab, stage);
  } else {
    // block b runs on XCD b % 8; the liquid blocks' offset nb_ice only rotates
    // which XCD receives which contiguous range of column blocks
    sed_block<R, LPC, L, WPB, SED_LIQ>(p, sed_order_block<LPC>(p, b - nb_ice, (int)gridDim.x - nb_ice), nullptr, NoStage{});
  }
}

}  // namespace p3d
