// CLOUDSC for gfx950 -- the column kernel.  See cloudsc_kernel.h for the
// data layout and the register-level reformulation.  Line citations refer to
// ifs-source/arpifs/phys_ec/cloudsc.F90 unless another file is named.
#include <hip/hip_runtime.h>

#include <map>
#include <type_traits>
#include <mutex>
#include <utility>

#include "cloudsc_device.h"
#include "cloudsc_kernel.h"
#include "cloudsc_budget.h"
#include "cloudsc_truncation.h"
#include "satadj_device.h"

namespace cloudsc_gpu {

// The reference's negative-condensate warnings (cloudsc.F90:3794 liquid, :3802 ice) as counts: one atomic add per
// wave and counter, by the wave's first active lane, only when some lane of the wave warns.
__device__ __forceinline__ void count_warnings(uint32_t* n, bool wl, bool wi) {
  const uint64_t bl = __ballot(wl), bi = __ballot(wi);
  if ((bl | bi) == 0) return;
  const uint64_t act = __ballot(1);
  if (__lane_id() == (unsigned)(__ffsll((long long)act) - 1)) {
    if (bl) atomicAdd(n, (uint32_t)__popcll(bl));
    if (bi) atomicAdd(n + 1, (uint32_t)__popcll(bi));
  }
}

// KC / KCD: constants of the working precision R and of the water-budget precision RD, either the run-time
// structure KConst or the compile-time default configuration KConstDefault (same member names).
// UNI: every wave lies in one block (NPROMA a multiple of 64), so block-dependent offsets are wave-uniform.
// SAT: the fused CALLPAR sequence (callpar.F90:1253-1293): on every level at or below NCLDTOP the column first runs
// CLOUD_SATADJ for the point (satadj_point), adds its tendencies to TENDENCY_CML in place (STATE_INCREMENT,
// :1278-1279), stores them as TENDENCY_SATADJ (STATE_COPY, :1289), and CLOUDSC then reads the incremented CML
// tendencies from registers.
// BUD: the process budgets (LCLDBUD*) are recorded per level and written into PEXTRA (cloudsc_budget.h).
// WPE: minimum waves per SIMD the register allocation must allow (0: the compiler's choice); fewer registers per
// lane for more waves in flight, at the price of spills when the live state does not fit.
// KL: number of levels fixed at compile time (0: d.klev at run time), so that the level loop and every level
// offset are constants of the instantiation.
template <typename R, typename RD, typename KC, typename KCD, int BLOCK, bool UNI, bool SAT, bool BUD, int WPE = 0,
          int KL = 0>
__global__ __launch_bounds__(BLOCK) __attribute__((amdgpu_waves_per_eu(WPE > 0 ? WPE : 1))) void
cloudsc_column_kernel(const KArgs<R, KC, KCD> args) {
  const KC& c = args.c;
  const KCD& cd = args.cd;
  const KPtrs<R>& p = args.p;
  const KDims& d = args.d;
  const KSatPtrs<R>& s = args.s;
  const KBudPtrs<R>& bp = args.bp;
  const int ssc_off = args.ssc_off;
  // The ~40 array bases exceed the scalar registers: held across the level loop they would be spilled to vector
  // lanes and come back through v_readlane (57 in the mixed kernel's code, 172 with the loads ahead).  Inside the loop
  // they are read from the kernel arguments (scalar cache) where they are used; the empty asm hides that the address
  // is loop-invariant.
  typedef const __attribute__((address_space(4))) KArgs<R, KC, KCD> CArgs;
  auto fresh = [] {
    uint64_t a = (uint64_t)__builtin_amdgcn_kernarg_segment_ptr();
    asm volatile("" : "+s"(a));
    return (CArgs*)a;
  };
  const uint32_t g = xcd_group(blockIdx.x, gridDim.x) * BLOCK + threadIdx.x;
  const uint32_t nproma = (uint32_t)d.nproma, klev = KL > 0 ? (uint32_t)KL : (uint32_t)d.klev;
  if (g >= (uint32_t)d.ngpblks * nproma) return;
  uint32_t b = g / nproma;
  if (UNI) b = __builtin_amdgcn_readfirstlane(b);
  const uint32_t jl = g - b * nproma;  // 0-based JL-1
  constexpr uint32_t E = sizeof(R);
  const uint32_t jo = jl * E, joi = jl * 4u;           // lane offsets (R and int32 arrays)
  const uint32_t u1 = b * nproma * E, u1i = b * nproma * 4u;
  // PRAINFRAC_TOPRFZ is zeroed for all KLON columns of the block (:1010)
  ST(p.prainfrac_toprfz, u1, jo, R(0));
  const int kfdia = min(d.kfdia, d.ngptot - (int)(b * nproma));
  if ((int)jl < d.kidia - 1 || (int)jl >= kfdia) return;

  const uint32_t s2 = nproma * klev;
  const uint32_t lstep = nproma * E;                  // one level
  const uint32_t sstep = s2 * E;                      // one species of a (NPROMA,KLEV,n) array
  const uint32_t b2 = b * s2 * E;                     // (NPROMA,KLEV) level 0
  const uint32_t bh = b * (s2 + nproma) * E;          // (NPROMA,KLEV+1) level 0
  const uint32_t b5 = b * s2 * 5 * E, b4 = b * s2 * 4 * E, b2x = b * s2 * 2 * E;

  const R ptsphy = c.ptsphy, zqtmst = c.zqtmst, zepsec = R(1.e-14);
  const R rlmin = c.rlmin;
  R* bud_lds = nullptr;  // this lane's budget entries and vertical-integral sums (BUD only)
  ViAcc<R> vacc{nullptr, BLOCK};
  const uint32_t kfx = (uint32_t)bp.kfldx;
  auto ext = [&](int fld, uint32_t kk) {  // byte offset of PEXTRA(JL,kk,fld) of this block
    return (((b * kfx + (uint32_t)(fld - 1)) * klev + (kk - 1)) * nproma) * E + jo;
  };
  if constexpr (BUD) {
    __shared__ R s_bud[(NBUD + NVI) * BLOCK];
    bud_lds = s_bud + threadIdx.x;
    vacc.s = s_bud + NBUD * BLOCK + threadIdx.x;
    if (bp.flags & BUD_VERTINT) vertint_begin(vacc, bp, ext);
  }
  // LRAD_CLOUD_INHOMOG / LCLOUD_INHOMOG: grid length of the column (diagnostic instantiation only)
  const R zgridlen = (BUD && (bp.fsd || bp.inhomog)) ? fsd_gridlen(bp.ra, bp.rpi, LD(bp.pgaw, u1, jo)) : R(0);

  // Per-column inputs
  const R plsm = LD(p.plsm, u1, jo);
  const int32_t ktype = LD(p.ktype, u1i, joi);
  const bool ldcum = LD(p.ldcum, u1i, joi) != 0;
  const R peis = LD(p.peis, u1, jo);
  const R paph_surf = LD(p.paph, bh + klev * lstep, jo);
  const R zadvw = (ktype == 1 && c.rmfadvw > R(0)) ? R(1) - c.rmfadvw : R(1);                  // :696-703
  const R zadvwd = (ktype == 1 && c.rmfadvw > R(0)) ? R(1) - c.rmfadvw * c.rmfadvwdd : R(1);
  const R zconst = plsm > R(0.5) ? c.rcl_kk_cloud_num_land : c.rcl_kk_cloud_num_sea;          // :2063-2069
  const R zconst_pow = s_pow(zconst, c.rcl_kkbaun);
  const int ncldtop0 = c.ncldtop - 1;  // 0-based first level of the cloud scheme

  // Level-carried state (:1205-1211 and :1011)
  R qxnm1_l = R(0), qxnm1_i = R(0), qxnm1_r = R(0), qxnm1_s = R(0);
  R zanewm1 = R(0), zcovptot = R(0), zcovpmax = R(0), zcldtopdist = R(0);
  bool llrainliq = true;
  R prainfrac = R(0);
  R pf_i = R(0), pf_r = R(0), pf_s = R(0);  // ZPFPLSX(JK) of the falling species
  R za_prev = R(0), qr_prev = R(0), qs_prev = R(0), t_prev = R(0), pap_prev = R(0);
  // DDH flux running sums at the upper half level (:4231-4242)
  R sqlf = R(0), sqif = R(0), cqlng = R(0), cqnng = R(0), sqltur = R(0), sqitur = R(0);
  ST(p.pfsqlf, bh, jo, R(0));
  ST(p.pfsqif, bh, jo, R(0));
  ST(p.pfsqrf, bh, jo, R(0));
  ST(p.pfsqsf, bh, jo, R(0));
  ST(p.pfcqlng, bh, jo, R(0));
  ST(p.pfcqnng, bh, jo, R(0));
  ST(p.pfcqrng, bh, jo, R(0));
  ST(p.pfcqsng, bh, jo, R(0));
  ST(p.pfsqltur, bh, jo, R(0));
  ST(p.pfsqitur, bh, jo, R(0));

  R paph_k = LD(p.paph, bh, jo);
  R pmfu_k = LD(p.pmfu, b2, jo), pmfd_k = LD(p.pmfd, b2, jo);

  // The inputs of one level (and PMFU, PMFD, PLU of the level below it).  They are loaded near the end of the level
  // before, after its implicit solve and ahead of its ~20 stores: loads and stores share one in-order wait counter, so loads issued after the stores
  // would also wait for those.  At that point few temporaries are live and the ~26 values raise no register peak
  // (FP32 138 -> 140, mixed 167 -> 166).  With the bases read where they are used (above), same box: mixed 655,360 x
  // L137 4.17 -> 3.84 ms, FP32 327,680 x L137 2.24 -> 2.02 ms, FP64 65,536 x L137 2.29 -> 1.99 ms, FP32 40,007 x L91 in
  // blocks of 100 563 -> 466 us, fused FP32 262,144 x L137 2.85 -> 2.45 ms.
  // Earlier (before the truncation) the peak grows: mixed 3.84 -> 4.50 ms.
#include "sweep_load.inc"

  const bool tsat = SAT && s.tsat_t;

  Level nxt = load(0);
  for (uint32_t k = 0; k < klev; ++k) {
    const uint32_t i2 = b2 + k * lstep;        // level k of a (NPROMA,KLEV) array
    const uint32_t ih0 = bh + k * lstep;       // upper half level of layer k
    const uint32_t ih1 = ih0 + lstep;          // lower half level
    const uint32_t i5 = b5 + k * lstep;        // (all wave-uniform with UNI; the lane adds jo)
    const bool has_next = k + 1 < klev;
    const Level in = nxt;
    const R pmfu_n = in.mfu_n, pmfd_n = in.mfd_n, plu_n = in.lu_n, paph_k1 = in.paph1, pap = in.pap;
    const R pt = in.t, pq = in.q, pa = in.a, pvfl = in.vfl, pvfi = in.vfi, pludeli1 = in.lude1, pludeli2 = in.lude2;
    const R pcl_l = in.ql, pcl_i = in.qi;
    R tcml_t = in.ct, tcml_q = in.cq, tcml_a = in.ca, tcml_l = in.cl, tcml_i = in.ci;

#include "sweep_satadj.inc"
#include "sweep_state.inc"
    // Outputs of this level; defaults are those of levels above NCLDTOP.
    R qxn_l = R(0), qxn_i = R(0), qxn_r = R(0), qxn_s = R(0);
    R tcld_l = R(0), tcld_i = R(0), tcld_r = R(0), tcld_s = R(0), ta = R(0);
#include "sweep_fluxes.inc"
    // ZLFSD, ZANEWP, ZRATFSD of this level (LRAD_CLOUD_INHOMOG); above NCLDTOP they keep these values (:944-951)
    R fsd_liq = BUD ? bp.rcloud_frac_std : R(0), fsd_anewp = R(0), fsd_rat = R(0);

    if ((int)k >= ncldtop0) {
      const bool above_top = (int)k > ncldtop0;  // JK > NCLDTOP
      Bud<R, BUD> bud(bud_lds, BLOCK);  // ZBUDCC/ZBUDL/ZBUDI of this level, zeroed (:1271-1273)
      // FP32: the 3D budget words are loaded here and arrive during the level; FP64 loads them at section 7
      // (holding them across the level would spill)
      Pre3D<R> bud_pre;
      if constexpr (BUD && sizeof(R) == 4) budget_prefetch(bud_pre, bp, ext, k + 1);
      R zrainaut = R(0), zrainacc = R(0), zsnowaut = R(0), zsnowrime = R(0);  // (:1239-1242)
      const R plude_in = in.lude;
#include "sweep_derived.inc"
#include "sweep_early.inc"
#define EARLY(n, ...) early_##n(__VA_ARGS__)
#include "sweep_processes.inc"
#undef EARLY
#include "sweep_tendencies.inc"
      if (has_next) nxt = load(k + 1);
#include "sweep_supersat.inc"
      STN<UNI>(fresh()->p.pcovptot, i2, jo, zcovptot);  // (:3814-3816)
      if constexpr (BUD) {
        if (bp.fsd) {
          // cloud fraction at the end of the step with the precipitation fraction (:3818-3822); ZDA = ZANEW - ZAORIG
          const R a_end = pa + (zanewm1 - zaorig);
          if (a_end > R(0.001)) fsd_anewp = m_max(m_max(a_end, zcovptot), R(0.1));
          // detrained share of the condensate (:4112-4121), from PLUDE as rescaled above
          if (ql0 + qi0 + plude > rlmin) fsd_rat = m_max(R(0), m_min(R(1), m_share(plude, plude + ql0 + qi0)));
        }
      }
      // section 7 (:3826-4101), only when a budget writes PEXTRA: otherwise the budget inputs may be NULL (a run
      // with only LRAD_CLOUD_INHOMOG)
      if constexpr (BUD) {
        if (bp.flags & BUD_OUT) {
          const R zdz = m_div(zdp, zrho * c.rg);
          if constexpr (sizeof(R) == 8) budget_prefetch(bud_pre, bp, ext, k + 1);
          budget_write<R>(bud, vacc, bud_pre, bp, ext, k + 1, i2 + jo, zqtmst, ptsphy, zdz, qxn_l, qxn_i, c.ralvdcp,
                          c.ralsdcp, bp.ralfdcp);
        }
      }
    }

    if constexpr (BUD) {
      if (bp.fsd) {  // PFSD of every level (:4307-4359); ZQX and ZTP1 are the tidied start-of-step state
        const R zrho_f = m_div(pap, c.rd * ztp1);
        ST(bp.pfsd, i2, jo, cloud_fsd(bp.rcloud_frac_std, zgridlen, qv, qi, paph_k1 - paph_k, zrho_f, c.rg,
                                      fsd_anewp, fsd_rat, qxn_i, qxn_l, fsd_liq));
      }
    }

    if (has_next && (int)k < ncldtop0) nxt = load(k + 1);

#include "sweep_store.inc"
    // carry to the next level
    za_prev = za;
    qr_prev = qr;
    qs_prev = qs;
    t_prev = ztp1;
    pap_prev = pap;
    paph_k = paph_k1;
    pmfu_k = pmfu_n;
    pmfd_k = pmfd_n;
  }
  if constexpr (BUD) {
    if (bp.flags & BUD_VERTINT) vertint_end(vacc, bp, ext, prainfrac, ktype, peis, u1i + joi, (int)klev - ncldtop0);
  }
  // precipitation fluxes at the surface half level
  {
    const uint32_t ih = bh + klev * lstep;
    const R fl = pf_r + R(0), fn = pf_s + pf_i;
    ST(p.pfplsl, ih, jo, fl);
    ST(p.pfplsn, ih, jo, fn);
    ST(p.pfhpsl, ih, jo, -c.rlvtt * fl);
    ST(p.pfhpsn, ih, jo, -c.rlstt * fn);
  }
  ST(p.prainfrac_toprfz, u1, jo, prainfrac);
}

// ---------------------------------------------------------------------------
// The same sweep by three waves to 64 columns, a level apart: the first loads level t and computes what depends on it
// alone (and adjusts it, SAT), the second runs the processes and the implicit solve of level t - 1, the third the tendencies, the
// supersaturation check and the stores of level t - 2.  They pass what the next one needs through LDS, a barrier per
// level.  The parts are the ones of the kernel above, so the results are the same bit for bit.  A wave alone issues a
// vector instruction in about half of its cycles and waits in a quarter (1,190 instructions a level, 3.6 us); here the
// second wave, a chain of short branches, bounds a level: 2.3 us, against 1.6 us with the second wave's processes left
// out.  Without the early factors in the first wave it is 2.5 us.
// ---------------------------------------------------------------------------
// What the first wave passes to the second (the level's state is read from SWEEP_KEEP), to the third, and the second to
// the third.
#define SWEEP_HEAD(F)                                                                                              \
  F(ztp1) F(za) F(zaorig) F(zqsliq) F(zqsice) F(zqsmix) F(zliqfrac) F(zicefrac) F(zli) F(zdp) F(zrho)    \
  F(zdtgdp) F(zrdtgdp) F(zcorqsliq) F(zcorqsice) F(zdqsmixdt) F(zcorqsmix) F(zevaplimmix) F(ztmpa) F(plude_in)      \
  F(plu_n) F(snde1) F(snde2) F(pmfu_n) F(pmfd_n)                                                                    \
  F(e_erosion) F(e_fallspeed) F(e_autoconversion) F(e_accretion) F(e_critical_rh) F(e_evaporation) F(e_evap_fall)   \
  F(e_evap_corr) F(e_deposition) F(e_nucleation) F(e_supersaturation) F(e_snow_growth) F(e_snow_air) F(e_snow_corr) \
  F(e_snow_rate) F(e_melting) F(e_freezing) F(e_rime_fall) F(e_sublimation_q) F(e_sublimation)
#define SWEEP_SHARED(F) F(ql) F(qi) F(qr) F(qs) F(qv) F(paph_k1) F(pap) F(pludeli1) F(pludeli2)
#define SWEEP_REST(F)                                                                                              \
  F(pt) F(pq) F(pa) F(tcml_t) F(tcml_q) F(tcml_a) F(ql0) F(qi0) F(qr0) F(qs0) F(tt) F(tq) F(zlneg_l) F(zlneg_i)     \
  F(zlneg_r) F(zlneg_s) F(pvfl) F(pvfi)
#define SWEEP_KEEP(F) SWEEP_SHARED(F) SWEEP_REST(F)
#define SWEEP_SOLVE(F)                                                                                             \
  F(qxn_l) F(qxn_i) F(qxn_r) F(qxn_s) F(qxn_v) F(zda) F(fq_l) F(fq_i) F(fq_r) F(fq_s) F(pf_i) F(pf_r) F(pf_s) F(zcovptot)
#define SWEEP_COUNT(n) +1
#define SWEEP_PUT(n) to[i++ * 64] = n;
#define SWEEP_GET(n) R n = from[i++ * 64];
#define SWEEP_SET(n) n = from[i++ * 64];

template <typename R, typename RD, typename KC, typename KCD, bool UNI, bool SAT>
__global__ __launch_bounds__(192) void cloudsc_pipeline_kernel(const KArgs<R, KC, KCD> args) {
  constexpr bool BUD = false;
  constexpr int NHEAD = 0 SWEEP_HEAD(SWEEP_COUNT), NKEEP = 0 SWEEP_KEEP(SWEEP_COUNT), NSOLVE = 0 SWEEP_SOLVE(SWEEP_COUNT);
  __shared__ R s_head[2][NHEAD][64], s_keep[3][NKEEP][64], s_solve[2][NSOLVE][64];
  const KC& c = args.c;
  const KPtrs<R>& p = args.p;
  const KDims& d = args.d;
  const int ssc_off = args.ssc_off;
  typedef const __attribute__((address_space(4))) KArgs<R, KC, KCD> CArgs;
  auto fresh = [] {
    uint64_t a = (uint64_t)__builtin_amdgcn_kernarg_segment_ptr();
    asm volatile("" : "+s"(a));
    return (CArgs*)a;
  };
  const uint32_t lane = threadIdx.x & 63u;
  const int role = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const uint32_t g = xcd_group(blockIdx.x, gridDim.x) * 64u + lane;
  const uint32_t nproma = (uint32_t)d.nproma, klev = (uint32_t)d.klev;
  if (g >= (uint32_t)d.ngpblks * nproma) return;  // the same lanes in all three waves
  uint32_t b = g / nproma;
  if (UNI) b = __builtin_amdgcn_readfirstlane(b);
  const uint32_t jl = g - b * nproma;
  constexpr uint32_t E = sizeof(R);
  const uint32_t jo = jl * E, joi = jl * 4u;
  const uint32_t u1 = b * nproma * E, u1i = b * nproma * 4u;
  if (role == 1) ST(p.prainfrac_toprfz, u1, jo, R(0));
  const int kfdia = min(d.kfdia, d.ngptot - (int)(b * nproma));
  if ((int)jl < d.kidia - 1 || (int)jl >= kfdia) return;
  const uint32_t s2 = nproma * klev;
  const uint32_t lstep = nproma * E, sstep = s2 * E;
  const uint32_t b2 = b * s2 * E, bh = b * (s2 + nproma) * E;
  const uint32_t b5 = b * s2 * 5 * E, b4 = b * s2 * 4 * E, b2x = b * s2 * 2 * E;
  const R ptsphy = c.ptsphy, zqtmst = c.zqtmst, zepsec = R(1.e-14);
  const R rlmin = c.rlmin;
  const int ncldtop0 = c.ncldtop - 1;
  // A level is passed on: this wave's LDS accesses are done (its global ones need not be), then everyone's.
  auto pass = [] {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(15 | (3 << 14) | (7 << 4));  // lgkmcnt(0)
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  };

  if (role == 0) {
    R paph_k = LD(p.paph, bh, jo);
    const R paph_surf = LD(p.paph, bh + klev * lstep, jo);
    const R zconst = LD(p.plsm, u1, jo) > R(0.5) ? c.rcl_kk_cloud_num_land : c.rcl_kk_cloud_num_sea;
    const R zconst_pow = s_pow(zconst, c.rcl_kkbaun);
#include "sweep_load.inc"
    const KCD& cd = args.cd;
    const bool tsat = SAT && args.s.tsat_t;
    Level nxt = load(0);
    for (uint32_t k = 0; k < klev; ++k) {
      const uint32_t i2 = b2 + k * lstep, i5 = b5 + k * lstep;
      const Level in = nxt;
      if (k + 1 < klev) nxt = load(k + 1);
      const R pmfu_n = in.mfu_n, pmfd_n = in.mfd_n, plu_n = in.lu_n, paph_k1 = in.paph1, pap = in.pap;
      const R pt = in.t, pq = in.q, pa = in.a, pvfl = in.vfl, pvfi = in.vfi, pludeli1 = in.lude1, pludeli2 = in.lude2;
      const R pcl_l = in.ql, pcl_i = in.qi, plude_in = in.lude, snde1 = in.snde1, snde2 = in.snde2;
      R tcml_t = in.ct, tcml_q = in.cq, tcml_a = in.ca, tcml_l = in.cl, tcml_i = in.ci;
#include "sweep_satadj.inc"
#include "sweep_state.inc"
#include "sweep_derived.inc"
#include "sweep_early.inc"
      R e_erosion = R(0), e_autoconversion = R(0), e_accretion = R(0), e_evaporation = R(0), e_evap_fall = R(0);
      R e_evap_corr = R(0), e_deposition = R(0), e_nucleation = R(0), e_snow_growth = R(0), e_snow_air = R(0);
      R e_snow_corr = R(0), e_snow_rate = R(0), e_melting = R(0), e_freezing = R(0), e_rime_fall = R(0);
      const auto fallcorr_base = s_base(m_div(c.rdensref, zrho));
      const R e_fallspeed = early_fallspeed(fallcorr_base), e_critical_rh = early_critical_rh();
      const R e_supersaturation = early_supersaturation();
      const R e_sublimation_q = early_sublimation_q(), e_sublimation = early_sublimation();
      // the others where the level alone does not rule their process out
      if (zli > zepsec) e_erosion = early_erosion();
      if (zliqcld > zepsec) {
        const auto liq_base = s_base(zliqcld);
        e_autoconversion = early_autoconversion(c.c_aut, liq_base);
        e_accretion = early_accretion(c.c_acc, liq_base);
      }
      if (m_max(R(0), m_min(qv, zqsliq)) < R(0.9) * zqsliq) {  // the humidity limit of evaporation is 0.9 at most
        const R zcorr2 = evap_corr2();
        e_evaporation = early_evaporation(zcorr2);
        e_evap_fall = early_evap_fall(fallcorr_base);
        e_evap_corr = early_evap_corr(zcorr2);
      }
      if (ztp1 <= c.rtt) {
        const R zvpice = m_div(foeeice * c.rv, c.rd);
        e_rime_fall = early_rime_fall(fallcorr_base);
        e_snow_rate = early_snow_rate();
        if (ztp1 < c.rtt - R(5.)) {
          const R zsupersatice = m_div(zqsliq - zqsice, zqsice), zicenuclei = ice_nuclei(zsupersatice);
          e_deposition = early_deposition(zsupersatice, zicenuclei, zvpice);
          e_nucleation = early_nucleation(zicenuclei);
        }
        if (e_supersaturation > R(0)) {
          const R zcorrfac2 = snow_corr2();
          e_snow_growth = early_snow_growth(e_supersaturation, zcorrfac2, zvpice);
          e_snow_air = early_snow_air();
          e_snow_corr = early_snow_corr(zcorrfac2);
        }
        if (qr > zepsec) e_freezing = early_freezing();
      } else {
        e_melting = early_melting();
      }
      {
        R* to = &s_head[k & 1][0][lane];
        int i = 0;
        SWEEP_HEAD(SWEEP_PUT)
      }
      {
        R* to = &s_keep[k % 3][0][lane];
        int i = 0;
        SWEEP_KEEP(SWEEP_PUT)
      }
      paph_k = paph_k1;
      pass();
    }
    pass();
    pass();
  } else if (role == 1) {
    const int32_t ktype = LD(p.ktype, u1i, joi);
    const bool ldcum = LD(p.ldcum, u1i, joi) != 0;
    const R peis = LD(p.peis, u1, jo);
    const R zadvw = (ktype == 1 && c.rmfadvw > R(0)) ? R(1) - c.rmfadvw : R(1);
    const R zadvwd = (ktype == 1 && c.rmfadvw > R(0)) ? R(1) - c.rmfadvw * c.rmfadvwdd : R(1);
    R qxnm1_l = R(0), qxnm1_i = R(0), qxnm1_r = R(0), qxnm1_s = R(0);
    R zanewm1 = R(0), zcovptot = R(0), zcovpmax = R(0), zcldtopdist = R(0);
    bool llrainliq = true;
    R prainfrac = R(0);
    R pf_i = R(0), pf_r = R(0), pf_s = R(0);
    R za_prev = R(0), qr_prev = R(0), qs_prev = R(0), t_prev = R(0), pap_prev = R(0);
    R paph_k = LD(p.paph, bh, jo);
    R pmfu_k = LD(p.pmfu, b2, jo), pmfd_k = LD(p.pmfd, b2, jo);
    pass();
    for (uint32_t k = 0; k < klev; ++k) {
      const R* from = &s_head[k & 1][0][lane];
      int i = 0;
      SWEEP_HEAD(SWEEP_GET)
      from = &s_keep[k % 3][0][lane];
      i = 0;
      SWEEP_SHARED(SWEEP_GET)
      if ((int)k >= ncldtop0) {
        const uint32_t i2 = b2 + k * lstep;
        const bool has_next = k + 1 < klev, above_top = (int)k > ncldtop0;
        Bud<R, BUD> bud(nullptr, 64);
        const KBudPtrs<R>& bp = args.bp;
        const R zgridlen = R(0);
        R fsd_liq = R(0);
        const struct {
          R snde1, snde2;
        } in = {snde1, snde2};
        R qxn_l, qxn_i, qxn_r, qxn_s;
        // (arguments of the early factors, which are not evaluated here)
        const R foeeice = R(1);
        auto evap_corr2 = [] { return R(1); };
        auto snow_corr2 = [] { return R(1); };
        auto ice_nuclei = [](R) { return R(1); };
        R zrainaut = R(0), zrainacc = R(0), zsnowaut = R(0), zsnowrime = R(0);
        R zliqcld = ql * ztmpa, zicecld = qi * ztmpa;
        const R zlicld = zliqcld + zicecld;
#define EARLY(n, ...) e_##n
#include "sweep_processes.inc"
#undef EARLY
        R* to = &s_solve[k & 1][0][lane];
        int i = 0;
        SWEEP_SOLVE(SWEEP_PUT)
      }
      za_prev = za;
      qr_prev = qr;
      qs_prev = qs;
      t_prev = ztp1;
      pap_prev = pap;
      paph_k = paph_k1;
      pmfu_k = pmfu_n;
      pmfd_k = pmfd_n;
      pass();
    }
    pass();
    ST(p.prainfrac_toprfz, u1, jo, prainfrac);
  } else {
    R pf_i = R(0), pf_r = R(0), pf_s = R(0);
    R sqlf = R(0), sqif = R(0), cqlng = R(0), cqnng = R(0), sqltur = R(0), sqitur = R(0);
    ST(p.pfsqlf, bh, jo, R(0));
    ST(p.pfsqif, bh, jo, R(0));
    ST(p.pfsqrf, bh, jo, R(0));
    ST(p.pfsqsf, bh, jo, R(0));
    ST(p.pfcqlng, bh, jo, R(0));
    ST(p.pfcqnng, bh, jo, R(0));
    ST(p.pfcqrng, bh, jo, R(0));
    ST(p.pfcqsng, bh, jo, R(0));
    ST(p.pfsqltur, bh, jo, R(0));
    ST(p.pfsqitur, bh, jo, R(0));
    R paph_k = LD(p.paph, bh, jo);
    pass();
    pass();
    for (uint32_t k = 0; k < klev; ++k) {
      const uint32_t i2 = b2 + k * lstep, ih0 = bh + k * lstep, ih1 = ih0 + lstep, i5 = b5 + k * lstep;
      const R* from = &s_keep[k % 3][0][lane];
      int i = 0;
      SWEEP_KEEP(SWEEP_GET)
      R qxn_l = R(0), qxn_i = R(0), qxn_r = R(0), qxn_s = R(0);
      R tcld_l = R(0), tcld_i = R(0), tcld_r = R(0), tcld_s = R(0), ta = R(0);
#include "sweep_fluxes.inc"
      if ((int)k >= ncldtop0) {
        Bud<R, BUD> bud(nullptr, 64);
        R qxn_v, zda, fq_l, fq_i, fq_r, fq_s, zcovptot;
        {
          const R* from = &s_solve[k & 1][0][lane];
          int i = 0;
          SWEEP_SOLVE(SWEEP_SET)
        }
#include "sweep_tendencies.inc"
#include "sweep_supersat.inc"
        STN<UNI>(fresh()->p.pcovptot, i2, jo, zcovptot);
      }
#include "sweep_store.inc"
      paph_k = paph_k1;
      pass();
    }
    const uint32_t ih = bh + klev * lstep;
    const R fl = pf_r + R(0), fn = pf_s + pf_i;
    ST(p.pfplsl, ih, jo, fl);
    ST(p.pfplsn, ih, jo, fn);
    ST(p.pfhpsl, ih, jo, -c.rlvtt * fl);
    ST(p.pfhpsn, ih, jo, -c.rlstt * fn);
  }
}

// ---------------------------------------------------------------------------
// Host-side launchers (declared in cloudsc_launch.h)
// ---------------------------------------------------------------------------
template <typename T>
KConst<T> make_kconst(const cloudsc_params_t& q, double ptsphy_in) {
  KConst<T> c{};
  const T ptsphy = T(ptsphy_in);
  c.rg = T(q.rg); c.rd = T(q.rd); c.rv = T(q.rv); c.retv = T(q.retv); c.rtt = T(q.rtt);
  c.rlvtt = T(q.rlvtt); c.rlstt = T(q.rlstt); c.rpi = T(q.rpi);
  c.rv_rd = c.rv / c.rd;
  c.r2es = T(q.r2es); c.r3les = T(q.r3les); c.r3ies = T(q.r3ies); c.r4les = T(q.r4les); c.r4ies = T(q.r4ies);
  c.r5les = T(q.r5les); c.r5ies = T(q.r5ies); c.r5alvcp = T(q.r5alvcp); c.r5alscp = T(q.r5alscp);
  c.ralvdcp = T(q.ralvdcp); c.ralsdcp = T(q.ralsdcp); c.rtwat = T(q.rtwat); c.rtice = T(q.rtice);
  c.rtwat_rtice_r = T(q.rtwat_rtice_r); c.rkoop1 = T(q.rkoop1); c.rkoop2 = T(q.rkoop2);
  c.ramid = T(q.ramid); c.ramin = T(q.ramin); c.rlmin = T(q.rlmin); c.rcldiff = T(q.rcldiff);
  c.rcldiff_convi = T(q.rcldiff_convi); c.rkconv = T(q.rkconv);
  c.rsnowlin1 = T(q.rsnowlin1); c.rsnowlin2 = T(q.rsnowlin2); c.rlcritsnow = T(q.rlcritsnow);
  c.rvice = T(q.rvice); c.rvrain = T(q.rvrain); c.rvsnow = T(q.rvsnow); c.rxfallspeedrain = T(q.rxfallspeedrain);
  c.rcldtopcf = T(q.rcldtopcf); c.rdepliqrefrate = T(q.rdepliqrefrate); c.rdepliqrefdepth = T(q.rdepliqrefdepth);
  c.rcl_overlapliqice = T(q.rcl_overlapliqice); c.rcl_effrime = T(q.rcl_effrime); c.riceinit = T(q.riceinit);
  c.rthomo = T(q.rthomo); c.rprecrhmax = T(q.rprecrhmax); c.rpecons = T(q.rpecons); c.rvrfactor = T(q.rvrfactor);
  c.rcovpmin = T(q.rcovpmin); c.rtaumel = T(q.rtaumel); c.rssicefactor = T(q.rssicefactor);
  c.rdenswat = T(q.rdenswat); c.rdensref = T(q.rdensref);
  c.rcl_dr = T(q.rcl_dr); c.rcl_x1r = T(q.rcl_x1r); c.rcl_x2r = T(q.rcl_x2r); c.rcl_x1s = T(q.rcl_x1s);
  c.rcl_lam1r = T(q.rcl_lam1r); c.rcl_lam2r = T(q.rcl_lam2r); c.rcl_lam1s = T(q.rcl_lam1s); c.rcl_lam2s = T(q.rcl_lam2s);
  c.rcl_cdenom1 = T(q.rcl_cdenom1); c.rcl_cdenom2 = T(q.rcl_cdenom2); c.rcl_cdenom3 = T(q.rcl_cdenom3);
  c.rcl_const1r = T(q.rcl_const1r); c.rcl_const2r = T(q.rcl_const2r); c.rcl_const3r = T(q.rcl_const3r);
  c.rcl_const4r = T(q.rcl_const4r); c.rcl_const5r = T(q.rcl_const5r); c.rcl_const6r = T(q.rcl_const6r);
  c.rcl_const7r = T(q.rcl_const7r); c.rcl_kkaac = T(q.rcl_kkaac); c.rcl_kkbac = T(q.rcl_kkbac);
  c.rcl_kkaau = T(q.rcl_kkaau);
  c.rcl_kkbauq = T(q.rcl_kkbauq); c.rcl_kkbaun = T(q.rcl_kkbaun);
  c.rcl_kk_cloud_num_sea = T(q.rcl_kk_cloud_num_sea); c.rcl_kk_cloud_num_land = T(q.rcl_kk_cloud_num_land);
  c.rcl_fzrab = T(q.rcl_fzrab); c.rcl_apb1 = T(q.rcl_apb1); c.rcl_apb2 = T(q.rcl_apb2); c.rcl_apb3 = T(q.rcl_apb3);
  c.rcl_const1s = T(q.rcl_const1s); c.rcl_const2s = T(q.rcl_const2s); c.rcl_const3s = T(q.rcl_const3s);
  c.rcl_const4s = T(q.rcl_const4s); c.rcl_const5s = T(q.rcl_const5s); c.rcl_const6s = T(q.rcl_const6s);
  c.rcl_const7s = T(q.rcl_const7s); c.rcl_const8s = T(q.rcl_const8s);
  c.rmfadvw = T(q.rmfadvw); c.rmfadvwdd = T(q.rmfadvwdd);
  c.ptsphy = ptsphy;
  c.zqtmst = T(1) / ptsphy;                   // :798
  c.zrdcp = c.rd / T(q.rcpd);                 // :800
  c.zrg_r = T(1) / c.rg;                      // :803
  c.zrldcp = T(1) / (c.ralsdcp - c.ralvdcp);  // :804
  c.zepsilon = T(100) * std::numeric_limits<T>::epsilon();  // :693
  c.rdtg_r = T(1) / (ptsphy * c.rg);          // :1285
  c.c_aut = T(q.rcl_inhomogaut) * ptsphy * T(q.rcl_kkaau);
  c.c_acc = T(q.rcl_inhomogacc) * ptsphy * T(q.rcl_kkaac);
  c.ncldtop = q.ncldtop;
  c.lmfdsnow = q.lmfdsnow;
  return c;
}

template <typename T>
KConstDefault<T> make_kconst_default(const cloudsc_params_t& q, double ptsphy_in) {
  KConstDefault<T> c{};
  const T ptsphy = T(ptsphy_in);
  c.ptsphy = ptsphy;
  c.zqtmst = T(1) / ptsphy;
  c.rdtg_r = T(1) / (ptsphy * KConstDefault<T>::rg);
  c.c_aut = T(cloudsc_defaults::rcl_inhomogaut) * ptsphy * T(cloudsc_defaults::rcl_kkaau);
  c.c_acc = T(cloudsc_defaults::rcl_inhomogacc) * ptsphy * T(cloudsc_defaults::rcl_kkaac);
  c.rssicefactor = T(q.rssicefactor);
  c.ncldtop = q.ncldtop;
  return c;
}

// True when every configuration value except RSSICEFACTOR (time step) and NCLDTOP (levels)
// equals the default configuration the specialised kernels are compiled with.
bool is_default_config(const cloudsc_params_t& q) {
  using namespace cloudsc_defaults;
#define CLOUDSC_SAME(name) (q.name == name) &&
  return CLOUDSC_SAME(rg) CLOUDSC_SAME(rd) CLOUDSC_SAME(rv) CLOUDSC_SAME(rcpd) CLOUDSC_SAME(retv) CLOUDSC_SAME(rtt)
      CLOUDSC_SAME(rlvtt) CLOUDSC_SAME(rlstt) CLOUDSC_SAME(rpi) CLOUDSC_SAME(r2es) CLOUDSC_SAME(r3les)
      CLOUDSC_SAME(r3ies) CLOUDSC_SAME(r4les) CLOUDSC_SAME(r4ies) CLOUDSC_SAME(r5les) CLOUDSC_SAME(r5ies)
      CLOUDSC_SAME(r5alvcp) CLOUDSC_SAME(r5alscp) CLOUDSC_SAME(ralvdcp) CLOUDSC_SAME(ralsdcp) CLOUDSC_SAME(rtwat)
      CLOUDSC_SAME(rtice) CLOUDSC_SAME(rtwat_rtice_r) CLOUDSC_SAME(rkoop1) CLOUDSC_SAME(rkoop2) CLOUDSC_SAME(ramid)
      CLOUDSC_SAME(ramin) CLOUDSC_SAME(rlmin) CLOUDSC_SAME(rcldiff) CLOUDSC_SAME(rcldiff_convi)
      CLOUDSC_SAME(rcl_inhomogaut) CLOUDSC_SAME(rcl_inhomogacc) CLOUDSC_SAME(rsnowlin1) CLOUDSC_SAME(rsnowlin2)
      CLOUDSC_SAME(rlcritsnow) CLOUDSC_SAME(rvice) CLOUDSC_SAME(rvrain) CLOUDSC_SAME(rvsnow)
      CLOUDSC_SAME(rxfallspeedrain) CLOUDSC_SAME(rcldtopcf) CLOUDSC_SAME(rdepliqrefrate)
      CLOUDSC_SAME(rdepliqrefdepth) CLOUDSC_SAME(rcl_overlapliqice) CLOUDSC_SAME(rcl_effrime) CLOUDSC_SAME(riceinit)
      CLOUDSC_SAME(rthomo) CLOUDSC_SAME(rprecrhmax) CLOUDSC_SAME(rpecons) CLOUDSC_SAME(rvrfactor)
      CLOUDSC_SAME(rcovpmin) CLOUDSC_SAME(rtaumel) CLOUDSC_SAME(rdenswat) CLOUDSC_SAME(rdensref) CLOUDSC_SAME(rcl_dr)
      CLOUDSC_SAME(rcl_x1r) CLOUDSC_SAME(rcl_x2r) CLOUDSC_SAME(rcl_x1s) CLOUDSC_SAME(rcl_lam1r)
      CLOUDSC_SAME(rcl_lam2r) CLOUDSC_SAME(rcl_lam1s) CLOUDSC_SAME(rcl_lam2s) CLOUDSC_SAME(rcl_cdenom1)
      CLOUDSC_SAME(rcl_cdenom2) CLOUDSC_SAME(rcl_cdenom3) CLOUDSC_SAME(rcl_const1r) CLOUDSC_SAME(rcl_const2r)
      CLOUDSC_SAME(rcl_const3r) CLOUDSC_SAME(rcl_const4r) CLOUDSC_SAME(rcl_const5r) CLOUDSC_SAME(rcl_const6r)
      CLOUDSC_SAME(rcl_const7r) CLOUDSC_SAME(rcl_kkaac) CLOUDSC_SAME(rcl_kkbac) CLOUDSC_SAME(rcl_kkaau)
      CLOUDSC_SAME(rcl_kkbauq) CLOUDSC_SAME(rcl_kkbaun) CLOUDSC_SAME(rcl_kk_cloud_num_sea)
      CLOUDSC_SAME(rcl_kk_cloud_num_land) CLOUDSC_SAME(rcl_fzrab) CLOUDSC_SAME(rcl_apb1) CLOUDSC_SAME(rcl_apb2)
      CLOUDSC_SAME(rcl_apb3) CLOUDSC_SAME(rcl_const1s) CLOUDSC_SAME(rcl_const2s) CLOUDSC_SAME(rcl_const3s)
      CLOUDSC_SAME(rcl_const4s) CLOUDSC_SAME(rcl_const5s) CLOUDSC_SAME(rcl_const6s) CLOUDSC_SAME(rcl_const7s)
      CLOUDSC_SAME(rcl_const8s) CLOUDSC_SAME(rmfadvw) CLOUDSC_SAME(rmfadvwdd) (q.lmfdsnow == lmfdsnow);
#undef CLOUDSC_SAME
}
template <typename R>
KPtrs<R> offset_ptrs(const KPtrs<R>& p, int64_t b0, int64_t nproma, int64_t klev) {
  const int64_t s1 = nproma, s2 = nproma * klev, sh = nproma * (klev + 1);
  KPtrs<R> q = p;
  q.pt += b0 * s2; q.pq += b0 * s2; q.tcml_t += b0 * s2; q.tcml_q += b0 * s2; q.tcml_a += b0 * s2;
  q.tcml_cld += b0 * s2 * 5; q.tloc_t += b0 * s2; q.tloc_q += b0 * s2; q.tloc_a += b0 * s2;
  q.tloc_cld += b0 * s2 * 5; q.pvfl += b0 * s2; q.pvfi += b0 * s2; q.pap += b0 * s2; q.paph += b0 * sh;
  q.plsm += b0 * s1; q.ldcum += b0 * s1; q.ktype += b0 * s1; q.peis += b0 * s1; q.plu += b0 * s2;
  q.plude += b0 * s2; q.pludeli += b0 * s2 * 4; q.psnde += b0 * s2 * 2; q.pmfu += b0 * s2; q.pmfd += b0 * s2;
  q.pa += b0 * s2; q.pclv += b0 * s2 * 5; q.pcovptot += b0 * s2; q.prainfrac_toprfz += b0 * s1;
  R** h[] = {&q.pfsqlf, &q.pfsqif, &q.pfcqnng, &q.pfcqlng, &q.pfsqrf, &q.pfsqsf, &q.pfcqrng,
             &q.pfcqsng, &q.pfsqltur, &q.pfsqitur, &q.pfplsl, &q.pfplsn, &q.pfhpsl, &q.pfhpsn};
  for (R** x : h) *x += b0 * sh;
  return q;
}

// Launch configuration per (arithmetic variant, KLEV), set by a caller or from the autotuner's records
// (include/cloudsc_tune.h): work-group size, minimum waves per SIMD of the register allocation, and whether the level
// count is compiled in.  Default: 256 columns per group, the compiler's register allocation, run-time KLEV.
namespace {
std::mutex g_tune_mutex;
std::map<std::pair<int, int>, LaunchCfg> g_tuned;
}  // namespace

template <typename R, typename RD>
constexpr int variant_id() {
  return sizeof(R) == 8 ? 0 : (sizeof(RD) == 8 ? 2 : 1);  // 0 dp, 1 sp, 2 mixed
}

// Waves-per-SIMD bounds instantiated for each variant besides 0: dp holds its state in more than 256 registers (1 wave),
// sp in 138 and mixed in 166 (3 waves each, so mixed's bound of 3 changes nothing); each gets the next occupancy steps
// that its state fits.
bool valid_wpe(int variant, int wpe) {
  if (wpe == 0) return true;
  switch (variant) {
    case 0: return wpe == 2;
    case 1: return wpe == 4;
    case 2: return wpe == 3 || wpe == 4;
    default: return false;
  }
}

bool valid_launch(int variant, const LaunchCfg& l) {
  const bool blk = l.block == 64 || l.block == 128 || l.block == 256 || l.block == 512;
  if (!blk || !valid_wpe(variant, l.wpe) || (l.kspec != 0 && l.kspec != 1)) return false;
  // register bounds and compiled-in level counts are instantiated for 128- and 256-column groups only
  return (l.wpe == 0 && l.kspec == 0) || l.block == 128 || l.block == 256;
}

LaunchCfg tuned_launch(int variant, int klev) {
  std::lock_guard<std::mutex> lk(g_tune_mutex);
  const auto it = g_tuned.find({variant, klev});
  return it == g_tuned.end() ? LaunchCfg{} : it->second;
}

void set_tuned_launch(int variant, int klev, const LaunchCfg* l) {
  std::lock_guard<std::mutex> lk(g_tune_mutex);
  if (!l)
    g_tuned.erase({variant, klev});
  else
    g_tuned[{variant, klev}] = *l;
}

// Work-groups of `block` columns.  Columns of the last block beyond NGPTOT only have their PRAINFRAC_TOPRFZ cleared (:1010);
// where they would be whole groups of a launch that fills the chip (a group on each CU), that is done apart (zero_padding):
// in the XCD order the empty groups push full ones to other XCDs.  131,072 columns in blocks of 100 are 512 groups of 256 and
// an empty one; dealt as 513, one XCD had 65 full groups and the chip ran a round for it: FP32 L137 1,430 us, 1,165
// without, mixed 1,360 and 1,155, fused mixed 2,280 and 1,695.
unsigned groups(const KDims& d, unsigned ncols, unsigned block) {
  const unsigned active = std::min(ncols, (unsigned)d.ngptot), n = (ncols + block - 1) / block;
  return n > 256u ? std::max(256u, (active + block - 1) / block) : n;
}

template <typename R>
__global__ void clear(R* x, unsigned n) {
  const unsigned i = blockIdx.x * 256u + threadIdx.x;
  if (i < n) x[i] = R(0);
}
template <typename R>
void zero_padding(const KPtrs<R>& p, unsigned ncols, unsigned ngroups, unsigned block, hipStream_t stream) {
  const unsigned done = ngroups * block;
  if (done < ncols)
    hipLaunchKernelGGL(clear<R>, dim3((ncols - done + 255) / 256), dim3(256), 0, stream, p.prainfrac_toprfz + done,
                       ncols - done);
}

template <int BLOCK, int WPE, int KL, bool SAT, typename R, typename RD, typename KC, typename KCD>
hipError_t launch_one(unsigned ncols, const KC& c, const KCD& cd, const KPtrs<R>& p, const KDims& d, int ssc_off,
                      const KSatPtrs<R>& s, hipStream_t stream) {
  const KBudPtrs<R> nb{};
  const unsigned n = groups(d, ncols, BLOCK);
  zero_padding(p, ncols, n, BLOCK, stream);
  hipLaunchKernelGGL((cloudsc_column_kernel<R, RD, KC, KCD, BLOCK, true, SAT, false, WPE, KL>), dim3(n), dim3(BLOCK), 0,
                     stream, KArgs<R, KC, KCD>{c, cd, p, d, ssc_off, s, nb});
  return hipGetLastError();
}

// Level count of the tuned instantiation: the compiled-in 137 or 91 when asked for and matching, else run time.
template <int BLOCK, int WPE, bool SAT, typename R, typename RD, typename KC, typename KCD>
hipError_t launch_kl(int kspec, unsigned ncols, const KC& c, const KCD& cd, const KPtrs<R>& p, const KDims& d,
                     int ssc_off, const KSatPtrs<R>& s, hipStream_t stream) {
  if (kspec && d.klev == 137) return launch_one<BLOCK, WPE, 137, SAT, R, RD>(ncols, c, cd, p, d, ssc_off, s, stream);
  if (kspec && d.klev == 91) return launch_one<BLOCK, WPE, 91, SAT, R, RD>(ncols, c, cd, p, d, ssc_off, s, stream);
  return launch_one<BLOCK, WPE, 0, SAT, R, RD>(ncols, c, cd, p, d, ssc_off, s, stream);
}

// FP64 takes more than 256 registers, so one wave to a SIMD; bounded to 256, with some 20 words spilled, two fit.  That
// pays as soon as the launch has more waves than the chip has SIMDs (4 x 256): 66,000 columns x L137 2.96 -> 2.43 ms,
// 131,072 3.00 -> 2.63, 200,000 5.84 -> 5.12, with run-time constants 3.04 -> 2.74, 3.12 -> 2.95 and 6.07 -> 5.71, but
// 65,536 (a wave to each SIMD) 1.56 -> 1.84 ms.  Fused with the saturation adjustment it spills 100 and more and loses
// everywhere: 66,000 columns 4.00 -> 4.13 ms, 131,072 4.10 -> 4.61, 200,000 7.92 -> 8.54, with run-time constants 3.99 ->
// 4.66, 4.20 -> 5.31 and 8.08 -> 9.98.
template <typename R, typename RD>
constexpr bool is_fp64 = std::is_same<R, double>::value && std::is_same<RD, double>::value;
inline bool two_waves(const LaunchCfg& l, const KDims& d, unsigned ncols) {
  return l.scope < 2 && std::min(ncols, (unsigned)d.ngptot) > 64u * 4u * 256u;  // lanes of padding columns end at once
}

template <int BLOCK, bool SAT, typename R, typename RD, typename KC, typename KCD>
hipError_t launch_wpe(const LaunchCfg& l, unsigned ncols, const KC& c, const KCD& cd, const KPtrs<R>& p,
                      const KDims& d, int ssc_off, const KSatPtrs<R>& s, hipStream_t stream) {
  constexpr int v = variant_id<R, RD>();
  constexpr int w1 = v == 0 ? 2 : (v == 1 ? 4 : 3);
  constexpr int w2 = 4;  // mixed only
  if (l.wpe == w1 || (is_fp64<R, RD> && l.wpe == 0 && two_waves(l, d, ncols)))
    return launch_kl<BLOCK, w1, SAT, R, RD>(l.kspec, ncols, c, cd, p, d, ssc_off, s, stream);
  if constexpr (v == 2)
    if (l.wpe == w2) return launch_kl<BLOCK, w2, SAT, R, RD>(l.kspec, ncols, c, cd, p, d, ssc_off, s, stream);
  return launch_kl<BLOCK, 0, SAT, R, RD>(l.kspec, ncols, c, cd, p, d, ssc_off, s, stream);
}

template <bool SAT, typename R, typename RD, typename KC, typename KCD>
hipError_t launch_variant(const LaunchCfg& l, bool uni, unsigned ncols, const KC& c, const KCD& cd,
                          const KPtrs<R>& p, const KDims& d, int ssc_off, const KSatPtrs<R>& s, hipStream_t stream) {
  const KBudPtrs<R> nb{};
  if (!uni) {  // blocks not aligned to waves: per-lane block offsets, 256-lane groups
    const unsigned n = groups(d, ncols, 256);
    zero_padding(p, ncols, n, 256, stream);
    if constexpr (is_fp64<R, RD> && !SAT) {
      if (two_waves(l, d, ncols)) {
        hipLaunchKernelGGL((cloudsc_column_kernel<R, RD, KC, KCD, 256, false, SAT, false, 2>), dim3(n), dim3(256), 0, stream,
                           KArgs<R, KC, KCD>{c, cd, p, d, ssc_off, s, nb});
        return hipGetLastError();
      }
    }
    hipLaunchKernelGGL((cloudsc_column_kernel<R, RD, KC, KCD, 256, false, SAT, false>), dim3(n), dim3(256), 0, stream,
                       KArgs<R, KC, KCD>{c, cd, p, d, ssc_off, s, nb});
    return hipGetLastError();
  }
  // the tuned instantiations (register bound, compiled-in KLEV) exist for the default configuration of CLOUDSC
  constexpr bool tuned = !SAT && std::is_same<KC, KConstDefault<R>>::value;
  switch (l.block) {
    case 64:
      return launch_one<64, 0, 0, SAT, R, RD>(ncols, c, cd, p, d, ssc_off, s, stream);
    case 128:
      if constexpr (tuned) return launch_wpe<128, SAT, R, RD>(l, ncols, c, cd, p, d, ssc_off, s, stream);
      return launch_one<128, 0, 0, SAT, R, RD>(ncols, c, cd, p, d, ssc_off, s, stream);
    case 512:
      return launch_one<512, 0, 0, SAT, R, RD>(ncols, c, cd, p, d, ssc_off, s, stream);
    default:
      if constexpr (tuned) return launch_wpe<256, SAT, R, RD>(l, ncols, c, cd, p, d, ssc_off, s, stream);
      if constexpr (is_fp64<R, RD> && !SAT)
        if (two_waves(l, d, ncols)) return launch_one<256, 2, 0, SAT, R, RD>(ncols, c, cd, p, d, ssc_off, s, stream);
      return launch_one<256, 0, 0, SAT, R, RD>(ncols, c, cd, p, d, ssc_off, s, stream);
  }
}

// Launches with fewer waves than the chip has SIMDs (1,024) take the time of one wave, whatever their size; three waves to
// 64 columns then cut it.  The line lies where the work-groups no longer all run at once: LDS holds 3 of them on a CU in
// FP32, 1 in FP64.  FP32 x L137 in blocks of 128: 16,384 columns 515 -> 321 us, 32,768 532 -> 366, 49,152 547 -> 410, but
// 50,000 559 -> 713.  Blocks that are no multiple of 64 columns are slower there: of 42 kinds of launch (FP32, mixed, fused,
// run-time constants; L91, L137; blocks of 32, 75, 100) all gain at 45,000 columns, from 0 to 2 % (FP32 x L137, blocks of
// 32 and 75, 700 -> 677 us) to 30 % (FP32 x L91, blocks of 100 434 -> 334, blocks of 32 459 -> 364), but at 49,000 those x
// L91 gain or lose 5 % (FP32, blocks of 100 440 -> 426, blocks of 75 469 -> 491), so the line is at 704 groups there.
// Mixed 2,048 in blocks of 32 491 -> 328 us.  FP64 16,384 x L137 1.45 -> 0.84 ms.  Fused with the saturation adjustment:
// FP32 2,048 652 -> 393 us, 49,152 761 -> 657; mixed 10,000 780 -> 474 us; FP64 16,000 1.88 -> 1.17 ms.
// A launch that a caller has set (cloudsc_tune_set_launch) is one of the one-wave kernel at every size.
template <typename R>
bool pipelined(const LaunchCfg& l, unsigned ncols, bool uni) {
  return l.scope < 2 && ncols <= 64u * 256u * (sizeof(R) == 8 ? 1u : 3u) && (uni || ncols <= 45056u);
}

template <typename R, typename RD, typename KC, typename KCD>
hipError_t launch_either(bool sat, const LaunchCfg& l, bool uni, unsigned ncols, const KC& c, const KCD& cd,
                         const KPtrs<R>& p, const KDims& d, int ssc_off, const KSatPtrs<R>& s,
                         const KBudPtrs<R>* bud, hipStream_t stream) {
  if (bud) {  // budget-instrumented kernel: one instantiation per variant (diagnostic runs); one wave per group
    hipLaunchKernelGGL((cloudsc_column_kernel<R, RD, KC, KCD, 64, false, false, true>), dim3((ncols + 63) / 64),
                       dim3(64), 0, stream, KArgs<R, KC, KCD>{c, cd, p, d, ssc_off, s, *bud});
    return hipGetLastError();
  }
  if (pipelined<R>(l, ncols, uni)) {
    const KBudPtrs<R> nb{};
    auto* kernel = sat ? (uni ? cloudsc_pipeline_kernel<R, RD, KC, KCD, true, true>
                              : cloudsc_pipeline_kernel<R, RD, KC, KCD, false, true>)
                       : (uni ? cloudsc_pipeline_kernel<R, RD, KC, KCD, true, false>
                              : cloudsc_pipeline_kernel<R, RD, KC, KCD, false, false>);
    const unsigned n = groups(d, ncols, 64);
    zero_padding(p, ncols, n, 64, stream);
    hipLaunchKernelGGL(kernel, dim3(n), dim3(192), 0, stream,
                       KArgs<R, KC, KCD>{c, cd, p, d, ssc_off, s, nb});
    return hipGetLastError();
  }
  return sat ? launch_variant<true, R, RD>(l, uni, ncols, c, cd, p, d, ssc_off, s, stream)
             : launch_variant<false, R, RD>(l, uni, ncols, c, cd, p, d, ssc_off, s, stream);
}

template <typename R>
KSatPtrs<R> offset_sat_ptrs(const KSatPtrs<R>& p, int64_t b0, int64_t nproma, int64_t klev) {
  const int64_t s2 = nproma * klev;
  KSatPtrs<R> q = p;
  q.phrsw += b0 * s2; q.phrlw += b0 * s2; q.tvdf_t += b0 * s2; q.tvdf_q += b0 * s2; q.pvervel += b0 * s2;
  q.tcml_t += b0 * s2; q.tcml_q += b0 * s2; q.tcml_a += b0 * s2; q.tcml_cld += b0 * s2 * 5;
  if (q.tsat_t) {
    q.tsat_t += b0 * s2; q.tsat_q += b0 * s2; q.tsat_a += b0 * s2; q.tsat_cld += b0 * s2 * 5;
  }
  return q;
}

template <typename R>
KBudPtrs<R> offset_bud_ptrs(const KBudPtrs<R>& p, int64_t b0, int64_t nproma, int64_t klev) {
  const int64_t s2 = nproma * klev;
  KBudPtrs<R> q = p;
  auto adv = [](auto*& x, int64_t n) {  // arrays of a diagnostic that is off are NULL
    if (x) x += n;
  };
  adv(q.pvfa, b0 * s2); adv(q.pdyna, b0 * s2); adv(q.pdynl, b0 * s2); adv(q.pdyni, b0 * s2);
  adv(q.pdyns, b0 * s2); adv(q.phrsw, b0 * s2); adv(q.phrlw, b0 * s2); adv(q.pvfl, b0 * s2); adv(q.pvfi, b0 * s2);
  adv(q.kpbltype, b0 * nproma); adv(q.kctop, b0 * nproma);
  adv(q.pextra, b0 * s2 * q.kfldx);
  adv(q.pgaw, b0 * nproma); adv(q.pfsd, b0 * s2);
  return q;
}

template <typename R, typename RD>
hipError_t launch_cloudsc(const cloudsc_params_t& q, double ptsphy, const KPtrs<R>& p, const KDims& d, int ssc_off,
                          hipStream_t stream, const KSatPtrs<R>* sat, const KBudPtrs<R>* bud) {
  const bool def = is_default_config(q);
  const LaunchCfg tl = def ? tuned_launch(variant_id<R, RD>(), d.klev) : LaunchCfg{};
  // every wave inside one block (64-lane waves, 64 | NPROMA): block offsets are uniform across the wave
  const bool uni = d.nproma % 64 == 0;
  // blocks per launch: the largest array, (NPROMA,KLEV,5) or PEXTRA (NPROMA,KLEV,KFLDX), stays below 4 GiB
  const int64_t nfld = bud ? std::max<int64_t>(5, bud->kfldx) : 5;
  const int64_t per_block = (int64_t)d.nproma * d.klev * nfld * (int64_t)sizeof(R);
  const int64_t max_blocks = std::max<int64_t>(1, ((int64_t)1 << 32) / per_block - 1);
  // launches of equal size: a short last launch would leave most of the GPU idle while it runs
  const int64_t nlaunch = (d.ngpblks + max_blocks - 1) / max_blocks;
  const int64_t step = (d.ngpblks + nlaunch - 1) / nlaunch;
  for (int64_t b0 = 0; b0 < d.ngpblks; b0 += step) {
    const int64_t nb = std::min<int64_t>(step, d.ngpblks - b0);
    KDims dc = d;
    dc.ngpblks = (int32_t)nb;
    dc.ngptot = (int32_t)(d.ngptot - b0 * d.nproma);
    const KPtrs<R> pc = offset_ptrs(p, b0, d.nproma, d.klev);
    const KSatPtrs<R> sc = sat ? offset_sat_ptrs(*sat, b0, d.nproma, d.klev) : KSatPtrs<R>{};
    const KBudPtrs<R> bc = bud ? offset_bud_ptrs(*bud, b0, d.nproma, d.klev) : KBudPtrs<R>{};
    const unsigned ncols = (unsigned)(nb * d.nproma);
    hipError_t e;
    if (def) {
      const KConstDefault<R> c = make_kconst_default<R>(q, ptsphy);
      const KConstDefault<RD> cd = make_kconst_default<RD>(q, ptsphy);
      e = launch_either<R, RD>(sat != nullptr, tl, uni, ncols, c, cd, pc, dc, ssc_off, sc, bud ? &bc : nullptr,
                               stream);
    } else {
      const KConst<R> c = make_kconst<R>(q, ptsphy);
      const KConst<RD> cd = make_kconst<RD>(q, ptsphy);
      e = launch_either<R, RD>(sat != nullptr, LaunchCfg{}, uni, ncols, c, cd, pc, dc, ssc_off, sc,
                               bud ? &bc : nullptr, stream);
    }
    if (e != hipSuccess) return e;
  }
  return hipSuccess;
}

template KConst<float> make_kconst<float>(const cloudsc_params_t&, double);
template KConst<double> make_kconst<double>(const cloudsc_params_t&, double);
template KConstDefault<float> make_kconst_default<float>(const cloudsc_params_t&, double);
template KConstDefault<double> make_kconst_default<double>(const cloudsc_params_t&, double);

template hipError_t launch_cloudsc<double, double>(const cloudsc_params_t&, double, const KPtrs<double>&,
                                                   const KDims&, int, hipStream_t, const KSatPtrs<double>*,
                                                   const KBudPtrs<double>*);
template hipError_t launch_cloudsc<float, float>(const cloudsc_params_t&, double, const KPtrs<float>&, const KDims&,
                                                 int, hipStream_t, const KSatPtrs<float>*, const KBudPtrs<float>*);
template hipError_t launch_cloudsc<float, double>(const cloudsc_params_t&, double, const KPtrs<float>&, const KDims&,
                                                  int, hipStream_t, const KSatPtrs<float>*, const KBudPtrs<float>*);

}  // namespace cloudsc_gpu
