// Batched FP64 isobaric-reactor chemistry on gfx950: net production rates, RHS, and the exact analytic
// Jacobian (griffon's option-0 sensitivities + isobaric transform), one workgroup per S states.
//
// Math restated from the reference: thermodynamics_kernels.cpp:45-351 (NASA7 cp, dcp/dT, h),
// chemistry_kernels.cpp:35-463 (production rates), rates_sensitivities_exact.cpp:33-1028 (exact
// sensitivities), isobaric_reactor_kernels.cpp:19-98, 319-343 (RHS, primitive Jacobian, transform).
//
// Structure: persistent workgroups (LDS-limited), each owning a contiguous range of states processed S at
// a time. The compact gather tables of the mechanism are copied into LDS once per workgroup; all
// per-state intermediates live in LDS; no atomics, so results are deterministic:
//   P0  one wave per state, lane = species: mixture thermo; wave-shuffle reductions for sum(y/M), cp, dcp/dT
//   P1  lane = (reaction, state), a reaction's S states in adjacent lanes: kf, Kc, falloff factor, mass
//       action and all partial derivatives.
//       dq_r/dY_s = sum_p v_{r,p} delta(s,p) + a_r (1/M_s - 1/M_last) + b_r, so each reaction stores five
//       scalars (q, dq/drho, dq/dT, a, b) and one value v per participant slot.
//   P2  lane = (species k, state): gathers over the reactions with k in their net
//       stoichiometry give w_k, dw_k/drho, dw_k/dT, the rank-1 coefficients and the diagonal sensitivity
//       entry of column k; then one wave per state, lane = species: wave reductions give the enthalpy-weighted sums;
//       the RHS is written here.
//   P3  one wave per Jacobian column, lane = row (plus one lane for the last species), looping over the S
//       states: off-diagonal sparse gather + rank-1 part give the species rows (chem_jac_isobaric + the
//       (rho,T,Y)->(T,Y) transform at constant pressure); the temperature row is the enthalpy-weighted
//       wave sum of the column; each column of each state is one contiguous 53-double store.
//
// What bounds it is latency, with few wavefronts: the Jacobian kernel's state (28 KB of LDS a state, 256 registers) leaves room
// for eight waves per compute unit, the rates' registers for twelve (held to 168: at 186 they were eight and
// 100,003 states took 1,033 us instead of 803). The Jacobian's are held to 256: with six more, small mechanisms, whose LDS has
// room for two workgroups of 256 threads, had one of them (4,000 states of 10 species 73 us instead of 48). The states of
// a group are interleaved in LDS, so that neighbouring lanes read
// neighbouring words, and a reaction's record is read whole, its short lists unrolled with factors of one beyond their
// ends: field by field, with loops of one to four trips around dependent loads, P1 took 41,000 cycles for a group
// of four states with derivatives and now takes 32,000. 53 species, 325 reactions, before and after (us): RHS of 512 / 7,600 /
// 100,003 states 16.5 / 85 / 880 -> 14.7 / 78 / 795; with Jacobian 512 / 4,000 / 100,000 38 / 169 / 3,938 -> 31 / 138 / 3,196.
// Of the latter, P3: the blocks' offsets instead of pointers that may be null (those were stored through as flat addresses,
// which every later LDS load waits for) 3,572 -> 3,429, and what only lane 0 needs read by all lanes ahead of a column's
// sums instead of under its condition, four times 200 cycles a column, -> 3,196.
// Tried without gain: P3's slot sums dealt to the lanes by length through LDS (every lane busy, but the same words through
// the banks again: 38,000 -> 45,000 cycles a group); 16 waves at 128 registers (226 spilled).
#include "gf_internal.h"
#include "gf_thermo.h"
#include "../../include/griffon_amd.h"

#include <algorithm>
#include <cstdlib>
#include <cstring>

namespace gfa {

namespace {

constexpr int SP_STRIDE = NS_MAX;   // per-species LDS arrays
constexpr int N_SPEC_ARR = 12;      // y h cpi G dBdT w ws0 ws1 A B pr DG
constexpr int N_SPEC_ARR_RHS = 4;   // the RHS-only kernel keeps y h cpi G
constexpr int N_SCAL = 16;

enum { Y_ = 0, H_, CPI_, G_, DBDT_, W_, WS0_, WS1_, A_, B_, PR_, DG_ };
enum { S_T = 0, S_RHO, S_MMW, S_CP, S_CPST, S_INVT, S_LOGT, S_CT, S_INVM, S_LOGPORT, S_RHS0, S_HS0, S_HS1, S_WCP,
       S_HA, S_HB };

using ChemArgs = ChemIO;

// one DPP step of the wave scan: v + (the value of lane l - shift), 0 where no such lane (old value 0)
template <int CTRL, int ROWMASK>
__device__ __forceinline__ double dpp_add(double v) {
  const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(v), CTRL, ROWMASK, 0xF, false);
  const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(v), CTRL, ROWMASK, 0xF, false);
  return v + __hiloint2double(hi, lo);
}

// Sum over the 64 lanes, the same value returned to every lane: an inclusive scan by DPP row shifts and row
// broadcasts (no LDS traffic), read from lane 63. The summation order is fixed, so results are reproducible.
__device__ __forceinline__ double wave_sum(double v) {
  v = dpp_add<0x111, 0xF>(v);  // row_shr:1
  v = dpp_add<0x112, 0xF>(v);  // row_shr:2
  v = dpp_add<0x114, 0xF>(v);  // row_shr:4
  v = dpp_add<0x118, 0xF>(v);  // row_shr:8
  v = dpp_add<0x142, 0xA>(v);  // row_bcast:15
  v = dpp_add<0x143, 0xC>(v);  // row_bcast:31
  return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(v), 63),
                          __builtin_amdgcn_readlane(__double2loint(v), 63));
}

// Swaps of 32-bit halves between two lane groups, applied to both words of a double: with 32, the upper 32
// lanes of a with the lower 32 lanes of b; with 16, the odd 16-lane rows of a with the even rows of b.
template <int W>
__device__ __forceinline__ void lane_swap(double &a, double &b) {
  const auto hi = W == 32 ? __builtin_amdgcn_permlane32_swap(__double2hiint(a), __double2hiint(b), false, false)
                          : __builtin_amdgcn_permlane16_swap(__double2hiint(a), __double2hiint(b), false, false);
  const auto lo = W == 32 ? __builtin_amdgcn_permlane32_swap(__double2loint(a), __double2loint(b), false, false)
                          : __builtin_amdgcn_permlane16_swap(__double2loint(a), __double2loint(b), false, false);
  a = __hiloint2double((int)hi[0], (int)lo[0]);
  b = __hiloint2double((int)hi[1], (int)lo[1]);
}

// Sums over the 64 lanes of four vectors at once, returned to every lane. Lanes l and l + 32 are added
// (two vectors per register after a 32-lane swap), then rows r and r + 1 (four vectors per register after a
// 16-lane swap), then the 16 lanes of each row by a DPP scan. Each vector is summed by the same tree whatever
// its position (every pairwise sum is commutative), so a vector's sum does not depend on what the other three
// hold; about a third of the instructions of four separate wave sums.
__device__ __forceinline__ void wave_sum4(const double (&v)[4], double (&out)[4]) {
  double a0 = v[0], b0 = v[1], a1 = v[2], b1 = v[3];
  lane_swap<32>(a0, b0);  // a0 = [v0 lanes 0-31 | v1 lanes 0-31], b0 = [v0 lanes 32-63 | v1 lanes 32-63]
  lane_swap<32>(a1, b1);
  double p = a0 + b0, q = a1 + b1;  // p: v0 in lanes 0-31, v1 in lanes 32-63; q likewise v2, v3
  lane_swap<16>(p, q);              // p = rows (p0, q0, p2, q2), q = rows (p1, q1, p3, q3)
  double t = p + q;                 // rows hold v0, v2, v1, v3
  t = dpp_add<0x111, 0xF>(t);       // row_shr:1
  t = dpp_add<0x112, 0xF>(t);       // row_shr:2
  t = dpp_add<0x114, 0xF>(t);       // row_shr:4
  t = dpp_add<0x118, 0xF>(t);       // row_shr:8: lane 15 of each row holds the row's sum
  const int src[4] = {15, 47, 31, 63};
#pragma unroll
  for (int k = 0; k < 4; ++k)
    out[k] = __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(t), src[k]),
                              __builtin_amdgcn_readlane(__double2loint(t), src[k]));
}

__device__ __forceinline__ double arrh(const double *k, double logT, double invT) {
  return k[0] * exp(k[1] * logT - k[2] * invT);
}
__device__ __forceinline__ double arrh_sens_over_k(const double *k, double invT) { return invT * (k[1] + k[2] * invT); }

__device__ __forceinline__ double kf_of(const DevRxn &R, double T, double logT, double invT) {
  switch (R.kForm) {
    case KF_CONSTANT: return R.kf[0];
    case KF_LINEAR: return R.kf[0] * T;
    case KF_QUADRATIC: return R.kf[0] * T * T;
    case KF_RECIPROCAL: return R.kf[0] * invT;
    default: return arrh(R.kf, logT, invT);
  }
}

__device__ __forceinline__ double ipow3(double c, int st) {  // c^st for st in 1..3
  return st == 1 ? c : (st == 2 ? c * c : c * c * c);
}

__device__ __forceinline__ double troe_fcent(const DevRxn &R, double T, double invT, double &dfdT) {
  const double *t = R.troe;
  double f = 0., d = 0.;
  const int tf = R.troeForm;
  const bool has1 = (tf == TF_T1 || tf == TF_T12 || tf == TF_T13 || tf == TF_T123);
  const bool has2 = (tf == TF_T2 || tf == TF_T12 || tf == TF_T23 || tf == TF_T123);
  const bool has3 = (tf == TF_T3 || tf == TF_T13 || tf == TF_T23 || tf == TF_T123);
  if (has1) { const double e = exp(-T / t[1]); f += (1 - t[0]) * e; d += (t[0] - 1) / t[1] * e; }
  if (has2) { const double e = exp(-T / t[2]); f += t[0] * e; d += -t[0] / t[2] * e; }
  if (has3) { const double e = exp(-invT * t[3]); f += e; d += e * t[3] * invT * invT; }
  dfdT = d;
  return f;
}

template <int S, int THREADS, bool JAC>
__global__ void __launch_bounds__(THREADS) __attribute__((amdgpu_waves_per_eu(JAC ? 2 : 3))) chem_kernel(MechView mv, ChemArgs a, long groups_per_wg) {
  static_assert(S >= 1 && S <= 4, "the temperature-row sums take at most four states at once");
  extern __shared__ double lds[];
  const int ns = mv.ns, nr = mv.nr, nm = ns - 1;
  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  constexpr int NSA = JAC ? N_SPEC_ARR : N_SPEC_ARR_RHS;
  const long ngroups = (a.n + S - 1) / S;
  // each workgroup owns a contiguous range of state groups (neighbouring states share SoA input lines)
  const long g0 = (long)blockIdx.x * groups_per_wg;
  const long g1 = min(ngroups, g0 + groups_per_wg);

  // gather tables -> LDS (the RHS-only kernel needs only the species gather)
  const int tcopy = JAC ? mv.tbl_bytes : ((mv.exo_at + 15) & ~15);
  for (int q = threadIdx.x; q < tcopy / 16; q += THREADS)
    reinterpret_cast<uint4 *>(lds)[q] = reinterpret_cast<const uint4 *>(mv.tbl)[q];
  const char *tb = reinterpret_cast<const char *>(lds);
  const uint32_t *sgx_off = reinterpret_cast<const uint32_t *>(tb);
  const uint64_t *sgx = reinterpret_cast<const uint64_t *>(tb + mv.sgx_at);
  const uint16_t *exo = reinterpret_cast<const uint16_t *>(tb + mv.exo_at);
  const uint32_t *exx = reinterpret_cast<const uint32_t *>(tb + mv.exx_at);
  const double *tbe = reinterpret_cast<const double *>(tb + mv.tbe_at);  // third-body lists and 1/M in LDS
  const int *tbi = reinterpret_cast<const int *>(tb + mv.tbi_at);
  const int *tbsl = reinterpret_cast<const int *>(tb + mv.tbs_at);
  const double *imw = reinterpret_cast<const double *>(tb + mv.imw_at);
  // a group's S states are interleaved: entry e of state s at e * S + s
  double *sbase = lds + tcopy / 8;
  auto SP = [&](int array, int k, int s) -> double & { return sbase[(array * SP_STRIDE + k) * S + s]; };
  auto SC = [&](int e, int s) -> double & { return sbase[(NSA * SP_STRIDE + e) * S + s]; };
  double *rqb = sbase + (NSA * SP_STRIDE + N_SCAL) * S;  // per reaction: rate and its derivatives
  double *vb = rqb + 5L * nr * S;                       // per slot
  __syncthreads();

  for (long group = g0; group < g1; ++group) {
    const long first = group * S;

    // ---------------- P0: mixture thermo (wave per state, lane = species) ----------------
    if (wave < S) {
      const long il = first + wave;
      if (il < a.n) {
        const long i = a.sel ? (long)a.sel[il] : il;
        const double *xi = a.x + i * a.xs_i;
        const double T = xi[0];
        double yk = 0.;
        if (a.rho_given == 1) {
          if (lane < ns) yk = xi[(1 + lane) * a.xs_v];
        } else {
          if (lane < nm) yk = xi[(1 + lane) * a.xs_v];
          const double sy = wave_sum(yk);
          if (lane == nm) yk = 1. - sy;
        }
        const double mm = wave_sum(lane < ns ? yk * mv.invmw[lane] : 0.);
        const double mmw = 1. / mm;
        const double invT = 1. / T, logT = log(T);
        const double rho = a.rho_given ? a.p[i * a.ps] : a.p[i * a.ps] * mmw / (T * mv.Ru);
        double cp = 0., cps = 0., h = 0., Gk = 0., dB = 0.;
        if (lane < ns) species_thermo(mv, lane, T, logT, invT, cp, cps, h, Gk, dB);
        if (lane < ns) {
          SP(Y_, lane, wave) = yk;
          SP(H_, lane, wave) = h;
          SP(CPI_, lane, wave) = cp;
          SP(G_, lane, wave) = Gk;
          if (JAC) SP(DBDT_, lane, wave) = dB;
        }
        const double cpm = wave_sum(lane < ns ? yk * cp : 0.);
        // a constant-cp species resets the dcp/dT accumulation (thermodynamics_kernels.cpp:200-203)
        const double cpsm = wave_sum((lane < ns && lane > mv.last_const) ? yk * cps : 0.);
        if (a.aux && lane < 4) a.aux[i * 4 + lane] = lane == 0 ? rho : (lane == 1 ? cpm : (lane == 2 ? cpsm : mmw));
        if (a.cpi && lane < ns) a.cpi[i * ns + lane] = cp;
        if (a.hsp && lane < ns) a.hsp[i * ns + lane] = h;
        if (lane == 0) {
          SC(S_T, wave) = T; SC(S_RHO, wave) = rho; SC(S_MMW, wave) = mmw; SC(S_CP, wave) = cpm; SC(S_CPST, wave) = cpsm;
          SC(S_INVT, wave) = invT; SC(S_LOGT, wave) = logT; SC(S_CT, wave) = rho * mm; SC(S_INVM, wave) = mm;
          SC(S_LOGPORT, wave) = log(mv.pref * invT * mv.invRu);
        }
      }
    }
    __syncthreads();

    // ---------------- P1: reactions (lane = (reaction, state); a reaction's S states are adjacent lanes) -------
    for (int it = threadIdx.x; it < S * nr; it += THREADS) {
      const int r = it / S, s = it - r * S;
      const long i = first + s;
      if (i >= a.n) continue;
      auto y = [&](int k) { return SP(Y_, k, s); };
      auto rq = [&](int e) -> double & { return rqb[e * S + s]; };
      const double T = SC(S_T, s), rho = SC(S_RHO, s), invT = SC(S_INVT, s), logT = SC(S_LOGT, s), ct = SC(S_CT, s),
                   invM = SC(S_INVM, s);
      const DevRxn R = mv.rx[r];  // the whole record at once; arrays in it are indexed by constants below
      const double kf = kf_of(R, T, logT, invT);

      // third-body / falloff multiplier
      double tbsum = 0.;
      for (int q = 0; q < R.n_tb; q += 4) {  // four at a time, so that their loads overlap; missing ones add zero
        double e[4], ye[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          const int at = R.tb_off + min(q + u, R.n_tb - 1);
          e[u] = tbe[at];
          ye[u] = y(tbi[at]);
        }
#pragma unroll
        for (int u = 0; u < 4; ++u) tbsum = q + u < R.n_tb ? fma(e[u], ye[u], tbsum) : tbsum;
      }
      // concentration factors of the reactants and products (1 beyond the list), and the net Gibbs function
      double C[NRC_MAX], F[NRC_MAX], Cp[NPD_MAX], Fp[NPD_MAX], sg = 0., sb = 0.;
      if (!R.hasOrders) {
#pragma unroll
        for (int j = 0; j < NRC_MAX; ++j) {
          C[j] = y(R.rc_idx[j]) * rho * imw[R.rc_idx[j]];
          F[j] = j < R.n_rc ? ipow3(C[j], R.rc_st[j]) : 1.;
        }
        if (R.reversible) {
#pragma unroll
          for (int j = 0; j < NPD_MAX; ++j) {
            Cp[j] = y(R.pd_idx[j]) * rho * imw[R.pd_idx[j]];
            Fp[j] = j < R.n_pd ? ipow3(Cp[j], R.pd_st[j]) : 1.;
          }
#pragma unroll
          for (int q = 0; q < NNET_MAX; ++q) {
            const double g = SP(G_, R.net_idx[q], s);
            sg = q < R.n_net ? fma(R.net_st[q], g, sg) : sg;
            if (JAC) {
              const double d = SP(DBDT_, R.net_idx[q], s);
              sb = q < R.n_net ? fma(R.net_st[q], d, sb) : sb;
            }
          }
        }
      }

      if (!JAC) {
        // production_rates formulation (chemistry_kernels.cpp:140-461)
        double k = kf, kr = 0.;
        const double M = R.baseEff * ct + rho * tbsum;
        if (R.type == RK_THIRD_BODY) {
          k *= M;
        } else if (R.type == RK_LINDEMANN) {
          k /= (1 + k / (arrh(R.kp, logT, invT) * M));
        } else if (R.type == RK_TROE) {
          const double pr = arrh(R.kp, logT, invT) / k * M;
          double dd;
          const double logFc = log10(troe_fcent(R, T, invT, dd));
          const double logPrC = log10(fmax(pr, 1.e-300)) + (-0.4 - 0.67 * logFc);
          const double F1 = logPrC / ((0.75 - 1.27 * logFc) - 0.14 * logPrC);
          k = k * pow(10., logFc / (1 + F1 * F1)) * pr / (1 + pr);
        }
        if (R.hasOrders) {
#pragma unroll 1
          for (int q = 0; q < R.n_sp; ++q) {
            const int sidx = mv.sp_idx[R.sp_off + q];
            k *= pow(fmax(y(sidx) * rho * mv.sp_invmw[R.sp_off + q], 0.), mv.sp_ord[R.sp_off + q]);
          }
        } else {
          if (R.reversible) kr = k * exp(R.sumStoich * SC(S_LOGPORT, s) - invT * mv.invRu * sg);
#pragma unroll
          for (int j = 0; j < NRC_MAX; ++j) k *= F[j];
          if (R.reversible) {
#pragma unroll
            for (int j = 0; j < NPD_MAX; ++j) kr *= Fp[j];
          }
        }
        rq(r) = k - kr;
        continue;
      }

      double Ctbaf = 1., dCdrho = 0., dCdT = 0., cdense = 0., tbs = 0.;
      double qaC = 0.;  // d(q)/d(ln A) = Rnet * qaC; A is the forward (high-pressure) pre-exponential
      if (R.type == RK_THIRD_BODY) {
        Ctbaf = R.baseEff * ct + rho * tbsum;
        dCdrho = R.baseEff * invM + tbsum;
        cdense = rho * R.baseEff;
        tbs = rho;
      } else if (R.type == RK_LINDEMANN || R.type == RK_TROE) {
        const double flf = R.baseEff * ct + rho * tbsum;
        const double kpk = arrh(R.kp, logT, invT) / kf;
        const double pr = kpk * flf;
        const double dlnk = arrh_sens_over_k(R.kp, invT) - arrh_sens_over_k(R.kf, invT);
        double nsT;
        if (R.type == RK_LINDEMANN) {
          Ctbaf = pr / (1. + pr);
          dCdT = Ctbaf / (1. + pr) * dlnk;
          nsT = kpk / ((1. + pr) * (1. + pr));
        } else {  // rates_sensitivities_exact.cpp:905-995
          double dfc;
          const double fc = troe_fcent(R, T, invT, dfc);
          const double l10pr = log10(fmax(pr, 1.e-300));
          const double l10fc = log10(fmax(fc, 1.e-300));
          const double lfc = log(fmax(fc, 1.e-300));
          const double ln10 = 2.302585092994045684;  // log(10)
          const double aT = l10pr - 0.67 * l10fc - 0.4;
          const double bT = -0.14 * l10pr - 1.1762 * l10fc + 0.806;
          const double gT = 1 / (1 + (aT / bT) * (aT / bT));
          const double fT = pow(fc, gT);
          Ctbaf = fT * pr / (1 + pr);
          const double dfTdT = fT * (gT / fc * dfc + lfc * (-2.0 * gT * gT / ln10 * aT / (bT * bT * bT) *
                                                              ((bT + 0.14 * aT) * dlnk - (0.67 * bT - 1.1762 * aT) * dfc / fc)));
          dCdT = 1. / (1. + 1. / pr) * dfTdT + fT * pr / ((1. + pr) * (1. + pr)) * dlnk;
          nsT = kpk * (-2.0 / (1. + pr) * fT * lfc * gT * gT / ln10 * aT / (bT * bT * bT) * (bT + 0.14 * aT) +
                       fT / ((1. + pr) * (1 + pr)));
        }
        dCdrho = nsT * R.baseEff * invM + nsT * tbsum;
        cdense = nsT * rho * R.baseEff;
        tbs = nsT * rho;
        // Pr = k0 [M] / kinf: d ln(q) / d ln(kinf) = 1 - (Pr / Ctbaf) dCtbaf/dPr, and nsT = (k0 / kinf) dCtbaf/dPr
        qaC = Ctbaf - flf * nsT;
      }

      if (a.notbaf) {  // rates_sensitivity_option 1: no derivatives of the third-body / falloff multiplier
        dCdrho = 0.;
        dCdT = 0.;
        cdense = 0.;
        tbs = 0.;
      }
      auto vr = [&](int q) -> double & { return vb[(R.slot_off + q) * S + s]; };
      for (int q = 0; q < R.n_slot; ++q) vr(q) = 0.;
      double Rnet, dRdrho, dRdT, U = 0.;
      const double ksens = arrh_sens_over_k(R.kf, invT);
      if (R.hasOrders) {  // rates_sensitivities_exact.cpp:198-281
        auto conc = [&](int q) { return y(mv.sp_idx[R.sp_off + q]) * rho * mv.sp_invmw[R.sp_off + q]; };
        auto order = [&](int q) { return mv.sp_ord[R.sp_off + q]; };
        Rnet = kf;
        double sumO = 0.;
#pragma unroll 1
        for (int q = 0; q < R.n_sp; ++q) {
          Rnet *= pow(fmax(conc(q), 0.), order(q));
          sumO += order(q);
        }
        dRdrho = Rnet / ct * invM * sumO;
        dRdT = Rnet * ksens;
#pragma unroll 1
        for (int j = 0; j < R.n_sp; ++j) {
          const double im = mv.sp_invmw[R.sp_off + j];
          const bool last = (mv.sp_idx[R.sp_off + j] == ns - 1);
          double m = kf;
#pragma unroll 1
          for (int l = 0; l < R.n_sp; ++l) {
            const double o = order(l), cl = conc(l);
            // of its own species the derivative o C^(o-1), of the others the factor itself
            const bool own = l == j, inv = own && !(last || o > 1);
            const double f = pow(own ? fmax(cl, 1.e-16) : last ? cl : fmax(cl, 0.), own ? (inv ? 1. - o : o - 1.) : o);
            if (!own) m *= f;
            else if (inv) m *= o * rho * im / f;
            else m *= o * rho * im * f;
          }
          if (last) U -= m;
          else {
            int slot = R.sp_slot[0];
#pragma unroll
            for (int u = 1; u < NSP_MAX; ++u) slot = j == u ? R.sp_slot[u] : slot;
            vr(slot) += Ctbaf * m;
          }
        }
      } else {
        Rnet = kf;
#pragma unroll
        for (int j = 0; j < NRC_MAX; ++j) Rnet *= F[j];
        dRdrho = Rnet / ct * invM * R.sumRc;
        dRdT = Rnet * ksens;
#pragma unroll
        for (int j = 0; j < NRC_MAX; ++j)
          if (j < R.n_rc) {
            double d = kf * rho * imw[R.rc_idx[j]] * R.rc_st[j] * (R.rc_st[j] == 1 ? 1. : ipow3(C[j], R.rc_st[j] - 1));
#pragma unroll
            for (int l = 0; l < NRC_MAX; ++l)
              if (l != j) d *= F[l];
            if (R.rc_slot[j] >= 0) vr(R.rc_slot[j]) += Ctbaf * d;
            else U -= d;
          }
        if (R.reversible) {
          const double Kc = exp(-(R.sumStoich * SC(S_LOGPORT, s) - invT * mv.invRu * sg));
          const double kr = kf / Kc;
          double Rr = kr;
#pragma unroll
          for (int j = 0; j < NPD_MAX; ++j) Rr *= Fp[j];
          Rnet -= Rr;
          dRdrho -= Rr / ct * invM * R.sumPd;
          dRdT -= Rr * (ksens + sb);
#pragma unroll
          for (int j = 0; j < NPD_MAX; ++j)
            if (j < R.n_pd) {
              double d = kr * rho * imw[R.pd_idx[j]] * R.pd_st[j] * (R.pd_st[j] == 1 ? 1. : ipow3(Cp[j], R.pd_st[j] - 1));
#pragma unroll
              for (int l = 0; l < NPD_MAX; ++l)
                if (l != j) d *= Fp[l];
              if (R.pd_slot[j] >= 0) vr(R.pd_slot[j]) -= Ctbaf * d;
              else U += d;
            }
        }
      }
      double Elast = 0.;
      for (int q = 0; q < R.n_tb; q += 4) {
        int slot[4];
        double e[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          const int at = R.tb_off + min(q + u, R.n_tb - 1);
          slot[u] = tbsl[at];
          e[u] = tbe[at];
        }
#pragma unroll
        for (int u = 0; u < 4; ++u)
          if (q + u < R.n_tb) {
            if (slot[u] >= 0) vr(slot[u]) += Rnet * tbs * e[u];
            else if (q + u == R.tb_last) Elast = tbs * e[u];
          }
      }
      rq(r) = Rnet * Ctbaf;
      if (a.qa) {
        const long q = a.sel ? (long)a.sel[i] : i;
        a.qa[q * nr + R.orig] = Rnet * ((R.type == RK_LINDEMANN || R.type == RK_TROE) ? qaC : Ctbaf);
      }
      rq(nr + r) = dRdrho * Ctbaf + dCdrho * Rnet;
      rq(2 * nr + r) = dRdT * Ctbaf + dCdT * Rnet;
      rq(3 * nr + r) = Rnet * cdense;
      rq(4 * nr + r) = Ctbaf * U - Rnet * Elast;
    }
    __syncthreads();

    // ---------------- P2: species gathers (lane = (species, state), as in P1) ----------------
    // With room for two lanes each, half of the waves gather the rates and half the rank-1 and diagonal terms.
    {
      constexpr int HALF = THREADS / 2;
      const bool two = JAC && HALF >= ns * S;
      const int part = two && threadIdx.x >= HALF ? 1 : 0;
      for (int it = threadIdx.x - part * HALF; it < ns * S; it += two ? HALF : THREADS) {
        const int k = it / S, s = it - k * S;
        const double Mk = mv.mw[k];
        const uint32_t e0 = sgx_off[k], e1 = sgx_off[k + 1];
        auto rq = [&](int e) { return rqb[e * S + s]; };
        uint32_t e = e0;
        if (!JAC || !two || part == 0) {
          double w = 0., w0 = 0., w1 = 0.;
          for (; e + 1 < e1; e += 2) {  // two reactions per trip: their LDS loads overlap (same summation order)
            const uint64_t ra = sgx[e], rb = sgx[e + 1];
            const int r0 = (int)(ra & 0xFFFFu), r1 = (int)(rb & 0xFFFFu);
            const double c0 = -(double)(int8_t)(ra >> 32) * Mk, c1 = -(double)(int8_t)(rb >> 32) * Mk;
            const double q0 = rq(r0), q1 = rq(r1);
            if (JAC) {
              const double a00 = rq(nr + r0), a01 = rq(nr + r1), a10 = rq(2 * nr + r0), a11 = rq(2 * nr + r1);
              w0 += c0 * a00; w0 += c1 * a01;
              w1 += c0 * a10; w1 += c1 * a11;
            }
            w += c0 * q0; w += c1 * q1;
          }
          if (e < e1) {
            const uint64_t rec = sgx[e];
            const int r = (int)(rec & 0xFFFFu);
            const double c = -(double)(int8_t)(rec >> 32) * Mk;  // -nu * M_k (rates_sensitivities_exact.cpp:1018)
            w += c * rq(r);
            if (JAC) {
              w0 += c * rq(nr + r);
              w1 += c * rq(2 * nr + r);
            }
          }
          SP(JAC ? W_ : G_, k, s) = w;  // (the rates need G no more)
          if (JAC) {
            SP(WS0_, k, s) = w0;
            SP(WS1_, k, s) = w1;
          }
        }
        if (JAC && (!two || part == 1)) {
          double A = 0., B = 0., DG = 0.;
          for (e = e0; e + 1 < e1; e += 2) {
            const uint64_t ra = sgx[e], rb = sgx[e + 1];
            const int r0 = (int)(ra & 0xFFFFu), r1 = (int)(rb & 0xFFFFu);
            const double c0 = -(double)(int8_t)(ra >> 32) * Mk, c1 = -(double)(int8_t)(rb >> 32) * Mk;
            const int d0 = (int)((ra >> 16) & 0xFFFFu), d1 = (int)((rb >> 16) & 0xFFFFu);
            const double a20 = rq(3 * nr + r0), a21 = rq(3 * nr + r1), a30 = rq(4 * nr + r0), a31 = rq(4 * nr + r1);
            const double v0 = d0 != 0xFFFF ? vb[d0 * S + s] : 0., v1 = d1 != 0xFFFF ? vb[d1 * S + s] : 0.;
            A += c0 * a20; A += c1 * a21;
            B += c0 * a30; B += c1 * a31;
            if (d0 != 0xFFFF) DG += c0 * v0;
            if (d1 != 0xFFFF) DG += c1 * v1;
          }
          if (e < e1) {
            const uint64_t rec = sgx[e];
            const int r = (int)(rec & 0xFFFFu);
            const double c = -(double)(int8_t)(rec >> 32) * Mk;
            A += c * rq(3 * nr + r);
            B += c * rq(4 * nr + r);
            const int ds = (int)((rec >> 16) & 0xFFFFu);
            if (ds != 0xFFFF) DG += c * vb[ds * S + s];
          }
          SP(A_, k, s) = A;
          SP(B_, k, s) = B;
          SP(DG_, k, s) = DG;
        }
      }
    }
    __syncthreads();
    // reductions over the species (wave per state, lane = species)
    if (wave < S) {
      const long il = first + wave;
      if (il < a.n) {
        const long i = a.sel ? (long)a.sel[il] : il;
        const double w = lane < ns ? SP(JAC ? W_ : G_, lane, wave) : 0.;
        const double w0 = JAC && lane < ns ? SP(WS0_, lane, wave) : 0., w1 = JAC && lane < ns ? SP(WS1_, lane, wave) : 0.;
        const double h = lane < ns ? SP(H_, lane, wave) : 0.;
        const double rho = SC(S_RHO, wave), cp = SC(S_CP, wave);
        const double HW = wave_sum(h * w);
        const double rhs0 = -HW / (rho * cp);
        const double iR = 1. / rho;
        if (a.rhs) {
          double *ro = a.rhs + i * a.rs_i;
          if (lane == 0) ro[0] = rhs0;
          if (lane < nm) ro[(1 + lane) * a.rs_v] = w * iR;
        }
        if (a.wout && lane < ns) a.wout[i * ns + lane] = w;
        if (JAC) {
          const double cpi = lane < ns ? SP(CPI_, lane, wave) : 0.;
          const double HS0 = wave_sum(h * w0), HS1 = wave_sum(h * w1), WCP = wave_sum(w * cpi);
          const double iRC = 1. / (rho * cp);
          if (lane < nm) SP(PR_, 1 + lane, wave) = iR * (w0 - iR * w);
          if (lane == 0) {
            SP(PR_, 0, wave) = -iRC * HS0 - iR * rhs0;
            SC(S_RHS0, wave) = rhs0; SC(S_HS0, wave) = HS0; SC(S_HS1, wave) = HS1; SC(S_WCP, wave) = WCP;
          }
        }
      }
    }
    if (JAC) {
      __syncthreads();
      // ---------------- P3: Jacobian columns (wave = column, lane = row; lane ns = the last species) -------
      // Every multiply-add here is written as an explicit fma or a rounded product (__dmul_rn), so the compiler's
      // contraction choices cannot differ between launch shapes and every shape gives bitwise the same Jacobian.
      int nact = 0;
      double iR[S], iRC[S], ric[S], rmw[S];  // 1/rho, 1/(rho cp), rhs0/cp, -rho M of each state
      long jo[S];  // offset of each state's Jacobian block (negative: none)
      for (int s = 0; s < S; ++s) {
        jo[s] = -1;
        if (first + s < a.n) {
          nact = s + 1;
          const long q = a.sel ? (long)a.sel[first + s] : first + s;
          if (a.jac) jo[s] = a.js_off ? a.js_off[q] : q * a.js_i;
        }
        iR[s] = 1. / SC(S_RHO, s);
        iRC[s] = 1. / (SC(S_RHO, s) * SC(S_CP, s));
        ric[s] = SC(S_RHS0, s) / SC(S_CP, s);
        rmw[s] = -SC(S_RHO, s) * SC(S_MMW, s);
      }
      if (a.jac) {
        constexpr int NW = THREADS / 64;
        // per-row values of every state, loaded once for all the columns this wave assembles
        const int iiL = lane - 1;
        const bool rowL = lane >= 1 && lane <= ns;
        double rA[S], rB[S], rH[S], rP[S], rD[S], cn[S];
        // the row's molecular weight (loaded here: in the column loop the Jacobian stores could alias it)
        const double MiL = rowL ? mv.mw[iiL] : 0.;
        for (int s = 0; s < S; ++s) {
          rA[s] = rowL ? SP(A_, iiL, s) : 0.;
          rB[s] = rowL ? SP(B_, iiL, s) : 0.;
          rH[s] = rowL ? SP(H_, iiL, s) : 0.;
          rP[s] = lane < ns ? SP(PR_, lane, s) : 0.;
          rD[s] = rowL ? SP(DG_, iiL, s) : 0.;
          cn[s] = SP(CPI_, nm, s);
        }
        for (int c = wave; c < ns; c += NW) {
          double val[S];
          if (c == 0) {
            for (int s = 0; s < S; ++s) {
              const double roT = SC(S_RHO, s) / SC(S_T, s);
              const double T00 = fma(-iRC[s], SC(S_HS1, s) + SC(S_WCP, s), -__dmul_rn(ric[s], SC(S_CPST, s)));
              val[s] = (lane == 0) ? fma(-roT, SP(PR_, 0, s), T00)
                                   : (lane < ns ? fma(-roT, SP(PR_, lane, s), __dmul_rn(SP(WS1_, lane - 1, s), iR[s]))
                                                : 0.);
            }
          } else {
            const int j = c - 1;
            const double dj = imw[j] - imw[nm];
            const int ii = lane - 1;  // species row; lane ns is the last species (temperature row only)
            const bool row = lane >= 1 && lane <= ns;
            // (what lane 0 alone needs is read by all, ahead of the sums: a load under its condition waits by itself)
            double full[S], cj[S];
            for (int s = 0; s < S; ++s) {
              full[s] = (row && ii == j) ? rD[s] : 0.;
              cj[s] = SP(CPI_, j, s) - cn[s];
            }
            if (row) {
              const double Mi = MiL;
              const int ee = j * ns + ii;
              const int t0 = exo[ee], t1 = exo[ee + 1];
              int t = t0;
              for (; t + 1 < t1; t += 2) {  // two entries per trip: their LDS loads overlap (same summation order)
                const uint32_t ra = exx[t], rb = exx[t + 1];
                const int sa = (int)(ra & 0xFFFFu), sb = (int)(rb & 0xFFFFu);
                const double ca = -(double)(int8_t)(ra >> 16) * Mi, cb = -(double)(int8_t)(rb >> 16) * Mi;
                double va[S], vbv[S];
                for (int s = 0; s < S; ++s) {
                  va[s] = vb[sa * S + s];
                  vbv[s] = vb[sb * S + s];
                }
                for (int s = 0; s < S; ++s) {
                  full[s] = fma(ca, va[s], full[s]);
                  full[s] = fma(cb, vbv[s], full[s]);
                }
              }
              if (t < t1) {
                const uint32_t rec = exx[t];
                const int slot = (int)(rec & 0xFFFFu);
                const double coef = -(double)(int8_t)(rec >> 16) * Mi;
                for (int s = 0; s < S; ++s) full[s] = fma(coef, vb[slot * S + s], full[s]);
              }
              for (int s = 0; s < S; ++s) full[s] += fma(dj, rA[s], rB[s]);
            }
            // temperature row: -(1/(rho cp)) sum_k h_k dw_k/dY_j over every species (isobaric_reactor_kernels.cpp:58-98),
            // the S states' sums formed together (absent states are zero vectors)
            double hv[4], hsum[4];
#pragma unroll
            for (int s = 0; s < 4; ++s) hv[s] = (s < S && row) ? __dmul_rn(rH[s < S ? s : 0], full[s < S ? s : 0]) : 0.;
            wave_sum4(hv, hsum);
            for (int s = 0; s < S; ++s) {
              const double hs = hsum[s];
              const double rd = __dmul_rn(rmw[s], dj), rp = __dmul_rn(rd, rP[s]);
              const double t = fma(-iRC[s], hs, fma(rd, rP[s], -__dmul_rn(ric[s], cj[s])));
              val[s] = lane == 0 ? t : fma(iR[s], full[s], rp);
            }
          }
          if (lane < ns) {
#pragma unroll
            for (int s = 0; s < S; ++s)
              if (jo[s] >= 0) a.jac[jo[s] + c * ns + lane] = val[s];
          }
        }
      }
      if (a.sens) {
        // raw option-0 sensitivities, (ns+1)^2 column-major with stride ns+1 (rates_sensitivities_exact.cpp:1011-1026); wave =
        // column, lane = row, gathered from the tables in LDS as the Jacobian's species rows are
        constexpr int NW = THREADS / 64;
        const double Mk = lane < ns ? mv.mw[lane] : 0.;
        for (int c = wave; c <= ns; c += NW) {
          double val[S];
          for (int s = 0; s < S; ++s) val[s] = 0.;
          if (lane < ns) {
            if (c < 2) {
              for (int s = 0; s < S; ++s) val[s] = SP(c == 0 ? WS0_ : WS1_, lane, s);
            } else {
              const int j = c - 2;
              const double dj = imw[j] - imw[nm];
              if (lane == j)
                for (int s = 0; s < S; ++s) val[s] = SP(DG_, j, s);
              const int t1 = exo[j * ns + lane + 1];
              for (int t = exo[j * ns + lane]; t < t1; ++t) {
                const uint32_t rec = exx[t];
                const int slot = (int)(rec & 0xFFFFu);
                const double coef = -(double)(int8_t)(rec >> 16) * Mk;
                for (int s = 0; s < S; ++s) val[s] = fma(coef, vb[slot * S + s], val[s]);
              }
              for (int s = 0; s < S; ++s) val[s] = fma(dj, SP(A_, lane, s), val[s]) + SP(B_, lane, s);
            }
          }
          if (lane <= ns)
            for (int s = 0; s < nact; ++s) {
              const long q = a.sel ? (long)a.sel[first + s] : first + s;
              a.sens[(q * (ns + 1) + c) * (ns + 1) + lane] = val[s];
            }
        }
      }
    }
    __syncthreads();  // the next group reuses the LDS
  }
}

template <int S, int THREADS, bool JAC>
size_t lds_bytes(const gf_mech *m) {
  const size_t t = JAC ? (size_t)m->view.tbl_bytes : (((size_t)m->view.exo_at + 15) & ~size_t(15));
  return t + S * (JAC ? m->lds_per_state : m->lds_per_state_rhs);
}

template <int S, int THREADS, bool JAC>
int launch_cfg(const gf_mech *m, const ChemArgs &a, hipStream_t st) {
  const size_t lds = lds_bytes<S, THREADS, JAC>(m);
  auto kern = chem_kernel<S, THREADS, JAC>;
  if (lds > m->lds_max) return fail(GF_ERR_UNSUPPORTED, "mechanism needs more LDS per workgroup than the device allows");
  if (lds > 65536) {
    if (hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds) != hipSuccess)
      return fail(GF_ERR_UNSUPPORTED, "mechanism needs more LDS per workgroup than the device allows");
  }
  const long groups = (a.n + S - 1) / S;
  // persistent launch: as many workgroups as fit the device at once (LDS-limited, at most 2048 threads
  // per CU), each owning a contiguous range of groups
  const long per_cu = std::max<long>(1, std::min<long>((long)(std::max<size_t>(m->lds_max, 65536) / lds), 2048 / THREADS));
  const long width = std::max<long>(1, (long)std::max(m->n_cu, 1) * per_cu);
  const long nwg = std::min(groups, width);
  const long gpw = (groups + nwg - 1) / nwg;
  const long grid = (groups + gpw - 1) / gpw;
  hipLaunchKernelGGL(kern, dim3((unsigned)grid), dim3(THREADS), lds, st, m->view, a, gpw);
  if (hipGetLastError() != hipSuccess) return fail(GF_ERR_HIP, "chemistry kernel launch failed");
  return GF_OK;
}

}  // namespace

// Launch shapes: states per workgroup x threads per workgroup. Every shape computes each state with the same
// lanes in the same order (per-state waves and reductions do not depend on S), so their outputs are bitwise
// identical and only their speed differs.
namespace {
constexpr int kShapes = 5;  // 0: 1x128, 1: 2x256, 2: 4x512, 3: 4x256, 4: 2x512

bool shape_fits(const gf_mech *m, int c, bool J) {
  if (!J) return true;
  const size_t lim = m->lds_max;
  if (c == 2 || c == 3) return lds_bytes<4, 512, true>(m) <= lim;
  if (c == 1 || c == 4) return lds_bytes<2, 256, true>(m) <= lim;
  return true;
}

int launch_shape(const gf_mech *m, const ChemIO &a, hipStream_t st, int c, bool J) {
  if (J) {
    switch (c) {
      case 0: return launch_cfg<1, 128, true>(m, a, st);
      case 1: return launch_cfg<2, 256, true>(m, a, st);
      case 3: return launch_cfg<4, 256, true>(m, a, st);
      case 4: return launch_cfg<2, 512, true>(m, a, st);
      default: return launch_cfg<4, 512, true>(m, a, st);
    }
  }
  switch (c) {
    case 0: return launch_cfg<1, 128, false>(m, a, st);
    case 1: return launch_cfg<2, 256, false>(m, a, st);
    case 3: return launch_cfg<4, 256, false>(m, a, st);
    case 4: return launch_cfg<2, 512, false>(m, a, st);
    default: return launch_cfg<4, 512, false>(m, a, st);
  }
}

// The fastest feasible shape for this launch: each candidate runs once to warm up, then twice between HIP
// events on the caller's stream (the outputs are the caller's, written identically by every candidate).
int autotune_shape(const gf_mech *m, const ChemIO &a, hipStream_t st, bool J, int &best) {
  hipEvent_t e0, e1;
  if (hipEventCreate(&e0) != hipSuccess) return fail(GF_ERR_HIP, "hipEventCreate failed");
  if (hipEventCreate(&e1) != hipSuccess) {
    (void)hipEventDestroy(e0);
    return fail(GF_ERR_HIP, "hipEventCreate failed");
  }
  float tbest = 0.f;
  bool have = false;
  best = 2;
  int rc = GF_OK;
  for (int c = 0; c < kShapes && rc == GF_OK; ++c) {
    if (!shape_fits(m, c, J)) continue;
    rc = launch_shape(m, a, st, c, J);
    if (rc == GF_OK && hipEventRecord(e0, st) != hipSuccess) rc = fail(GF_ERR_HIP, "hipEventRecord failed");
    for (int k = 0; k < 2 && rc == GF_OK; ++k) rc = launch_shape(m, a, st, c, J);
    if (rc == GF_OK && hipEventRecord(e1, st) != hipSuccess) rc = fail(GF_ERR_HIP, "hipEventRecord failed");
    if (rc == GF_OK && hipEventSynchronize(e1) != hipSuccess) rc = fail(GF_ERR_HIP, "hipEventSynchronize failed");
    float ms = 0.f;
    if (rc == GF_OK && hipEventElapsedTime(&ms, e0, e1) != hipSuccess) rc = fail(GF_ERR_HIP, "hipEventElapsedTime failed");
    if (rc == GF_OK && (!have || ms < tbest)) {
      have = true;
      tbest = ms;
      best = c;
    }
  }
  (void)hipEventDestroy(e0);
  (void)hipEventDestroy(e1);
  return rc;
}
}  // namespace

// GF_CHEM_CFG=<S>x<threads> (or gf_set_chem_launch_shape) fixes the launch shape for every call. Otherwise
// the first launch of a kind
// (RHS + Jacobian, or RHS only) at a batch size in [2^k, 2^(k+1)) times the feasible shapes and the fastest is
// kept for that kind and size class on this mechanism; under stream capture the default 4x512 is used
// untimed. Concurrent first calls from several host threads on one mechanism may time twice.
namespace {
int g_fixed_shape = -2;  // -2: not read from the environment yet; -1: autotune; 0..4: that shape
int fixed_shape() {
  if (g_fixed_shape == -2) {
    g_fixed_shape = -1;
    if (const char *e = getenv("GF_CHEM_CFG")) {
      if (!strcmp(e, "1x128")) g_fixed_shape = 0;
      else if (!strcmp(e, "2x256")) g_fixed_shape = 1;
      else if (!strcmp(e, "4x512")) g_fixed_shape = 2;
      else if (!strcmp(e, "4x256")) g_fixed_shape = 3;
      else if (!strcmp(e, "2x512")) g_fixed_shape = 4;
    }
  }
  return g_fixed_shape;
}
}  // namespace

int set_chem_launch_shape(int shape) {
  if (shape < -1 || shape >= kShapes) return fail(GF_ERR_ARG, "launch shape must be -1 (timed) or 0..4");
  g_fixed_shape = shape;
  return GF_OK;
}

int launch_chem(const gf_mech *m, const ChemIO &a, hipStream_t st) {
  if (a.n <= 0) return GF_OK;
  const int fixed = fixed_shape();
  const bool J = a.jac || a.sens;
  auto fallback = [&](int c) {  // fewer states per workgroup where the LDS does not fit
    if ((c == 2 || c == 3) && !shape_fits(m, c, J)) c = 1;
    if ((c == 1 || c == 4) && !shape_fits(m, c, J)) c = 0;
    return c;
  };
  if (fixed >= 0) return launch_shape(m, a, st, fallback(fixed), J);
  hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
  if (hipStreamIsCapturing(st, &cs) != hipSuccess || cs != hipStreamCaptureStatusNone)
    return launch_shape(m, a, st, fallback(2), J);
  if (!m->chem_shape_init) {
    std::memset(m->chem_shape, -1, sizeof m->chem_shape);
    m->chem_shape_init = true;
  }
  const int k = 63 - __builtin_clzll((unsigned long long)a.n);
  signed char &slot = m->chem_shape[J ? 0 : 1][k];
  if (a.no_tune) return launch_shape(m, a, st, fallback(slot >= 0 ? slot : 2), J);
  if (slot < 0) {
    int best = 2;
    const int rc = autotune_shape(m, a, st, J, best);
    if (rc != GF_OK) return rc;
    slot = (signed char)best;
  }
  return launch_shape(m, a, st, slot, J);
}

}  // namespace gfa
