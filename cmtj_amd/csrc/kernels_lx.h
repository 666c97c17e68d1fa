// kernels_lx.h -- one layer per lane for the exact feature sets of the large
// batches: RK4 with anisotropy, bilinear IEC and field-step drives (PIMM
// sweeps, coupled chains), and Euler-Heun with anisotropy, SOT, temperature
// and trapezoid drives (switching ensembles).  Lane mapping as in
// kernels_ll.h: an instance of nl layers on L consecutive lanes, lane l
// integrating layer l, neighbours by DPP.
//
// What bounds it: these batches fill the chip, so the rate is the VALU
// instructions of a wave step over the 64 / L instances it advances.  The
// step is the one of kernels_cl.h with whole vectors in the lane: fields
// pre-scaled by g = -gamma dt / (1 + alpha^2), the field's constant matrix A
// (demagnetisation and anisotropy) applied as nine FMAs, the torque as
// m x (h + alpha m x h), the length correction a polynomial that is tested once
// per block of steps (RK4) or by one wave-uniform branch (Euler-Heun).  RK4
// steps are binary64 in either mode: a binary64 FMA issues as fast as a
// binary32 one here, and stages in plain binary64 take 139 instructions a step
// against 199 for binary32 increments about a binary64 anchor (33,000 points
// 0.81 -> 0.62 ms, 196,608 points 2.10 -> 1.94 ms for 2,000 steps at most),
// and with a diagonal field matrix 111 (65,536 points, 2,000 to 20,000 steps,
// 7.4 -> 6.7 ms).  Against the general form (kernels_ll.h): RK4 372 -> 111 VALU
// instructions (20.7 -> 6.7 ms with the waves paired), Euler-Heun 425 -> 257 in
// the loop's code, 244 counted (131,072 instances x 10,000 steps 24.9 -> 14.0 ms; a
// single wave of instances 1.14 -> 0.5 us per step; in binary64 with the same
// normals 1.68 us per step of the 131,072 against 1.45: 222 registers).
// WPE: waves per SIMD the register allocation must leave room for.
#pragma once

#include "kernels_cl.h"

namespace cmtj {

template <class R>
__device__ __forceinline__ V3<R> cross_plus(V3<R> a, V3<R> b, V3<R> y) {  // a x b + y
  return mk<R>(fma(a.y, b.z, fma(-a.z, b.y, y.x)), fma(a.z, b.x, fma(-a.x, b.z, y.y)),
               fma(a.x, b.y, fma(-a.y, b.x, y.z)));
}
template <class R>
__device__ __forceinline__ V3<R> axpy(R s, V3<R> x, V3<R> y) {
  return mk<R>(fma(s, x.x, y.x), fma(s, x.y, y.y), fma(s, x.z, y.z));
}
template <class R>
struct Mat3 {
  V3<R> r0, r1, r2;
  __device__ __forceinline__ V3<R> apply(V3<R> m, V3<R> y) const {  // A m + y
    return mk<R>(fma(r0.z, m.z, fma(r0.y, m.y, fma(r0.x, m.x, y.x))),
                 fma(r1.z, m.z, fma(r1.y, m.y, fma(r1.x, m.x, y.y))),
                 fma(r2.z, m.z, fma(r2.y, m.y, fma(r2.x, m.x, y.z))));
  }
};

// ND: number of time-dependent records when fixed at compile time, -1 to read
// it from the group.  RK4: workgroups of up to 4 WPE waves (see pair_waves in
// engine.hip).
template <class R, int L, int SOLVER, uint32_t FM, int WPE = 1, int ND = -1>
__global__ __launch_bounds__(SOLVER == CMTJ_RK4 ? 256 * WPE : 64) __attribute__((amdgpu_waves_per_eu(WPE))) void
k_junction_ll_exact(GroupArgs g) {
  constexpr bool RK4 = SOLVER == CMTJ_RK4;
  static_assert(L == 2 || L == 4, "L lanes per instance must divide a 16-lane DPP row");
  static_assert(FM & F_EXACT, "exact feature sets");
  static_assert(!RK4 || !((FM & F_ALL) & ~(F_ANIS | F_IEC | F_DYNH)), "RK4: anisotropy, IEC, field drives");
  static_assert(!RK4 || ((FM & F_KSTEP) && sizeof(R) == 8), "RK4: step drives, binary64");
  static_assert(RK4 || (SOLVER == CMTJ_EULER_HEUN && !((FM & F_ALL) & ~(F_ANIS | F_DYN | F_SOT | F_THERMAL)) &&
                        (FM & F_KTRAP)),
                "Euler-Heun: anisotropy, SOT, temperature, trapezoid drives of scalar slots");
  constexpr int NR = ND >= 0 ? ND : DREG;
  static_assert(NR <= DREG, "every record in registers");
  auto has_rec = [&](int r) { return ND >= 0 || r < g.ndyn; };
  const uint32_t gl = blockIdx.x * blockDim.x + threadIdx.x;
  const uint32_t inst = gl / L;
  if (inst >= g.n) return;
  const int ly = (int)(gl % L);
  const int nl = g.nl;
  const bool act = ly < nl;
  const int lyr = act ? ly : 0;  // idle lanes shadow layer 0 and write nothing
  const uint32_t jid = g.order[inst];
  if (jid == 0xFFFFFFFFu) return;  // a slot without an instance (pair_waves)
  const cmtj_junction* J = g.js + jid;
  const uint32_t nsteps = J->n_steps;
  const uint32_t W = J->write_every;
  const uint32_t NE = J->n_entries;
  const double dt = J->dt;
  const uint64_t seed = J->seed, stream = J->stream;
  const uint64_t lbase = J->log_offset;
  const bool logging = (g.log != nullptr) && g.log_mask != 0;
  const uint32_t esize = g.log_f32 ? 4u : 8u;
  char* const lp = logging ? (char*)g.log + lbase * esize : nullptr;
  const uint64_t cs = (uint64_t)NE * esize;
  const double Rp = J->Rp, Rap = J->Rap;
  const MRCoef mcoef = mr_coef(g, J, lyr, logging && act);
  const bool hasB = act && ly > 0, hasT = act && ly + 1 < nl;
  const uint32_t gshift = (threadIdx.x & 63u) & ~(uint32_t)(L - 1);  // first lane of the instance in the wave

  int bits = 0;
#pragma unroll
  for (int l = 0; l < L; ++l) bits = (lyr == l) ? g.lbits[l] : bits;
  // whether any layer takes its polariser from a neighbour (wave-uniform)
  bool nb_ref = false;
#pragma unroll
  for (int l = 0; l < L; ++l) nb_ref |= l < nl && ((g.lbits[l] & 3) == CMTJ_REF_TOP || (g.lbits[l] & 3) == CMTJ_REF_BOTTOM);

  // ---- constants of the lane's layer
  Mat3<double> A;
  V3<double> hb, m;
  double jt, jb, alpha, gdt;
  // spin-orbit torque: g, g alpha (0 without), static coefficients, drives' constants; noise
  [[maybe_unused]] R ga = 0, gaa = 0, dlt = 0, flt = 0, bI = 0, bFL = 0, bDL = 0, bT = 0, sig2 = 0, nsd = 0, nu = 0;
  [[maybe_unused]] R k2d = 0;  // 2 g / Ms, for a driven anisotropy
  [[maybe_unused]] V3<R> pol = mk<R>(0, 0, 0), an = mk<R>(0, 0, 0);
  [[maybe_unused]] bool cur = false, dyn_sot = false;
  {
    LP<double> P;
    DV<double> base;
    load_layer<double>(g.layers[J->layer_offset + lyr], g.c, P, base, m);
    alpha = P.alpha;
    gdt = P.gconv * dt;
    const double gm = gdt * P.ms_mu0, k2 = gdt * ((2.0 * base.K) * P.inv_ms);
    const V3<double> a = P.anis;
    A.r0 = mk<double>(k2 * a.x * a.x - P.N[0] * gm, k2 * a.x * a.y, k2 * a.x * a.z);
    A.r1 = mk<double>(k2 * a.y * a.x, k2 * a.y * a.y - P.N[4] * gm, k2 * a.y * a.z);
    A.r2 = mk<double>(k2 * a.z * a.x, k2 * a.z * a.y, k2 * a.z * a.z - P.N[8] * gm);
    hb = base.H * gdt;
    jt = hasT ? base.Jt * (gdt * P.inv_mst) : 0.0;
    jb = hasB ? base.Jb * (gdt * P.inv_mst) : 0.0;
    if constexpr (!RK4) {
      const bool sot = ((bits >> 2) & 3) == 2;
      dyn_sot = sot && ((bits >> 4) & 1) != 0;
      cur = sot && !dyn_sot;
      ga = sot ? (R)gdt : R(0);
      gaa = sot ? (R)(gdt * alpha) : R(0);
      dlt = cur ? (R)P.dl_t : R(0);
      flt = cur ? (R)P.fl_t : R(0);
      bI = cur ? (R)base.I : R(0);
      bFL = dyn_sot ? (R)base.FL : R(0);
      bDL = dyn_sot ? (R)base.DL : R(0);
      bT = (R)base.T;
      const bool fixed = sot && (bits & 3) == CMTJ_REF_FIXED;
      pol = mk<R>(fixed ? (R)P.ref.x : R(0), fixed ? (R)P.ref.y : R(0), fixed ? (R)P.ref.z : R(0));
      an = cvt<R>(a);
      k2d = (R)(gdt * 2.0 * P.inv_ms);
      // kick of a step: -gamma/(1 + a^2) sqrt(dt) sqrt(2 alpha kB T / (Ms V gamma)) m x (xi + alpha m x xi)
      const bool therm = ((bits >> 6) & 1) != 0;
      sig2 = therm ? (R)P.sig2 : R(0);
      nsd = (R)(P.gconv * sqrt(dt));
      nu = nsd * (R)sqrt(sig2 * bT);
    }
  }
  // RK4: the matrix less the identity times its last diagonal entry (a multiple
  // of m in the field moves nothing), and whether it is diagonal in every lane
  // of the wave: two FMAs a field evaluation instead of eight, the same bits
  // either way (as in kernels_cl.h)
  bool diag = false;
  if constexpr (RK4) {
    const double lam = A.r2.z;
    A.r0.x -= lam;
    A.r1.y -= lam;
    A.r2.z = 0.0;
    diag = __ballot(A.r0.y != 0.0 || A.r0.z != 0.0 || A.r1.x != 0.0 || A.r1.z != 0.0 || A.r2.x != 0.0 ||
                    A.r2.y != 0.0) == 0ull;
  }
  // ---- drive records
  DynRec dr[DREG];
  bool on[DREG];
  double win_lo = __builtin_inf(), win_hi = -__builtin_inf();
  [[maybe_unused]] bool t_driven = false, k_driven = false, sot_driven = false;
  [[maybe_unused]] R wI[DREG], wFL[DREG], wDL[DREG], wT[DREG], wK[DREG];
#pragma unroll
  for (int r = 0; r < NR; ++r) {
    on[r] = false;
    dr[r] = DynRec{0.0, 0.0, 0.0, 0.0, 0, 0};
    wI[r] = wFL[r] = wDL[r] = wT[r] = wK[r] = R(0);
    if (has_rec(r)) {
      dr[r] = load_rec<FM>(g.dyn + (size_t)r * g.n + inst);
      const int slot = (g.dmeta[r] >> 8) & 0xff;
      on[r] = act && (((g.dmeta[r] >> 16) & 0xff) >> ly & 1);
      if constexpr (!RK4) {  // a drive of a torque that the layer does not have stays out of it
        if (slot == CMTJ_SLOT_CURRENT) on[r] = on[r] && cur;
        if (slot == CMTJ_SLOT_FL || slot == CMTJ_SLOT_DL) on[r] = on[r] && dyn_sot;
        t_driven |= slot == CMTJ_SLOT_TEMPERATURE;
        k_driven |= slot == CMTJ_SLOT_K;
        sot_driven |= slot == CMTJ_SLOT_FL || slot == CMTJ_SLOT_DL;
        wI[r] = R(slot == CMTJ_SLOT_CURRENT ? 1 : 0);
        wFL[r] = R(slot == CMTJ_SLOT_FL ? 1 : 0);
        wDL[r] = R(slot == CMTJ_SLOT_DL ? 1 : 0);
        wT[r] = R(slot == CMTJ_SLOT_TEMPERATURE ? 1 : 0);
        wK[r] = R(slot == CMTJ_SLOT_K ? 1 : 0);
      }
      win_lo = fmin(win_lo, dr[r].p1);
      win_hi = fmax(win_hi, dr[r].p2);
    }
  }
  uint32_t k = 0;
  int code = CMTJ_OK, nan_layer = -1;
  uint32_t i = 0, iend = nsteps;
  cmtj_state* const S = g.state ? g.state + jid : nullptr;
  if (S) {  // resume: state of the previous slice
    m = mk<double>(S->m[lyr][0], S->m[lyr][1], S->m[lyr][2]);
    i = S->step;
    k = S->entries;
    code = S->code;
    nan_layer = (code == CMTJ_OK) ? -1 : S->nan_layer;
    iend = (code != CMTJ_OK) ? i : (uint32_t)min((uint64_t)nsteps, (uint64_t)i + g.slice);
  }
  // neighbours (m of layers ly - 1 and ly + 1) at the start of a step; two
  // layers swap lanes (either one's neighbour is the other)
  constexpr int QP_SWAP = 0xB1;  // quad_perm [1,0,3,2]
  V3<double> bot = mk<double>(0, 0, 0), top = bot;
  auto neighbours = [&]() __attribute__((always_inline)) {
    if constexpr (L == 2) {
      top = mk<double>(dpp_d<QP_SWAP>(m.x), dpp_d<QP_SWAP>(m.y), dpp_d<QP_SWAP>(m.z));
    } else {
      bot = from_prev(m, hasB);
      top = from_next(m, hasT);
    }
  };
  const double jn = hasT ? jt : jb;  // L = 2: towards the other layer
  [[maybe_unused]] const Mat3<R> AR{cvt<R>(A.r0), cvt<R>(A.r1), cvt<R>(A.r2)};
  [[maybe_unused]] const V3<R> hbR = cvt<R>(hb);
  const R alphaR = (R)alpha;
  // neighbours are read by the coupling, by a polariser and by the classic R
  const bool use_nb = (FM & F_IEC) != 0 || nb_ref || (logging && (g.log_mask & CMTJ_LOG_MR) && nl > 1);
  if (use_nb) neighbours();

  double dev = 0.0;
  unsigned long long hitb = 0ull;
  uint64_t next_log = 0;
  ERec<R> er;
  // One step (the tags as in k_junction_cl): DRV 0 outside every drive's
  // window, 1 inside, 2 every trapezoid on one line through the block.
  double lc[DREG] = {0.0, 0.0}, lt[DREG] = {0.0, 0.0}, la[DREG] = {0.0, 0.0};  // la + lc (t - lt)
  auto step = [&](auto drv_tag, auto log_tag, auto chk_tag) __attribute__((always_inline)) {
    constexpr int DRV = decltype(drv_tag)::value & 3;
    constexpr bool DG = (decltype(drv_tag)::value & 4) != 0;
    constexpr int LOGM = decltype(log_tag)::value;
    constexpr bool CHK = decltype(chk_tag)::value;
    const double t = (double)i * dt;
    V3<double> mn;
    if constexpr (RK4) {
      // scaled field of the step drives at ts
      auto drive = [&](double ts) __attribute__((always_inline)) -> V3<double> {
        V3<double> h = mk<double>(0, 0, 0);
#pragma unroll
        for (int r = 0; r < NR; ++r) {
          if (has_rec(r)) {
            const double v = (on[r] && ts >= dr[r].p1 && ts <= dr[r].p2) ? dr[r].A * gdt : 0.0;
            const int ax = ((g.dmeta[r] >> 8) & 0xff) % 3;
            h.x += ax == 0 ? v : 0.0;
            h.y += ax == 1 ? v : 0.0;
            h.z += ax == 2 ? v : 0.0;
          }
        }
        return h;
      };
      V3<double> B = hb, D0 = mk<double>(0, 0, 0);
      if constexpr (DRV != 0) {
        D0 = drive(t);
        B = B + D0;
      }
      if constexpr (FM & F_IEC) {
        if constexpr (L == 2) {
          B = axpy(jn, top, B);
        } else {
          B = axpy(jt, top, axpy(jb, bot, B));
        }
      }
      auto torque = [&](V3<double> s, V3<double> Bs, V3<double>& h, V3<double>& gg) __attribute__((always_inline)) {
        if constexpr (DG)
          h = mk<double>(fma(A.r0.x, s.x, Bs.x), fma(A.r1.y, s.y, Bs.y), Bs.z);
        else
          h = mk<double>(fma(A.r0.z, s.z, fma(A.r0.y, s.y, fma(A.r0.x, s.x, Bs.x))),
                         fma(A.r1.z, s.z, fma(A.r1.y, s.y, fma(A.r1.x, s.x, Bs.y))),
                         fma(A.r2.y, s.y, fma(A.r2.x, s.x, Bs.z)));
        gg = axpy(alpha, cross(s, h), h);
        return cross(s, gg);
      };
      // rk4_step (core/junction.hpp:1017-1041)
      {
        V3<double> h, gg, Bm = B, Be = B;
        if constexpr (DRV != 0) {
          Bm = B + (drive(t + 0.5 * dt) - D0);
          Be = B + (drive(t + dt) - D0);
        }
        const V3<double> k1 = torque(m, B, h, gg);
        const V3<double> k2 = torque(axpy(0.5, k1, m), Bm, h, gg);
        const V3<double> k3 = torque(axpy(0.5, k2, m), Bm, h, gg);
        const V3<double> k4 = torque(m + k3, Be, h, gg);
        mn = axpy(1.0 / 6.0, axpy(2.0, k2 + k3, k1 + k4), m);
      }
    } else {
      // eulerHeunSolverStep (core/junction.hpp:1709-1754): drift at t, the
      // stochastic torque (:824-831) at m and at m + g sqrt(dt), one dW per
      // step
      const V3<R> mr = cvt<R>(m);
      R I = bI, FL = bFL, DL = bDL, T = bT;
      V3<R> h = AR.apply(mr, hbR);
#pragma unroll
      for (int r = 0; r < NR; ++r) {
        if (has_rec(r)) {
          double v;
          if constexpr (DRV == 2)
            v = fma(lc[r], t - lt[r], la[r]);
          else
            v = wave_value<double, false, FM>(CMTJ_TRAPEZOID, dr[r], g, t, i, 0, 1);
          // to its slot by wave-uniform 0/1 weights (x is 0 on layers the
          // record does not feed, so a non-finite drive stays with its layer)
          const R x = on[r] ? (R)v : R(0);
          I = fma(wI[r], x, I);
          if (sot_driven) {
            FL = fma(wFL[r], x, FL);
            DL = fma(wDL[r], x, DL);
          }
          if (t_driven) T = fma(wT[r], x, T);
          if (k_driven) h = axpy((wK[r] * k2d * x) * dot(an, mr), an, h);
        }
      }
      V3<R> p = pol, f;
      if (nb_ref) {
        const int rt = bits & 3;
        const bool sot = ((bits >> 2) & 3) == 2;
        const V3<R> tr = cvt<R>(top), br = (L == 2) ? tr : cvt<R>(bot);
        const bool ut = sot && rt == CMTJ_REF_TOP && hasT, ub = sot && rt == CMTJ_REF_BOTTOM && hasB;
        p = mk<R>(ut ? tr.x : (ub ? br.x : p.x), ut ? tr.y : (ub ? br.y : p.y), ut ? tr.z : (ub ? br.z : p.z));
      }
      {
        // SOT (:770-812): m x (h + alpha m x h + a p + b m x p), the inner
        // products taken together
        const R Hdl = fma(dlt, I, DL), Hfl = fma(flt, I, FL);
        const R a = fma(ga, Hfl, -gaa * Hdl), b = fma(ga, Hdl, gaa * Hfl);
        f = cross(mr, cross_plus(mr, axpy(b, p, h * alphaR), axpy(a, p, h)));
      }
      R n1 = nu;
      if (t_driven) n1 = nsd * (R)sqrt(sig2 * T);
      const V3<R> dW = thermal_normals<R>(seed, stream, i, (uint32_t)lyr) * n1;
      auto kick = [&](V3<R> s) __attribute__((always_inline)) -> V3<R> {
        return cross(s, axpy(alphaR, cross(s, dW), dW));
      };
      const V3<R> k0 = kick(mr);
      const V3<R> k1 = kick(mr + k0);
      // drift and kick are added to m each in binary64: a kick far below the
      // drift would be lost in a binary32 sum (three conversions fewer, 13.4
      // against 14.0 ms)
      const V3<double> md = m + cvt<double>(f);
      mn = axpy(0.5, cvt<double>(k0 + k1), md);
    }
    // ---- CVector::normalize (core/cvector.hpp:185-192): (1 + e)^(-1/2) by its
    // series up to |e| = kUnitRange, exactly beyond
    const double e = fma(mn.z, mn.z, fma(mn.y, mn.y, fma(mn.x, mn.x, -1.0)));
    const double p = e * fma(e, fma(e, fma(e, 0.2734375, -0.3125), 0.375), -0.5);
    V3<double> ms = axpy(p, mn, mn);
    if constexpr (RK4 && !CHK) {
      dev = fma(e, e, dev);
    } else {
      const bool far = !(fabs(e) <= kUnitRange);
      if (__builtin_expect(__ballot(far) != 0ull, 0)) {
        const V3<double> mx = normalize_exact(mn);
        ms = mk<double>(far ? mx.x : ms.x, far ? mx.y : ms.y, far ? mx.z : ms.z);
      }
    }
    if constexpr (CHK) {
      // the reference updates layers in turn and stops at the first NaN:
      // layers up to and including it take the new value
      const unsigned long long bad = __ballot(act && isnan(ms.x));
      hitb = bad;
      if (__builtin_expect(bad != 0ull, 0)) {
        const uint32_t gb = (uint32_t)((bad >> gshift) & ((1ull << L) - 1));
        const bool take = gb != 0u && ly <= (int)__builtin_ctz(gb | 0x80000000u);
        m = mk<double>(take ? ms.x : m.x, take ? ms.y : m.y, take ? ms.z : m.z);
        return;
      }
    }
    m = ms;
    if (use_nb) neighbours();
    if (LOGM == 1 || (LOGM == 0 && (uint64_t)i == next_log)) {
      if (logging)
        write_entry_ll<R, L, FM, false>(g, J, ly, act, m, top, er, lp + (uint64_t)k * esize, cs, Rp, Rap, mcoef);
      ++k;
      next_log += W;
    }
  };
  bool stopped = false;
  using C0 = std::integral_constant<int, 0>;
  using C1 = std::integral_constant<int, 1>;
  using C2 = std::integral_constant<int, 2>;
  // Steps below lim in wave-uniform passes of blocks, as in k_junction_cl.
  auto phase = [&](uint32_t lim, auto drv_tag) __attribute__((always_inline)) {
    for (;;) {
      const uint32_t n = (!stopped && i < lim) ? lim - i : 0u;
      const uint32_t seg = wave_min_nonzero(n);
      if (seg == 0u) break;
      if (n != 0u) {
        const uint32_t i0 = i;
        uint32_t end = seg;  // wave-uniform
        next_log = (uint64_t)k * W;
        const uint32_t W0 = __builtin_amdgcn_readfirstlane(W);
        uint32_t cd = __builtin_amdgcn_readfirstlane((uint32_t)(next_log - i));
        const bool uni = __ballot(W != W0 || (uint32_t)(next_log - i) != cd || next_log < i) == 0ull;
        // steps [u0, ue) with tag DT, the entries on a scalar countdown where
        // the lanes agree on them
        auto steps = [&](uint32_t u0, uint32_t ue, auto dt_tag) __attribute__((always_inline)) {
          if (!uni) {
            for (uint32_t u = u0; u < ue; ++u) {
              i = i0 + u;
              step(dt_tag, C0{}, std::false_type{});
            }
            return;
          }
          for (uint32_t u = u0; u < ue;) {
            const uint32_t us = min(ue - u, cd), un = u + us;  // steps without an entry
            for (; u < un; ++u) {
              i = i0 + u;
              step(dt_tag, C2{}, std::false_type{});
            }
            cd -= us;
            if (u < ue) {
              i = i0 + u;
              step(dt_tag, C1{}, std::false_type{});
              ++u;
              cd = W0 - 1u;
            }
          }
        };
        uint32_t slow = 0;
        bool flagged = false;
        for (uint32_t u0 = 0; u0 < end;) {
          const uint32_t ue = min(u0 + (uint32_t)CL_BLOCK, end);
          if constexpr (!RK4) {
            // whether every trapezoid stays on one of its lines over the block
            // (constant 0 and A, rise, fall): value la + lc (t - lt)
            const double ta = (double)(i0 + u0) * dt, tb = (double)(i0 + ue - 1u) * dt;
            bool line = true;
#pragma unroll
            for (int r = 0; r < NR; ++r) {
              if (has_rec(r)) {
                const double t1 = dr[r].p1, t2 = t1 + dr[r].p2, t3 = t1 + dr[r].p2 + dr[r].p3,
                             t4 = t1 + 2 * dr[r].p2 + dr[r].p3;
                auto seg_of = [&](double t) { return t < t1 ? 0 : t <= t2 ? 1 : t <= t3 ? 2 : t <= t4 ? 3 : 4; };
                const int sa = seg_of(ta);
                line = line && sa == seg_of(tb);
                double slope;
                __builtin_memcpy(&slope, &dr[r].tidx, sizeof slope);
                lc[r] = sa == 1 ? slope : (sa == 3 ? -slope : 0.0);
                lt[r] = sa == 1 ? t1 : (sa == 3 ? t3 : 0.0);
                la[r] = (sa == 2 || sa == 3) ? dr[r].A : 0.0;
              }
            }
            if (__ballot(!line) == 0ull)
              steps(u0, ue, C2{});
            else
              steps(u0, ue, C1{});
          } else {
            const V3<double> m_b = m;
            const uint32_t k_b = k, cd_b = cd;
            bool redo = slow != 0u;
            if (!redo) {
              dev = 0.0;
              steps(u0, ue, drv_tag);
              redo = __ballot(!(dev <= kUnitRange * kUnitRange)) != 0ull;
              slow = (redo && flagged) ? 31u : 0u;
              flagged = redo;
              if (redo) {
                m = m_b;
                if (use_nb) neighbours();
              }
            } else {
              --slow;
            }
            if (__builtin_expect(redo, 0)) {
              k = k_b;
              next_log = (uint64_t)k * W;
              for (uint32_t u = u0; u < ue; ++u) {
                i = i0 + u;
                step(drv_tag, C0{}, std::true_type{});
                if (hitb) {
                  end = u;
                  break;
                }
              }
              if (uni) {  // the countdown after the block's steps
                cd = cd_b;
                const uint32_t ns = min(ue, end) - u0;
                cd = (ns <= cd) ? cd - ns : (W0 - 1u - (ns - cd - 1u) % W0);
              }
            }
          }
          u0 = ue;
        }
        i = i0 + end;
        if (hitb) {
          const uint32_t gb = (uint32_t)((hitb >> gshift) & ((1ull << L) - 1));
          bool stop = gb != 0u;
          if (gb) {
            nan_layer = __builtin_ctz(gb);
            code = CMTJ_ERR_NAN;
          }
          // (were no lane to stop, the pass would take the same step for ever)
          if (__ballot(stop) == 0ull) {
            code = CMTJ_ERR_NAN;
            stop = true;
          }
          stopped = stop;
          hitb = 0ull;
        }
      }
    }
  };
  if constexpr (RK4) {
    // steps [ia, ib) may meet a record's window, one step of margin each side
    uint32_t ia = iend, ib = iend;
    if (win_lo <= win_hi) {
      const double a = floor(win_lo / dt) - 2.0, b = floor(win_hi / dt) + 2.0;
      ia = a <= (double)i ? i : (a >= (double)iend ? iend : (uint32_t)a);
      ib = b <= (double)ia ? ia : (b >= (double)iend ? iend : (uint32_t)b);
    }
    auto run = [&](auto off, auto on) __attribute__((always_inline)) {
      phase(ia, off);
      phase(ib, on);
      phase(iend, off);
    };
    if (diag)
      run(std::integral_constant<int, 4>{}, std::integral_constant<int, 5>{});
    else
      run(C0{}, C1{});
  } else {
    phase(iend, C1{});
  }
  if (g.mag_out && act) {
    double* o = g.mag_out + ((size_t)jid * CMTJ_MAX_LAYERS + ly) * 3;
    o[0] = m.x;
    o[1] = m.y;
    o[2] = m.z;
  }
  if (g.status && ly == 0) {
    cmtj_status s;
    s.code = code;
    s.steps_done = i;
    s.entries_done = k;
    s.nan_layer = nan_layer;
    g.status[jid] = s;
  }
  if (S) {
    if (act) {
      S->m[ly][0] = m.x;
      S->m[ly][1] = m.y;
      S->m[ly][2] = m.z;
    }
    if (ly == 0) {
      S->step = i;
      S->entries = k;
      S->code = code;
      S->nan_layer = nan_layer;
    }
  }
}

}  // namespace cmtj
