// kernels_cl.h -- the junction kernel with one vector component per lane.
//
// Layer l of an instance occupies the lane quad 4l..4l+3: lanes 0, 1, 2 of
// the quad hold the x, y and z components of every per-layer vector (m, the
// effective field, the torques), lane 3 holds zeros.  An instance of at most
// L layers spans 4L lanes (L = 1, 2 or 4: 4L divides a 16-lane DPP row).
//
// A lane keeps its layer's whole start-of-step m (its own component and, by
// the DPP quad permutations [1,2,0,3] and [2,0,1,3], components c + 1 and
// c + 2), so dot products, the field at all three components and the first
// cross product are formed in the lane; what crosses lanes is each stage's m
// and, once per step, the neighbour layers' (start-of-step values,
// core/junction.hpp:1682-1707) by a row shift of 4 lanes.  A step of one wave
// issues fewer instructions than one layer per lane (PIMM set 100 against 114
// VALU, the binary64 step among the latter), and a batch occupies four times
// as many waves: on a batch too small to fill the chip both shorten the sweep,
// whose time is the step count of the longest instance times the latency of one
// wave step.
//
// Integrators: the anchored binary32 RK4 of the other FP32 kernels (rk4_step,
// core/junction.hpp:1017-1041): k1 and the state in binary64, stages 2-4 as
// binary32 increments f(m0 + d, t_s) - f(m0, t) (rhs_delta in kernels.h,
// same terms in component form, the cross products expanded about the
// anchor, so they round differently); and RK4, Heun and Euler-Heun in
// binary64.  Features of the binary32 form: demagnetisation with a diagonal
// tensor, first-order anisotropy, bilinear IEC with constant coupling,
// time-dependent drivers that feed field slots only; log channels m and the
// classic or strip magnetoresistance.  Results agree with the other kernels
// to rounding, not bitwise.
#pragma once

#include <type_traits>

#include "kernels_ll.h"

namespace cmtj {

constexpr int QP_ROT1 = 0xC9;   // quad_perm [1,2,0,3]: component c reads c + 1 (mod 3)
constexpr int QP_ROT2 = 0xD2;   // quad_perm [2,0,1,3]: component c reads c + 2 (mod 3)
constexpr int QP_SWAP1 = 0xB1;  // quad_perm [1,0,3,2]
constexpr int QP_SWAP2 = 0x4E;  // quad_perm [2,3,0,1]
constexpr int QP_BC0 = 0x00;    // quad_perm [0,0,0,0]: x to every lane of the quad
constexpr int QP_NEXT = 0x39;   // quad_perm [1,2,3,0]: the quad's values move down one lane
constexpr int DPP_ROW_SHR4 = 0x114;  // lane i reads lane i - 4 (0 outside the row)
constexpr int DPP_ROW_SHL4 = 0x104;  // lane i reads lane i + 4
constexpr int DPP_HALF_MIRROR = 0x141;  // lane i reads lane 7 - i of its 8
constexpr int DPP_MIRROR = 0x140;       // lane i reads lane 15 - i of its row

template <int CTRL>
__device__ __forceinline__ float dpp_f(float v) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xF, 0xF, true));
}
// v of the lane CTRL names, written only to the lanes of the banks (groups
// of 4 lanes in a 16-lane row) that BANK enables; the other lanes keep old.
template <int CTRL, int BANK>
__device__ __forceinline__ double dpp_keep(double old, double v) {
  const unsigned long long o = (unsigned long long)__double_as_longlong(old);
  const unsigned long long u = (unsigned long long)__double_as_longlong(v);
  const int lo = __builtin_amdgcn_update_dpp((int)(unsigned)(o & 0xffffffffull), (int)(unsigned)(u & 0xffffffffull),
                                             CTRL, 0xF, BANK, false);
  const int hi = __builtin_amdgcn_update_dpp((int)(unsigned)(o >> 32), (int)(unsigned)(u >> 32), CTRL, 0xF, BANK,
                                             false);
  return __longlong_as_double((long long)(((unsigned long long)(unsigned)hi << 32) | (unsigned)lo));
}
// Banks whose quad has a layer below (UP = false) or above (UP = true) in
// the same instance, for instances of L = 1, 2 or 4 layers (one quad per
// layer, instances aligned to 4L lanes): the row shifts by 4 lanes then
// never read another instance's lanes, and the lanes of the other banks
// keep the zero they start with.
template <int L, bool UP>
constexpr int neighbour_banks() {
  int m = 0;
  for (int b = 0; b < 4; ++b) {
    const int ly = b % L;
    if (UP ? (ly + 1 < L) : (ly > 0)) m |= 1 << b;
  }
  return m;
}
// Steps of one block of the component-lane step loop: what is tested or set
// right once per block (a NaN, the length correction's range, the phase of a
// sine drive) costs a step 1/64 of its instructions.
constexpr int CL_BLOCK = 64;

// |m|^2 - 1 of a step's new m up to which its length correction is the
// binomial series of (1 + d)^(-1/2) to fourth order: the first term left out
// is 63/256 d^5 < 7e-18 there.
constexpr double kUnitRange = 4.8828125e-4;  // 2^-11

// The smallest nonzero n over the active lanes of the wave (0 if none):
// wave-uniform, read lane by lane through the ballot.
__device__ __forceinline__ uint32_t wave_min_nonzero(uint32_t n) {
  unsigned long long act = __ballot(n != 0u);
  uint32_t best = 0u;
  while (act) {
    const uint32_t v = (uint32_t)__builtin_amdgcn_readlane((int)n, (int)__builtin_ctzll(act));
    best = (best == 0u || v < best) ? v : best;
    act &= act - 1ull;
  }
  return best;
}
template <int CTRL>
__device__ __forceinline__ double dpp_x(double v) {
  return dpp_d<CTRL>(v);
}
template <int CTRL>
__device__ __forceinline__ float dpp_x(float v) {
  return dpp_f<CTRL>(v);
}

// Entry (r, q) of a row-major 3 x 3 tensor in registers, by selects (the
// nine values by value: selects between addresses would keep the tensor in
// scratch memory).
#define CL_ENTRY(T, r, q) entry9(T[0], T[1], T[2], T[3], T[4], T[5], T[6], T[7], T[8], r, q)
__device__ __forceinline__ double pick3(double x, double y, double z, int k) { return k == 0 ? x : (k == 1 ? y : z); }
__device__ __forceinline__ double entry9(double a, double b, double c, double d, double e, double f, double g,
                                         double h, double i, int r, int q) {
  return pick3(pick3(a, b, c, q), pick3(d, e, f, q), pick3(g, h, i, q), r);
}

// A vector as one lane sees it: its own component c and the components c + 1
// and c + 2 (mod 3) of the other lanes of the quad.
template <class T>
struct Rot {
  T a, b, c;
};
template <class T>
__device__ __forceinline__ Rot<T> rot3(T v) {
  return {v, dpp_x<QP_ROT1>(v), dpp_x<QP_ROT2>(v)};
}
template <class T>
__device__ __forceinline__ T rdot(const Rot<T>& x, const Rot<T>& y) {
  return fma(x.c, y.c, fma(x.b, y.b, x.a * y.a));
}
// components c + 1 and c + 2 of x x y, and component c
template <class T>
__device__ __forceinline__ T cross_b(const Rot<T>& x, const Rot<T>& y) {
  return fma(x.c, y.a, -(x.a * y.c));
}
template <class T>
__device__ __forceinline__ T cross_c2(const Rot<T>& x, const Rot<T>& y) {
  return fma(x.a, y.b, -(x.b * y.a));
}
template <class T>
__device__ __forceinline__ T cross_a(const Rot<T>& x, T yb, T yc) {
  return fma(x.b, yc, -(x.c * yb));
}

// The binary32 stages of the anchored RK4: increments f(m0 + d, ts) - f(m0, t)
// at this lane's component, every field scaled by -gamma dt / (1 + alpha^2):
//   g = h + alpha m x h,  f = m x g  (the torque m x h + alpha m x (m x h)),
//   dh = dd + A d  (A: row c of the field's constant matrix),  s = m0 + d,
//   dP = s x dh + d x h0,  dg = dh + alpha dP,  df = s x dg + d x g0.
// Returns 2 k2 + 2 k3 + k4 (each relative to k1).  Fourteen instructions a
// stage and no wait state: the neighbour components of d, dh and dg are read
// through the DPP operand of the instruction that consumes them (the compiler
// emits a separate DPP move for the addend form of an FMA, and wait states
// after a fresh value), and two independent instructions follow every fresh
// value before its first DPP read, the number the read needs.  As separate
// moves and FMAs the stages took 84 of a step's 189 issue slots, here 50 of
// 120 (4096-point PIMM sweep, 200,000 steps: 64.4 -> 44.7 ms with the rest of
// the step's layout).
#define CL_ROT1 "quad_perm:[1,2,0,3] row_mask:0xf bank_mask:0xf\n\t"
#define CL_ROT2 "quad_perm:[2,0,1,3] row_mask:0xf bank_mask:0xf\n\t"
#define CL_STAGES(OFF) \
  "v_mul_f32 %[d], 0.5, %[k1]\n\t" \
  "v_cvt_f32_f64 %[g1], %[gb]\n\t" \
  "v_fma_f32 %[h], %[a0], %[d], %[dm]\n\t" \
  OFF \
  "v_add_f32_dpp %[s1], %[d], %[m1] " CL_ROT1 \
  "v_add_f32_dpp %[s2], %[d], %[m2] " CL_ROT2 \
  "v_mul_f32_dpp %[p], %[d], %[h2] " CL_ROT1 \
  "v_fmac_f32_dpp %[p], %[d], -%[h1] " CL_ROT2 \
  "v_fmac_f32_dpp %[p], %[h], %[s1] " CL_ROT2 \
  "v_fmac_f32_dpp %[p], %[h], -%[s2] " CL_ROT1 \
  "v_fmac_f32 %[h], %[al], %[p]\n\t" \
  "v_cvt_f32_f64 %[g2], %[gc]\n\t" \
  "v_mul_f32_dpp %[r], %[d], %[g2] " CL_ROT1 \
  "v_fmac_f32_dpp %[r], %[d], -%[g1] " CL_ROT2 \
  "v_fmac_f32_dpp %[r], %[h], %[s1] " CL_ROT2 \
  "v_fmac_f32_dpp %[r], %[h], -%[s2] " CL_ROT1 \
  "v_fmac_f32 %[d], 0.5, %[r]\n\t" \
  "v_add_f32 %[acc], %[r], %[r]\n\t" \
  "v_fma_f32 %[h], %[a0], %[d], %[dm]\n\t" \
  OFF \
  "v_add_f32_dpp %[s1], %[d], %[m1] " CL_ROT1 \
  "v_add_f32_dpp %[s2], %[d], %[m2] " CL_ROT2 \
  "v_mul_f32_dpp %[p], %[d], %[h2] " CL_ROT1 \
  "v_fmac_f32_dpp %[p], %[d], -%[h1] " CL_ROT2 \
  "v_fmac_f32_dpp %[p], %[h], %[s1] " CL_ROT2 \
  "v_fmac_f32_dpp %[p], %[h], -%[s2] " CL_ROT1 \
  "v_fmac_f32 %[h], %[al], %[p]\n\t" \
  "v_mul_f32_dpp %[r], %[d], %[g2] " CL_ROT1 \
  "v_fmac_f32_dpp %[r], %[d], -%[g1] " CL_ROT2 \
  "v_fmac_f32_dpp %[r], %[h], %[s1] " CL_ROT2 \
  "v_fmac_f32_dpp %[r], %[h], -%[s2] " CL_ROT1 \
  "v_add_f32 %[d], %[k1], %[r]\n\t" \
  "v_fmac_f32 %[acc], 2.0, %[r]\n\t" \
  "v_fma_f32 %[h], %[a0], %[d], %[de]\n\t" \
  OFF \
  "v_add_f32_dpp %[s1], %[d], %[m1] " CL_ROT1 \
  "v_add_f32_dpp %[s2], %[d], %[m2] " CL_ROT2 \
  "v_mul_f32_dpp %[p], %[d], %[h2] " CL_ROT1 \
  "v_fmac_f32_dpp %[p], %[d], -%[h1] " CL_ROT2 \
  "v_fmac_f32_dpp %[p], %[h], %[s1] " CL_ROT2 \
  "v_fmac_f32_dpp %[p], %[h], -%[s2] " CL_ROT1 \
  "v_fmac_f32 %[h], %[al], %[p]\n\t" \
  "v_mul_f32_dpp %[r], %[d], %[g2] " CL_ROT1 \
  "v_fmac_f32_dpp %[r], %[d], -%[g1] " CL_ROT2 \
  "v_fmac_f32_dpp %[r], %[h], %[s1] " CL_ROT2 \
  "v_fmac_f32_dpp %[r], %[h], -%[s2] " CL_ROT1 \
  "v_add_f32 %[acc], %[acc], %[r]"
#define CL_STAGE_OPERANDS \
  : [d] "=&v"(d), [g1] "=&v"(g1), [g2] "=&v"(g2), [h] "=&v"(h), [s1] "=&v"(s1), [s2] "=&v"(s2), [p] "=&v"(p), \
  [r] "=&v"(r), [acc] "=&v"(acc) \
  : [k1] "v"(k1), [a0] "v"(K.a0), [a1] "v"(K.a1), [a2] "v"(K.a2), [al] "v"(K.al), [m1] "v"(m1), [m2] "v"(m2), \
  [h1] "v"(h1), [h2] "v"(h2), [gb] "v"(gb), [gc] "v"(gc), [dm] "v"(dmid), [de] "v"(dend)
struct StageConst {
  float a0, a1, a2, al;  // the field matrix's row against components c, c + 1, c + 2; alpha
};
template <bool DG>
__device__ __forceinline__ float stage_increments(const StageConst& K, float k1, const Rot<double>& m,
                                                  const Rot<double>& h0, double gb, double gc, float dmid,
                                                  float dend) {
  const float m1 = (float)m.b, m2 = (float)m.c, h1 = (float)h0.b, h2 = (float)h0.c;
  float d, g1, g2, h, s1, s2, p, r, acc;
  if constexpr (DG)
    asm(CL_STAGES("") CL_STAGE_OPERANDS);
  else
    asm(CL_STAGES("v_fmac_f32_dpp %[h], %[d], %[a1] " CL_ROT1 "v_fmac_f32_dpp %[h], %[d], %[a2] " CL_ROT2)
            CL_STAGE_OPERANDS);
  return acc;
}

template <class T>
__device__ __forceinline__ T comp(V3<T> v, int c) {
  return c == 0 ? v.x : (c == 1 ? v.y : (c == 2 ? v.z : T(0)));
}

// Per-lane constants of one layer component.  Fields carry the factor
// g = -gamma dt / (1 + alpha^2), so that dm of a step is m x (h + alpha m x h).
struct CLConst {
  double g, hb, hb1, hb2;         // the factor; constant field at c, c + 1, c + 2
  double an0, an1, an2;           // anisotropy axis at c, c + 1, c + 2
  Rot<double> A0, A1, A2;         // rows c, c + 1, c + 2 of the field's constant matrix (demagnetisation,
                                  // constant first-order anisotropy) against components c, c + 1, c + 2
  double alpha;
  double jn[2];                   // bilinear IEC towards neighbour n (constant J)
  // binary64 kernels: the layer's scalar drives (constant parts) and spin
  // torques
  double k2, bI, bFL, bDL, bT, bFL2, bDL2;  // k2: 4 g K2 / Ms
  double bJ2[2];                  // 2 g J2 / (Ms t) towards neighbour n
  double Db[2], Dc[2];            // -g / (Ms t) times components c + 1, c + 2 of the IDMI vector of neighbour n
  double dp[2][3];                // dipole tensor rows towards neighbour n
  double ginv_ms, ginv_mst;       // g / Ms, g / (Ms t)
  Rot<double> ref, ref2;          // reference vectors: fixed (for the torque and the classic resistance), secondary
  Rot<double> pol;                // the torque's polariser where it is fixed, else 0
  double wp[2];                   // 1 where the polariser is neighbour n, else 0
  // spin torques, 0 on layers without them.  STT: factors of p and m x p,
  // eta = num / den, eta where den is constant; SOT: g, g alpha, static
  // coefficients; secondary SOT: g, g alpha
  double sta, stb, num, lam, lam2, wc;
  double ga, gaa, dlt, flt, g2, g2a;
  double sig2, kick, sg0;         // 2 alpha kB / (Ms V gamma), -gamma / (1 + alpha^2) sqrt(dt), kick sqrt(sig2 T)
  bool stt, alt, dyn_sot, stat_i, therm;  // STT; its alternative form; SOT from drivers; current-driven torque; thermal
};

// The drives of one stage time as a lane sees them: its (scaled) field
// component and its layer's scalar slots.
struct CLSpin {
  Rot<double> B, Q;               // the field with a p, and (b - alpha a) p
};
struct CLRows {
  Rot<double> a, b, c;            // rows c, c + 1, c + 2
};
struct CLDrive {
  double H;                       // with scalar drives: with all that the stage's m does not change
  double kd, k2;                  // 2 g K / Ms beyond the constant matrix's, 4 g K2 / Ms
  double I, FL, DL, T, FL2, DL2;
  double J2[2];                   // 2 g J2 / (Ms t)
};

// Sine of a drive's phase, carried from stage to stage: s and c are sine and
// cosine at the present stage time, sh = sin w and cm = cos w - 1 for w half
// a step's advance.  Turning by half a step takes six operations where a
// binary64 sine takes over a hundred; the phase is set again from its own
// time at every step whose index is a multiple of CL_BLOCK (in the reference's
// order of roundings), so what the turns add stays below 2e-15 of the
// amplitude, less than the rounding of the phase itself after some ten
// periods.  Setting it by step index makes a run independent of how it is cut
// into slices.
struct Osc {
  double s, c, sh, cm;
  __device__ __forceinline__ void half() {
    const double s0 = s, c0 = c;
    s = s0 + fma(s0, cm, c0 * sh);
    c = c0 + fma(c0, cm, -(s0 * sh));
  }
};
// (out of line: one copy per kernel, called once per block of steps)
static __device__ __noinline__ double2 osc_at(double f, double phase, double t) {
  double2 r;
  sincos(2 * M_PI * t * f + phase, &r.x, &r.y);
  return r;
}
__device__ __forceinline__ bool sine_kind(int type) {
  return type == CMTJ_SINE || type == CMTJ_POSINE || type == CMTJ_HALFSINE;
}

// Sum over two 16-lane rows of each half wave (ROWS 16), or over the halves
// (ROWS 32), of a value that is the same in all lanes of a row (half).
template <int ROWS>
__device__ __forceinline__ double add_rows(double v) {
  const unsigned long long u = (unsigned long long)__double_as_longlong(v);
  const unsigned lo = (unsigned)u, hi = (unsigned)(u >> 32);
  // swapped against itself: the first result holds the even row's value in
  // both rows of a pair, the second the odd row's
  const auto l = (ROWS == 16) ? __builtin_amdgcn_permlane16_swap(lo, lo, false, false)
                              : __builtin_amdgcn_permlane32_swap(lo, lo, false, false);
  const auto h = (ROWS == 16) ? __builtin_amdgcn_permlane16_swap(hi, hi, false, false)
                              : __builtin_amdgcn_permlane32_swap(hi, hi, false, false);
  return __longlong_as_double((long long)(((unsigned long long)h[0] << 32) | l[0])) +
         __longlong_as_double((long long)(((unsigned long long)h[1] << 32) | l[1]));
}

// What the waves of a dipole-coupled group share: the elements' top-layer m
// scaled by their source strengths, in two copies taken in turn (one barrier
// a step: a wave writes a copy again only after the barrier of the step
// between, which every wave reaches with its reads of that copy done), and a
// word per wave for the decisions the waves take together.
template <int GW, int EPW>
struct GroupClLds {
  alignas(32) double sm[2][GW * EPW][4];
  uint32_t word[GW];
};

// The barrier between LDS writes and other waves' reads; global stores in
// flight (log entries) are not waited for.
__device__ __forceinline__ void lds_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// ND: number of time-dependent records when fixed at compile time (exact
// kernels), -1 to read it from the group.  F64: every stage in binary64
// (the drop-in's arithmetic) instead of the anchored binary32 increments.
// LOGF: 0 reads the log layout from the group, 2 too but of binary32 entries;
// 1 compiles in m_x of every
// layer, the classic resistance and binary32 entries (the PIMM sweep's log).
// STK: the instances are members of electrically coupled stacks
// (Stack<T>::runSimulationKCL / runSimulationNonKCL with delayed coupling,
// core/stack.hpp:305-410): stack s on lanes [s pad, s pad + members x 4L)
// of one wave, member j on the 4L lanes from 4L j; the pair couplings come
// from the members' magnetisations at the start of the step and the stack
// current replaces the members' current at every stage, as in k_junction's
// stack form (binary64 only).
// GW: workgroup b of GW waves is dipole-coupled group b (GroupInteraction,
// core/reservoir.hpp:121-230, Kanao and Nomura coupling; binary64 RK4),
// element e on the 4L lanes from 4L e, at most GW 64/(4L) elements; the field
// of the step's other elements joins the frozen terms (see group_field_cl).
//
// What bounds it: with at most one wave per SIMD a step takes four cycles per
// instruction the wave issues (binary64 and binary32 alike, wait states
// included), times the steps of the longest instance.  The step is laid out
// for few instructions and few lane moves: a lane keeps its layer's whole
// start-of-step m and forms the field and the first torque at components
// c + 1 and c + 2 itself, so that one pair of lane moves per stage (the
// stage's m) is all that crosses lanes; the LLG torque is m x (h + alpha m x h)
// with the field pre-scaled; the length correction is a polynomial (a
// binary64 square root and division took a quarter of a binary64 step).
// Measured before and after all of it: R(H) loop, 101 one-layer instances x
// 50,000 binary64 steps 21.4 -> 10.0 ms; 512 oscillators x 50,000 steps 44.1 ->
// 10.7 ms; 1023 one-layer instances under a sine field x 10,000 steps 14.9 ->
// 2.6 ms (three binary64 sines a step before, see Osc).
template <int L, uint32_t FM, int ND, bool F64 = false, int SOLVER = CMTJ_RK4, int LOGF = 0, bool STK = false,
          int GW = 0, bool NF = false>
__global__ __launch_bounds__(64 * (GW > 0 ? GW : 1)) void k_junction_cl(GroupArgs g) {
  // the compiled-in layout's R is layer 0 against layer 1
  static_assert(LOGF != 1 || (L == 2 && (FM & F_EXACT) && (FM & F_IEC)), "two coupled layers");
  static_assert(!STK || (F64 && LOGF == 0 && !(FM & F_KSTEP)),
                "stacks: binary64, the group's log layout, every step through the same code");
  static_assert(!NF || (F64 && SOLVER != CMTJ_RK4 && (FM & F_THERMAL)), "binary32 normals: stochastic solvers");
  static_assert(GW == 0 || (F64 && SOLVER == CMTJ_RK4 && LOGF == 0 && !STK && L <= 2 && !(FM & F_KSTEP)),
                "groups: binary64 RK4, the group's log layout, every step through the same code");
  static_assert(L == 1 || L == 2 || L == 4, "4L lanes per instance must divide a 16-lane DPP row");
  static_assert(F64 || !(FM & (F_STT | F_SOT | F_SOT2 | F_DYN | F_THERMAL | F_ANIS2 | F_IEC2 | F_DEMAG_OFF |
                                F_IDMI | F_DIPOLE)),
                "binary64 kernels only");
  static_assert(SOLVER == CMTJ_RK4 || (F64 && (SOLVER == CMTJ_EULER_HEUN || SOLVER == CMTJ_HEUN)),
                "RK4, or Euler-Heun / Heun in binary64");
  // callback-driver samples are laid out for RK4's three stage times
  static_assert(!(FM & F_TABLE) || (F64 && SOLVER == CMTJ_RK4), "tabulated drivers: binary64 RK4 only");
  constexpr int LPI = 4 * L;
  constexpr int NN = (L == 1) ? 0 : (L == 2) ? 1 : 2;  // neighbours of a layer: none, the other one, top and bottom
  constexpr bool DYNS = (FM & F_DYN) != 0;              // time-dependent scalar slots
  // sine phases carried from stage to stage (binary32 increments logged in
  // binary64 keep their single-precision waveforms, see PLAIN32)
  constexpr bool OSC = (F64 || LOGF == 2) && (FM & (F_DYN | F_DYNH)) != 0 && !(FM & (F_KSTEP | F_KTRAP));
  const uint32_t gl = blockIdx.x * blockDim.x + threadIdx.x;
  uint32_t inst;
  int q;
  [[maybe_unused]] const cmtj_stack* sk = nullptr;
  [[maybe_unused]] int s_j = 0, s_n = 0, s_base = 0;
  [[maybe_unused]] const cmtj_group* gp = nullptr;
  [[maybe_unused]] int g_n = 0, g_e = 0, g_top = 0;
  bool own = true;  // the lanes hold an instance
  if constexpr (GW > 0) {
    // every lane stays for the barriers and lane moves: lanes past the
    // group's elements hold an element without layers (m = 0, strength 0)
    if (blockIdx.x >= g.group_n) return;
    gp = g.group + blockIdx.x;
    g_n = gp->n_elements;
    g_e = (int)(threadIdx.x / LPI);
    own = g_e < g_n;
    inst = blockIdx.x * (uint32_t)g_n + (uint32_t)(own ? g_e : 0);
    q = (int)(threadIdx.x % LPI);
    g_top = own ? gp->top[g_e] : 0;
  } else if constexpr (STK) {
    // a stack never straddles a wave (pad is a power of two of at most 64);
    // lanes past its members stay for the lane moves, as a member without
    // layers (m = 0)
    const uint32_t pad = g.stack_pad, sid = gl / pad;
    if (sid >= g.stack_n) return;
    sk = g.stack + sid;
    s_n = sk->n_junctions;
    s_j = (int)((gl % pad) / LPI);
    own = s_j < s_n;
    s_j = own ? s_j : 0;
    q = (int)(gl % LPI);
    inst = sid * (uint32_t)s_n + (uint32_t)s_j;
    s_base = (int)(threadIdx.x & ~(pad - 1));
  } else {
    inst = gl / LPI;
    if (inst >= g.n) return;
    q = (int)(gl % LPI);
  }
  const int ly = q >> 2, c = q & 3;
  const uint32_t fl = g.flags;
  const int nl = g.nl;
  const bool lact = own && ly < nl;   // the lane's layer exists
  const bool live = lact && c < 3;    // the lane holds a component
  const int lyr = lact ? ly : 0;
  const uint32_t jid = g.order[inst];
  const cmtj_junction* J = g.js + jid;
  const uint32_t nsteps = J->n_steps;
  const uint32_t W = J->write_every;
  const uint32_t NE = J->n_entries;
  const double dt = J->dt;
  const uint64_t lbase = J->log_offset;
  const bool logging = (g.log != nullptr) && g.log_mask != 0;
  const bool f32log = (LOGF == 1) ? true : g.log_f32;
  const uint32_t esize = f32log ? 4u : 8u;
  char* const lp = logging ? (char*)g.log + lbase * esize : nullptr;
  const uint64_t cs = (uint64_t)NE * esize;
  const double Rp = J->Rp, Rap = J->Rap;
  [[maybe_unused]] const double hR = (Rap - Rp) / 2.0;
  [[maybe_unused]] const uint64_t seed = J->seed, stream = J->stream;
  constexpr int sps = 3;
  const bool hasB = lact && ly > 0, hasT = lact && ly + 1 < nl;
  // whether neighbour n exists, and whether it is the top one (L = 2: the
  // other layer of the pair, whichever side it is on; L = 4: top, bottom)
  auto has_nb = [&](int n) { return L == 2 ? (hasT || hasB) : (n == 0 ? hasT : hasB); };
  auto nb_top = [&](int n) { return L == 2 ? hasT : n == 0; };
  const uint32_t gshift = (threadIdx.x & 63u) & ~(uint32_t)(LPI - 1);  // the instance's first lane in the wave
  const int cc = (c < 3) ? c : 0;  // (a pad lane's values are never used)
  const int c1 = (cc == 2) ? 0 : cc + 1, c2 = (cc == 0) ? 2 : cc - 1;

  // per-lane constants (loadLayer parameters of this layer, this component)
  CLConst K;
  Rot<double> m;  // start-of-step m of the lane's layer
  {
    const cmtj_layer& Ly = g.layers[J->layer_offset + lyr];
    LP<double> P;
    DV<double> base;
    V3<double> m3;
    load_layer<double>(Ly, g.c, P, base, m3);
    const double z = 0.0;
    m.a = live ? comp(m3, c) : z;
    K.g = P.gconv * dt;
    K.hb = live ? K.g * comp(base.H, c) : z;
    K.hb1 = live ? K.g * comp(base.H, c1) : z;
    K.hb2 = live ? K.g * comp(base.H, c2) : z;
    K.an0 = live ? comp(P.anis, c) : z;
    K.an1 = live ? comp(P.anis, c1) : z;
    K.an2 = live ? comp(P.anis, c2) : z;
    const double gm = K.g * P.ms_mu0;
    K.alpha = P.alpha;
    K.ginv_ms = K.g * P.inv_ms;
    K.ginv_mst = K.g * P.inv_mst;
    K.k2 = live ? (4.0 * base.K2) * K.ginv_ms : z;
    K.bI = base.I;
    K.bFL = base.FL;
    K.bDL = base.DL;
    K.bT = base.T;
    K.bFL2 = base.FL2;
    K.bDL2 = base.DL2;
#pragma unroll
    for (int n = 0; n < 2; ++n) {
      const bool on = live && has_nb(n), top = nb_top(n);
      K.jn[n] = on ? (top ? base.Jt : base.Jb) * K.ginv_mst : z;
      K.bJ2[n] = on ? (2.0 * (top ? base.J2t : base.J2b)) * K.ginv_mst : z;
      K.Db[n] = on ? -K.ginv_mst * comp(top ? base.Dt : base.Db, c1) : z;
      K.Dc[n] = on ? -K.ginv_mst * comp(top ? base.Dt : base.Db, c2) : z;
      K.dp[n][0] = on ? (top ? CL_ENTRY(P.Nt, cc, cc) : CL_ENTRY(P.Nb, cc, cc)) * gm : z;
      K.dp[n][1] = on ? (top ? CL_ENTRY(P.Nt, cc, c1) : CL_ENTRY(P.Nb, cc, c1)) * gm : z;
      K.dp[n][2] = on ? (top ? CL_ENTRY(P.Nt, cc, c2) : CL_ENTRY(P.Nb, cc, c2)) * gm : z;
    }
    {
      const double k2 = K.g * ((2.0 * base.K) * P.inv_ms);
      auto row = [&](double an, int r) -> Rot<double> {
        return {live ? k2 * an * K.an0 - CL_ENTRY(P.N, r, cc) * gm : z, live ? k2 * an * K.an1 - CL_ENTRY(P.N, r, c1) * gm : z,
                live ? k2 * an * K.an2 - CL_ENTRY(P.N, r, c2) * gm : z};
      };
      K.A0 = row(K.an0, cc);
      K.A1 = row(K.an1, c1);
      K.A2 = row(K.an2, c2);
    }
    const V3<double> r1 = mk<double>(Ly.ref[0], Ly.ref[1], Ly.ref[2]);
    const V3<double> r2 = mk<double>(Ly.ref2[0], Ly.ref2[1], Ly.ref2[2]);
    K.ref = {live ? comp(r1, c) : z, live ? comp(r1, c1) : z, live ? comp(r1, c2) : z};
    K.ref2 = {live ? comp(r2, c) : z, live ? comp(r2, c1) : z, live ? comp(r2, c2) : z};
    K.sig2 = P.sig2;
    const int bits = g.lbits[lyr];
    const int rt = bits & 3;
    const bool sot = live && ((bits >> 2) & 3) == 2;
    K.stt = live && ((bits >> 2) & 3) == 1;
    K.alt = ((bits >> 5) & 1) != 0;
    K.dyn_sot = sot && ((bits >> 4) & 1) != 0;
    K.stat_i = K.stt || (sot && !K.dyn_sot);
    const bool torque = K.stt || sot;
    // (component by component: a choice between two structs is a choice
    // between addresses, which would keep K in scratch memory)
    const bool fixed = torque && rt == CMTJ_REF_FIXED;
    K.pol = {fixed ? K.ref.a : z, fixed ? K.ref.b : z, fixed ? K.ref.c : z};
#pragma unroll
    for (int n = 0; n < 2; ++n)
      K.wp[n] = (torque && has_nb(n) && rt == (nb_top(n) ? (int)CMTJ_REF_TOP : (int)CMTJ_REF_BOTTOM)) ? 1.0 : z;
    const double cs_ = K.stt ? P.conv * dt * P.stt_pref : z;
    K.sta = cs_ * P.beta;
    K.stb = -cs_ * P.kappa;
    K.lam = P.lam;
    K.lam2 = P.lam2;
    K.num = K.alt ? P.P : P.P * P.lam2;
    K.wc = K.num / (P.lam2 + 1.0);
    K.ga = sot ? K.g : z;
    K.gaa = K.ga * K.alpha;
    K.dlt = K.stat_i ? P.dl_t : z;
    K.flt = K.stat_i ? P.fl_t : z;
    K.g2 = K.dyn_sot ? K.g : z;
    K.g2a = K.g2 * K.alpha;
    // a drive of a torque that the layer does not have stays out of it
    K.bI = K.stat_i ? K.bI : z;
    K.bFL = K.dyn_sot ? K.bFL : z;
    K.bDL = K.dyn_sot ? K.bDL : z;
    K.bFL2 = K.dyn_sot ? K.bFL2 : z;
    K.bDL2 = K.dyn_sot ? K.bDL2 : z;
    K.therm = live && ((bits >> 6) & 1) != 0;
    K.kick = P.gconv * sqrt(dt);
    K.sg0 = K.therm ? sqrt(K.sig2 * K.bT) * K.kick : z;
  }
  // A multiple of m added to the field changes no torque, so a lane takes the
  // matrix less the identity times its row c + 1's diagonal entry, which that
  // row then has no more (binary32 increments share their field between lanes
  // and stay as they are, and so do the stochastic solvers, whose one field a
  // step gains nothing).
  constexpr bool GAUGE = F64 && SOLVER == CMTJ_RK4;
  if constexpr (GAUGE) {
    const double lam = K.A1.b;
    K.A0.a -= lam;
    K.A1.b = 0.0;
    K.A2.c -= lam;
  }
  // Anisotropy along an axis and a diagonal demagnetising tensor, in every lane
  // of the wave: the matrix is diagonal, and a field evaluation takes two FMAs
  // instead of eight (binary32 increments: one instead of three).  Decided per
  // wave, with the same bits either way (a zero entry adds a zero).  Before and
  // after: R(H) loop 12.6 -> 10.0 ms, PIMM sweep 44.6 -> 40.4 ms, oscillators
  // 13.2 -> 10.7 ms, sine field 3.0 -> 2.6 ms.
  constexpr bool DGSET = SOLVER == CMTJ_RK4 && !(FM & (F_DEMAG_OFF | F_IEC2));
  const bool diag = DGSET && __ballot(K.A0.b != 0.0 || K.A0.c != 0.0 || K.A1.a != 0.0 || K.A1.c != 0.0 ||
                                      K.A2.a != 0.0 || K.A2.b != 0.0) == 0ull;
  // Binary32 sets that take waveforms run in two forms, by the log's entries.
  // With binary32 entries (LOGF 2): carried binary64 phases and the increments
  // of stage_increments.  With binary64 entries: single-precision waveforms and
  // increments about the anchor in the lane's own order, the slower form and
  // the one further off (256 one-layer instances under a sine field x 5,000
  // steps: 1.32 against 0.26 us per step, 2.0e-8 against 4.8e-9 of m from the
  // binary64 run), kept so that binary64 entries keep their values to 1e-9: the
  // other form moves them by 3e-8.
  constexpr bool PLAIN32 = !F64 && LOGF != 2 && !(FM & F_KSTEP);
  [[maybe_unused]] float p_an = 0, p_an1 = 0, p_an2 = 0, p_nms = 0, p_ak = 0, p_al = 0, p_g = 0;
  [[maybe_unused]] double ig = 0.0;
  if constexpr (PLAIN32) {
    LP<double> P;
    DV<double> base;
    V3<double> m3;
    load_layer<double>(g.layers[J->layer_offset + lyr], g.c, P, base, m3);
    p_an = (float)K.an0;
    p_an1 = (float)K.an1;
    p_an2 = (float)K.an2;
    const V3<double> nd = mk<double>(P.N[0], P.N[4], P.N[8]);
    p_nms = live ? (float)(comp(nd, c) * P.ms_mu0) : 0.f;
    p_ak = (float)(K.an0 * ((2.0 * base.K) * P.inv_ms));
    p_al = (float)P.alpha;
    p_g = (float)P.gconv * (float)dt;
    ig = 1.0 / K.g;
  }
  // eta's denominator is lam2 + 1 on every STT lane of the wave (lambda = 1,
  // the usual spacer): the torque then needs no division
  const bool den_const = (FM & F_STT) != 0 && __ballot(K.stt && (K.alt || K.lam2 != 1.0)) == 0ull;
  // whether a lane of the wave takes its polariser from a neighbour, and
  // whether a step reads the neighbours at all (else only a log entry's R
  // does).  Stochastic solvers only: an RK4 step gains nothing from the branch.
  constexpr bool RK = SOLVER == CMTJ_RK4;
  const bool nb_pol = RK || (NN > 0 && (FM & (F_STT | F_SOT)) != 0 && __ballot(K.wp[0] != 0.0 || K.wp[1] != 0.0) != 0ull);
  const bool nb_step = RK || STK || CMTJ_HAS(F_IEC) || CMTJ_HAS(F_IEC2) || CMTJ_HAS(F_IDMI) || CMTJ_HAS(F_DIPOLE) || nb_pol;
  // spin torques under constant currents: a p and (b - alpha a) p of a fixed
  // polariser are constants, of a neighbour two factors (see spin below)
  constexpr bool SPC = (FM & (F_STT | F_SOT)) != 0 && !DYNS && !STK;
  static_assert(!SPC || !(FM & F_SOT), "constant currents: STT");
  [[maybe_unused]] Rot<double> Q0 = {0.0, 0.0, 0.0};
  [[maybe_unused]] double swa[2] = {0.0, 0.0}, swb[2] = {0.0, 0.0};
  if constexpr (SPC) {
    const double w = den_const ? K.bI * K.wc : 0.0;
    const double a = K.sta * w, b = fma(-K.alpha, a, K.stb * w);
    K.hb = fma(a, K.pol.a, K.hb);
    K.hb1 = fma(a, K.pol.b, K.hb1);
    K.hb2 = fma(a, K.pol.c, K.hb2);
    Q0 = {b * K.pol.a, b * K.pol.b, b * K.pol.c};
#pragma unroll
    for (int n = 0; n < 2; ++n) {
      swa[n] = a * K.wp[n];
      swb[n] = b * K.wp[n];
    }
  }
  // the length correction's coefficients, held in registers (as literals they
  // would be moved to one at every step)
  double len2 = 0.375, len3 = -0.3125, len4 = 0.2734375;
  asm("" : "+v"(len2), "+v"(len3), "+v"(len4));
  // the lane's share of the -1 in |m|^2 - 1: binary64, the pad lane's of a sum
  // over the quad; binary32, every component's own sum
  const double unit = (F64 ? lact && c == 3 : live) ? -1.0 : 0.0;
  constexpr int NR = (ND >= 0) ? ND : DREG;  // records kept in registers
  static_assert(NR <= DREG, "at most DREG records in registers");
  DynRec dr[DREG];
  Osc osc[DREG];
  bool sel[DREG];  // whether record k feeds this lane (its field component, or a slot of its layer)
  double win_lo = __builtin_inf(), win_hi = -__builtin_inf();
  // whether a record feeds this lane: its field component, a scalar slot of
  // its layer, the coupling towards an existing neighbour, or this component
  // of an IDMI vector
  auto feeds_lane = [&](int meta) -> bool {
    const int slot = (meta >> 8) & 0xff;
    if ((meta & 0xff) == CMTJ_CONSTANT || !lact || !(((meta >> 16) & 0xff) >> ly & 1)) return false;
    if (slot < CMTJ_SLOT_K) return c < 3 && slot % 3 == c;
    if (slot == CMTJ_SLOT_CURRENT) return K.stat_i;
    if (slot == CMTJ_SLOT_FL || slot == CMTJ_SLOT_DL || slot == CMTJ_SLOT_FL2 || slot == CMTJ_SLOT_DL2)
      return K.dyn_sot;
    if (slot == CMTJ_SLOT_J_TOP || slot == CMTJ_SLOT_J2_TOP) return hasT;
    if (slot == CMTJ_SLOT_J_BOTTOM || slot == CMTJ_SLOT_J2_BOTTOM) return hasB;
    // (a component of the IDMI vector turns into field components across it)
    if (slot >= CMTJ_SLOT_IDMI_TOP && slot < CMTJ_SLOT_IDMI_BOTTOM)
      return hasT && c < 3 && slot - CMTJ_SLOT_IDMI_TOP != c;
    if (slot >= CMTJ_SLOT_IDMI_BOTTOM && slot < CMTJ_NSLOT)
      return hasB && c < 3 && slot - CMTJ_SLOT_IDMI_BOTTOM != c;
    return true;
  };
#pragma unroll
  for (int k = 0; k < DREG; ++k) {
    osc[k] = Osc{0.0, 0.0, 0.0, 0.0};
    if (k < NR && (ND >= 0 || k < g.ndyn)) {
      dr[k] = load_rec<FM>(g.dyn + (size_t)k * g.n + inst);
      win_lo = fmin(win_lo, dr[k].p1);
      win_hi = fmax(win_hi, dr[k].p2);
      sel[k] = feeds_lane(g.dmeta[k]);
      if constexpr (OSC) {
        if ((FM & F_KSINE) || sine_kind(g.dmeta[k] & 0xff)) {
          const double w = M_PI * dr[k].p1 * dt;  // half a step's advance
          const double sw = sin(0.5 * w);
          // a lane the record does not feed carries zeros: what is not finite
          // stays with the layer it drives
          osc[k].sh = sel[k] ? sin(w) : 0.0;
          osc[k].cm = sel[k] ? -2.0 * sw * sw : 0.0;
          dr[k].A = sel[k] ? dr[k].A : 0.0;
        }
      }
    } else {
      dr[k] = DynRec{0.0, 0.0, 0.0, 0.0, 0, 0};
      sel[k] = false;
    }
  }
  // whether a drive moves a temperature (else the noise strength is sg0), an
  // anisotropy (else it is in the constant matrix), a biquadratic coupling
  // (else it joins the matrix once a step), a field term (else one field
  // serves the stages)
  [[maybe_unused]] bool t_driven = false, k_driven = false, j2_driven = false, h_driven = false;
  auto field_slot = [](int slot) {
    return slot < CMTJ_SLOT_K || slot == CMTJ_SLOT_J_TOP || slot == CMTJ_SLOT_J_BOTTOM || slot >= CMTJ_SLOT_IDMI_TOP;
  };
  if constexpr (DYNS) {
    auto note = [&](int r) {
      const int slot = (g.dmeta[r] >> 8) & 0xff;
      t_driven |= slot == CMTJ_SLOT_TEMPERATURE;
      k_driven |= slot == CMTJ_SLOT_K;
      j2_driven |= slot == CMTJ_SLOT_J2_TOP || slot == CMTJ_SLOT_J2_BOTTOM;
      h_driven |= field_slot(slot);
    };
#pragma unroll
    for (int k = 0; k < DREG; ++k)
      if (k < NR && (ND >= 0 || k < g.ndyn)) note(k);
    for (int r = DREG; ND < 0 && !(FM & F_EXACT) && r < g.ndyn; ++r) note(r);
  }
  // The layer's normals of four steps at a time: lane c of the quad draws
  // those of step i + c (counter-based, so any lane can), and the step in turn
  // is read from lane 0, the others moving down.  A draw is most of a
  // stochastic step's instructions (650 of 840 in binary64), and the quad's
  // lanes would otherwise all make the same one.  NF: binary32 normals, those
  // of the other FP32 kernels.
  using NT = typename std::conditional<NF, float, double>::type;
  [[maybe_unused]] V3<NT> xi = mk<NT>(0, 0, 0);
  auto draw = [&](uint32_t step0) __attribute__((always_inline)) {
    if constexpr (SOLVER != CMTJ_RK4) {
      if (CMTJ_HAS(F_THERMAL)) xi = thermal_normals<NT>(seed, stream, step0 + (uint32_t)c, (uint32_t)lyr);
    }
  };
  auto next_normals = [&]() __attribute__((always_inline)) -> Rot<double> {
    auto move = [](auto tag, NT v) __attribute__((always_inline)) -> NT {
      constexpr int CTRL = decltype(tag)::value;
      if constexpr (NF)
        return dpp_f<CTRL>(v);
      else
        return dpp_d<CTRL>(v);
    };
    constexpr std::integral_constant<int, QP_BC0> BC{};
    constexpr std::integral_constant<int, QP_NEXT> NX{};
    const NT x = move(BC, xi.x), y = move(BC, xi.y), z = move(BC, xi.z);
    xi = mk<NT>(move(NX, xi.x), move(NX, xi.y), move(NX, xi.z));
    const NT a = (c == 0) ? x : (c == 1) ? y : z, b = (c == 0) ? y : (c == 1) ? z : x, d = (c == 0) ? z : (c == 1) ? x : y;
    return {(double)a, (double)b, (double)d};
  };
  // log layout of this lane (logLayerParams, core/junction.hpp:1580-1636):
  // its m channel, if it writes one, and the resistance channels after the
  // m channels of all layers
  const int lmask = logging ? ((LOGF == 1) ? (CMTJ_LOG_MX | CMTJ_LOG_MR) : g.log_mask) : 0;
  const int mrm = (LOGF == 1) ? CMTJ_MR_CLASSIC : g.mr_mode;
  const int nm = ((lmask & CMTJ_LOG_MX) ? 1 : 0) + ((lmask & CMTJ_LOG_MYZ) ? 2 : 0);
  const int mch = (lmask & CMTJ_LOG_MX) ? c : c - 1;
  const bool wm = live && nm && mch >= 0 && ((lmask & CMTJ_LOG_MYZ) || c == 0);
  const uint64_t om = wm ? (uint64_t)(ly * nm + mch) * cs : 0;
  const uint64_t orr = (uint64_t)(nl * nm) * cs;
  const bool classic = (lmask & CMTJ_LOG_MR) && mrm == CMTJ_MR_CLASSIC;
  const bool strip = (lmask & CMTJ_LOG_MR) && mrm == CMTJ_MR_STRIP;
  // one channel per lane, so that an entry of m and the classic R is one
  // store: the m channels on the lanes of their components, R on a lane that
  // writes no m (compiled-in layout: the y lane of layer 0; else layer 0's
  // pad lane, which takes it from the x lane)
  const bool rlane = own && classic && q == (LOGF == 1 ? 1 : 3);
  const bool wlog = wm || rlane;
  char* const lpl = lp + (rlane ? orr : om);  // the lane's entry 0
  // STRIP coefficients of the lane's layer, read once (the descriptors may
  // sit in host-mapped memory); 0.5 AHE and AMR_Y + SMR_Y are the reference's
  // own first products, so the entries round as before
  double sRx0 = 0.0, sAMRX = 0.0, sSMRX = 0.0, sRy0 = 0.0, sAHE2 = 0.0, sXY = 0.0;
  if (strip && lact && c == 0) {
    sRx0 = J->Rx0[ly];
    sAMRX = J->AMR_X[ly];
    sSMRX = J->SMR_X[ly];
    sRy0 = J->Ry0[ly];
    sAHE2 = 0.5 * J->AHE[ly];
    sXY = J->AMR_Y[ly] + J->SMR_Y[ly];
  }
  uint32_t k = 0;
  int code = CMTJ_OK, nan_layer = -1;
  uint32_t i = 0, iend = nsteps;
  cmtj_state* const S = g.state ? g.state + jid : nullptr;
  if (S) {  // resume: state of the previous slice
    m.a = live ? S->m[lyr][c] : 0.0;
    i = S->step;
    k = S->entries;
    code = S->code;
    nan_layer = (code == CMTJ_OK) ? -1 : S->nan_layer;
    iend = (code != CMTJ_OK) ? i : (uint32_t)min((uint64_t)nsteps, (uint64_t)i + g.slice);
  }
  m = rot3(m.a);
  // lanes whose NaN stops a run: component x of every existing layer
  const unsigned long long nan_lanes = __ballot(live && c == 0);
  // neighbour layers' m (start of step): lanes without a neighbour in the
  // instance hold 0 from here on, and the per-step row shifts (dpp_keep)
  // leave them alone.  Lanes of layers the junction does not have (nl < L)
  // hold m = 0 throughout (no field term moves a zero vector), so the
  // existing layer next to them reads 0 from them.
  constexpr int BANK_B = neighbour_banks<L, false>(), BANK_T = neighbour_banks<L, true>();
  Rot<double> nb[2] = {{0.0, 0.0, 0.0}, {0.0, 0.0, 0.0}};
  auto neighbours = [&](Rot<double> (&out)[2], double v) __attribute__((always_inline)) {
    if constexpr (L == 2) {  // the two layers swap: one register, both shifts
      double x = dpp_keep<DPP_ROW_SHR4, BANK_B>(out[0].a, v);
      x = dpp_keep<DPP_ROW_SHL4, BANK_T>(x, v);
      out[0] = rot3(x);
    } else if constexpr (L == 4) {
      out[0] = rot3(dpp_keep<DPP_ROW_SHL4, BANK_T>(out[0].a, v));
      out[1] = rot3(dpp_keep<DPP_ROW_SHR4, BANK_B>(out[1].a, v));
    }
  };
  neighbours(nb, m.a);
  // stacks: the member's constants and this step's stack current (stage
  // times t, t + dt/2, t + dt) with the stack log's I_j and C_j_{j+1}
  [[maybe_unused]] StackLane sl;
  [[maybe_unused]] int s_ti = 0;
  [[maybe_unused]] double sI[3] = {0.0, 0.0, 0.0};
  [[maybe_unused]] double sIlog = 0.0, sClog = 0.0;
  [[maybe_unused]] double s_w = 0.0;
  [[maybe_unused]] bool s_kcl = false, s_const = false;  // of the whole wave
  [[maybe_unused]] unsigned long long s_mask = 0ull;  // the stack's lanes
  [[maybe_unused]] Rot<double> s_pol = {0.0, 0.0, 0.0};
  if constexpr (STK) {
    sl = stack_lane(sk, s_j, s_n);
    s_ti = sk->top[s_j];
    s_mask = ((g.stack_pad >= 64) ? ~0ull : ((1ull << g.stack_pad) - 1)) << (unsigned)s_base;
    const V3<double> pv = mk<double>(sl.pol[0], sl.pol[1], sl.pol[2]);
    s_pol = {comp(pv, c), comp(pv, c1), comp(pv, c2)};
    // KCL: the stack's current is I0 (1 + sum_j C_j), C_j = c_j (d_j +- d_{j+1});
    // taken by members, d_j times c_j +- c_{j-1}, no member needs another's d
    const double cp = (own && s_j > 0) ? sk->coupling[s_j - 1] : 0.0;
    s_w = own ? (sl.series ? sl.cj + cp : sl.cj - cp) : 0.0;
    s_kcl = __ballot(!sl.kcl) == 0ull;
    s_const = __ballot(sl.current.type != CMTJ_CONSTANT) == 0ull;
  }

  // Groups: field of the other elements on this lane's component of its
  // element's top layer, from the start-of-step m (stepFunctionalSolver,
  // core/reservoir.hpp:126-147),
  //   sum_j s_j (3 (m_j . r) r / |r|^5 - m_j / |r|^3),  r = r_e - r_j,
  // s_j = (Ms_j / mu0) V_j (computeDipoleInteraction, :79-96) or Ms_j V_j /
  // mu0 / (4 pi) (computeDipoleInteractionNoumra, :106-119).  The geometry is
  // constant, so a lane keeps each of its pairs as four numbers, u = r
  // sqrt(3 / |r|^5) and w = 1 / |r|^3, and a pair costs nine FMAs on s_j m_j
  // from LDS: u (u . sm) - w sm.  The eight lanes of an octet take the
  // sources j = o (mod 8); with one-layer elements an octet is two elements
  // and a lane sums its sources for both (each source read once: with one
  // element a lane, reading the sources took longer than the FMAs).  The
  // octet's sums meet by lane moves, component c ends in lane c.
  constexpr int GS = (GW > 0) ? GW * (64 / LPI) / 8 : 1;  // sources per lane
  constexpr int GP = (L == 1) ? 2 : 1;                    // elements per octet
  [[maybe_unused]] Rot<double> gu[GP][GS];
  [[maybe_unused]] double gw[GP][GS];
  [[maybe_unused]] double g_s = 0.0;
  [[maybe_unused]] int g_buf = 0;
  [[maybe_unused]] bool g_lane = false, g_sink = false;  // the lane holds a component of a coupled top layer; its m
  __shared__ GroupClLds<(GW > 0 ? GW : 1), (GW > 0 ? 64 / LPI : 1)> glds;
  if constexpr (GW > 0) {
    // an uncoupled group takes no field whatever its positions: nothing is
    // checked about them, and two elements may share one
    g_lane = live && ly == g_top && gp->interaction != CMTJ_INTERACTION_NULL;
    g_sink = c < 3 && ly == g_top;
    const int o = (int)(threadIdx.x & 7u);
    if (g_lane) {
      const cmtj_layer& Ly = g.layers[J->layer_offset + g_top];
      const double V = Ly.thickness * Ly.cell_surface;
      g_s = (gp->interaction == CMTJ_INTERACTION_KANAO) ? (Ly.Ms / g.c.mu0) * V : Ly.Ms * V / g.c.mu0 / (4 * M_PI);
    }
#pragma unroll
    for (int p = 0; p < GP; ++p) {
      const int e = (p == 0) ? g_e : (g_e ^ 1);
#pragma unroll
      for (int s = 0; s < GS; ++s) {
        const int j = 8 * s + o;
        const bool on = e < g_n && j < g_n && j != e;
        const int ei = on ? e : 0, ji = on ? j : 0;
        const double dx = gp->pos[ei][0] - gp->pos[ji][0], dy = gp->pos[ei][1] - gp->pos[ji][1],
                     dz = gp->pos[ei][2] - gp->pos[ji][2];
        // the host has checked a coupled group's |r| against the reference's limits
        const double il = on ? 1.0 / sqrt(dx * dx + dy * dy + dz * dz) : 0.0, il2 = il * il;
        const double f = sqrt(3.0 * (il2 * il)) * il;
        gu[p][s] = {dx * f, dy * f, dz * f};
        gw[p][s] = il2 * il;
      }
    }
  }
  auto group_field_cl = [&]() __attribute__((always_inline)) -> double {
    if constexpr (GW > 0) {
      auto& sm = glds.sm[g_buf];
      g_buf ^= 1;
      if (g_sink) sm[g_e][c] = g_s * m.a;
      lds_barrier();
      V3<double> acc[GP];
#pragma unroll
      for (int p = 0; p < GP; ++p) acc[p] = mk<double>(0, 0, 0);
      const int o = (int)(threadIdx.x & 7u);
#pragma unroll
      for (int s = 0; s < GS; ++s) {
        const double x = sm[8 * s + o][0], y = sm[8 * s + o][1], z = sm[8 * s + o][2];
#pragma unroll
        for (int p = 0; p < GP; ++p) {
          const Rot<double>& u = gu[p][s];
          const double d = fma(u.c, z, fma(u.b, y, u.a * x)), w = -gw[p][s];
          acc[p].x = fma(u.a, d, fma(w, x, acc[p].x));
          acc[p].y = fma(u.b, d, fma(w, y, acc[p].y));
          acc[p].z = fma(u.c, d, fma(w, z, acc[p].z));
        }
      }
      V3<double> h = acc[0];
      h.x += dpp_d<DPP_HALF_MIRROR>(acc[GP - 1].x);
      h.y += dpp_d<DPP_HALF_MIRROR>(acc[GP - 1].y);
      h.z += dpp_d<DPP_HALF_MIRROR>(acc[GP - 1].z);
      // over the quad: lanes 0, 1 gather x and y, lanes 2, 3 gather z
      const bool up = c >= 2;
      const double a = (up ? h.z : h.x) + dpp_d<QP_SWAP2>(up ? h.x : h.z);
      const double b = h.y + dpp_d<QP_SWAP2>(h.y);
      const double r = (c == 1 ? b : a) + dpp_d<QP_SWAP1>(c == 0 ? b : a);
      return g_lane ? K.g * r : 0.0;
    } else {
      return 0.0;
    }
  };
  // whether any wave of the group says so (every wave calls it; the next
  // step's barrier lies before the next write)
  auto group_any = [&](bool mine) __attribute__((always_inline)) -> bool {
    if constexpr (GW > 1) {
      glds.word[threadIdx.x >> 6] = mine ? 1u : 0u;
      lds_barrier();
      uint32_t any = 0;
#pragma unroll
      for (int w = 0; w < GW; ++w) any |= glds.word[w];
      return __builtin_amdgcn_readfirstlane(any) != 0u;
    } else {
      return mine;
    }
  };

  // Exact sets with few records: whether a record feeds each scalar slot the
  // set has, as weights of one FMA a slot (the general form finds a record's
  // slot by a tree of scalar branches, some 30 instructions a step).
  constexpr bool SLOTW = DYNS && (FM & F_EXACT) != 0 && ND >= 1 && ND <= 2 &&
                         !(FM & (F_ANIS2 | F_IEC | F_IEC2 | F_IDMI | F_DIPOLE | F_SOT2 | F_DYNH));
  constexpr int NW = SLOTW ? ND : 1;
  [[maybe_unused]] double wK[NW], wI[NW], wFL[NW], wDL[NW];
  if constexpr (SLOTW) {
#pragma unroll
    for (int r = 0; r < NW; ++r) {
      const int slot = (g.dmeta[r] >> 8) & 0xff;
      wK[r] = slot == CMTJ_SLOT_K ? 2.0 * K.ginv_ms : 0.0;
      wI[r] = slot == CMTJ_SLOT_CURRENT ? 1.0 : 0.0;
      wFL[r] = slot == CMTJ_SLOT_FL ? 1.0 : 0.0;
      wDL[r] = slot == CMTJ_SLOT_DL ? 1.0 : 0.0;
    }
  }
  // Trapezoids of stochastic runs: where every record of the wave stays on one
  // of its straight pieces over a block, its value there is la + lc (t - lt).
  constexpr bool LINES = SOLVER == CMTJ_EULER_HEUN && (FM & F_KTRAP) != 0 && ND >= 1;
  constexpr int NLN = LINES ? ND : 1;
  [[maybe_unused]] double la[NLN], lc[NLN], lt[NLN];
  [[maybe_unused]] bool lines = false;
  auto set_lines = [&](uint32_t a, uint32_t b) __attribute__((always_inline)) {  // steps a to b
    if constexpr (LINES) {
      const double ta = (double)a * dt, tb = (double)b * dt;
      bool ok = true;
#pragma unroll
      for (int r = 0; r < NLN; ++r) {
        const double t1 = dr[r].p1, t2 = t1 + dr[r].p2, t3 = t2 + dr[r].p3, t4 = t1 + 2 * dr[r].p2 + dr[r].p3;
        auto piece = [&](double t) { return (t < t1) ? 0 : (t <= t2) ? 1 : (t <= t3) ? 2 : (t <= t4) ? 3 : 4; };
        const int p = piece(ta);
        ok = ok && p == piece(tb);
        double slope;
        __builtin_memcpy(&slope, &dr[r].tidx, sizeof slope);
        lc[r] = p == 1 ? slope : p == 3 ? -slope : 0.0;
        lt[r] = p == 1 ? t1 : p == 3 ? t3 : 0.0;
        la[r] = (p == 2 || p == 3) ? dr[r].A : 0.0;
      }
      lines = __ballot(!ok) == 0ull;
    }
  };

  // Value of record r at the present stage time (ts), 0 on lanes it does not feed: sine kinds from their
  // carried phase, the others from the waveform.
  auto rec_value = [&](auto ft_tag, int r, double ts, int stage) __attribute__((always_inline)) -> double {
    constexpr bool FT = decltype(ft_tag)::value;
    if constexpr (LINES) {
      if (lines) return sel[r] ? fma(lc[r], ts - lt[r], la[r]) : 0.0;
    }
    if constexpr (!OSC) {
      const double v = wave_value<double, FT, FM>(g.dmeta[r] & 0xff, dr[r], g, ts, i, stage, sps);
      return sel[r] ? v : 0.0;
    } else {
      const int ty = (FM & F_KSINE) ? (int)CMTJ_SINE : (g.dmeta[r] & 0xff);
      if (sine_kind(ty)) {
        const double v = dr[r].A * osc[r].s;
        if (ty == CMTJ_SINE) return v;
        return ty == CMTJ_POSINE ? fabs(v) : ((v <= 0) ? v : 0.0);
      }
      const double v = wave_value<double, FT, FM>(ty, dr[r], g, ts, i, stage, sps);
      return sel[r] ? v : 0.0;
    }
  };
  auto turn = [&]() __attribute__((always_inline)) {
    if constexpr (OSC) {
#pragma unroll
      for (int r = 0; r < NR; ++r)
        if (ND >= 0 || r < g.ndyn) osc[r].half();
    }
  };
  // The phases of step i: set at its block's first step, then turned.
  auto seek = [&]() __attribute__((always_inline)) {
    if constexpr (OSC) {
      const uint32_t i0 = i & ~(uint32_t)(CL_BLOCK - 1);
#pragma unroll
      for (int r = 0; r < NR; ++r) {
        if (ND >= 0 || r < g.ndyn) {
          if ((FM & F_KSINE) || sine_kind(g.dmeta[r] & 0xff)) {
            const double2 sc = osc_at(dr[r].p1, dr[r].p2, (double)i0 * dt);
            osc[r].s = sel[r] ? sc.x : 0.0;
            osc[r].c = sel[r] ? sc.y : 0.0;
          }
        }
      }
      for (uint32_t w = i0; w < i; ++w) {
        turn();
        turn();
      }
    }
  };

  // The end of a step: whether a NaN stops lanes (checked steps), the new m
  // and neighbours, the log entry.
  //
  // the lane's log value of a step, after it (calculateMagnetoresistance,
  // core/junction.hpp:1865-1867: layer 0 against layer 1, one layer against
  // the fixed reference vector, :1623-1629)
  auto lane_value = [&]() __attribute__((always_inline)) -> double {
    if constexpr (LOGF == 1) {
      const double rv = fma(-hR, rdot(m, nb[0]), Rp + hR);
      return rlane ? rv : m.a;
    } else {
      double v = m.a;
      if (classic) {
        double cosT;
        if (NN > 0 && nl > 1)
          cosT = rdot(m, nb[0]);
        else
          cosT = rdot(m, K.ref);
        const double rv = dpp_d<QP_BC0>(Rp + (((Rap - Rp) / 2.0) * (1.0 - cosT)));
        v = rlane ? rv : v;
      }
      return v;
    }
  };
  // DRV: the step's stage times may meet a time-dependent record; without it
  // the driver code is left out (kernels whose records are all step drivers
  // run the steps outside the records' windows that way: those records are
  // exactly 0 there).  LOGM: 0 tests per lane whether the step writes an
  // entry, 1 writes one, 2 writes none, 3 leaves its m and R entry in `lv`.  CHK: the step tests its new m for a
  // NaN and corrects a length outside the series' range exactly; without it
  // the step adds (|m|^2 - 1)^2 to dev, which the pass tests once per block of
  // steps (one instruction a step; a NaN stays a NaN in the sum).  `hitb` (wave-uniform)
  // keeps a checked step's NaN ballot: when it is not 0, only the lanes whose
  // run stops on it have taken the step (their m as the reference leaves
  // it); the others left their state alone and take the step again.
  unsigned long long hitb = 0ull;
  [[maybe_unused]] bool hitg = false;  // groups: a NaN in any wave of the group
  double dev = 0.0;
  uint64_t next_log = 0;   // LOGM 0: step of the next entry
  char* pk = lpl;          // the lane's next entry
  double lv = 0.0;
  auto step = [&](auto drv_tag, auto log_tag, auto chk_tag) __attribute__((always_inline)) {
    constexpr bool DRV = (decltype(drv_tag)::value & 1) != 0;
    constexpr bool DG = (decltype(drv_tag)::value & 2) != 0;
    constexpr int LOGM = decltype(log_tag)::value;
    constexpr bool CHK = decltype(chk_tag)::value;
    constexpr bool DRIVEN = DRV && (FM & (F_DYN | F_DYNH)) != 0;
    const double t = (double)i * dt;
    double mn;
    if constexpr (STK) {
      // pair couplings from the members' m at the start of the step
      // (storeMagnetisations, core/stack.hpp:65-76): d = m_top . p of the
      // member, p its bottom layer's m or the polarisation vector (members
      // have one or two layers: the bottom layer is the top layer's
      // neighbour, whose start-of-step m this lane holds)
      Rot<double> pv = s_pol;
      if constexpr (L > 1) {
        const bool two = sl.two_layer;
        pv = {two ? nb[0].a : s_pol.a, two ? nb[0].b : s_pol.b, two ? nb[0].c : s_pol.c};
      }
      double dq = rdot(m, pv);  // d in the top layer's quad
      if constexpr (L > 1) {
        // and in the member's other quads, by row shifts of 4 lanes
        const double below = dpp_d<DPP_ROW_SHR4>(dq), above = dpp_d<DPP_ROW_SHL4>(dq);
        dq = (ly == s_ti) ? dq : (ly == s_ti + 1) ? below : above;
      }
      if (s_kcl) {
        const double I0 = s_const ? sl.current.constant
                          : (sl.current.type == CMTJ_TABLE) ? g.tables[(size_t)sl.current.table_index + i]
                                                            : driver_value(sl.current, t);
        // sum over the members: every lane of a member's quads holds its term
        double S = s_w * dpp_d<QP_BC0>(dq);
        if (L == 1 && g.stack_pad >= 8) S += dpp_d<DPP_HALF_MIRROR>(S);
        if (g.stack_pad >= 16) S += dpp_d<DPP_MIRROR>(S);
        if (g.stack_pad >= 32) S = add_rows<16>(S);
        if (g.stack_pad >= 64) S = add_rows<32>(S);
        sI[0] = sI[1] = sI[2] = sIlog = fma(I0, S, I0);
        // C_j of the stack's log, where the step writes an entry
        if (LOGM == 1 || LOGM == 3 || (LOGM == 0 && (uint64_t)i == next_log)) {
          const bool last = s_j + 1 >= s_n;
          const double dn = __shfl(dq, s_base + (last ? s_j : s_j + 1) * LPI, 64);
          sClog = last ? 0.0 : sl.cj * (sl.series ? dq + dn : dq - dn);
        }
      } else {
        stack_current(sl, s_j, s_n, s_base, LPI, dq, t, dt, g.tables, i, sI, sIlog, sClog);
      }
    }
    [[maybe_unused]] const double gH = group_field_cl();
    // ---- drives at ts: this component's field slots and the layer's scalar
    // slots (the slot of a record is wave-uniform: one scalar branch)
    // With scalar drives, what of the field a stage's m does not change joins
    // d.H: constant field and couplings once per step (IEC, :654-675; IDMI,
    // :677-693; dipole tensors, :579-586, with this layer's Ms), and a record
    // of a field, IEC or IDMI slot by one FMA on its coefficient in this
    // lane's component, which the frozen neighbours fix for the step.
    auto base_field = [&](const Rot<double> (&nbs)[2]) __attribute__((always_inline)) -> double {
      double b = K.hb;
#pragma unroll
      for (int n = 0; n < NN; ++n) {
        if (CMTJ_HAS(F_IEC) || CMTJ_HAS(F_IEC2)) b = fma(nbs[n].a, K.jn[n], b);
        if (CMTJ_HAS(F_IDMI)) b = fma(K.Db[n], nbs[n].c, fma(-K.Dc[n], nbs[n].b, b));
        if (CMTJ_HAS(F_DIPOLE))
          b = fma(-K.dp[n][0], nbs[n].a, fma(-K.dp[n][1], nbs[n].b, fma(-K.dp[n][2], nbs[n].c, b)));
      }
      return b;
    };
    auto coef = [&](int slot, const Rot<double> (&nbs)[2]) __attribute__((always_inline)) -> double {
      if (slot < CMTJ_SLOT_K) return K.g;
      if constexpr (NN > 0) {
        const bool low = slot == CMTJ_SLOT_J_BOTTOM || slot >= CMTJ_SLOT_IDMI_BOTTOM;
        const bool second = NN > 1 && low;
        const double na = second ? nbs[1].a : nbs[0].a, n1 = second ? nbs[1].b : nbs[0].b,
                     n2 = second ? nbs[1].c : nbs[0].c;
        if (slot < CMTJ_SLOT_IDMI_TOP) return K.ginv_mst * na;
        const int k = slot - (low ? CMTJ_SLOT_IDMI_BOTTOM : CMTJ_SLOT_IDMI_TOP);
        return K.ginv_mst * (k == c1 ? -n2 : n1);  // -(e_k x n) of component c; lanes of component k are not fed
      } else {
        return 0.0;
      }
    };
    auto route = [&](CLDrive& d, int r, int meta, double x, double cf) __attribute__((always_inline)) {
      if constexpr (SLOTW) {
        d.kd = fma(wK[r], x, d.kd);
        d.I = fma(wI[r], x, d.I);
        d.FL = fma(wFL[r], x, d.FL);
        d.DL = fma(wDL[r], x, d.DL);
        if (t_driven) d.T += ((meta >> 8) & 0xff) == CMTJ_SLOT_TEMPERATURE ? x : 0.0;
        return;
      }
      const int slot = (meta >> 8) & 0xff;
      if (!DYNS || field_slot(slot)) {
        d.H = fma(cf, x, d.H);
        return;
      }
      if constexpr (DYNS) {
        switch (slot) {
          case CMTJ_SLOT_K: d.kd = fma(2.0 * K.ginv_ms, x, d.kd); break;
          case CMTJ_SLOT_K2: d.k2 = fma(4.0 * K.ginv_ms, x, d.k2); break;
          case CMTJ_SLOT_CURRENT: d.I += x; break;
          case CMTJ_SLOT_FL: d.FL += x; break;
          case CMTJ_SLOT_DL: d.DL += x; break;
          case CMTJ_SLOT_FL2: d.FL2 += x; break;
          case CMTJ_SLOT_DL2: d.DL2 += x; break;
          case CMTJ_SLOT_TEMPERATURE: d.T += x; break;
          case CMTJ_SLOT_J2_TOP: d.J2[0] = fma(2.0 * K.ginv_mst, x, d.J2[0]); break;
          default: d.J2[L == 2 ? 0 : 1] = fma(2.0 * K.ginv_mst, x, d.J2[L == 2 ? 0 : 1]); break;
        }
      }
    };
    // drives at ts on the field b, the neighbours being nbs
    auto drive = [&](auto ft_tag, double ts, int stage, double b,
                     const Rot<double> (&nbs)[2]) __attribute__((always_inline)) -> CLDrive {
      CLDrive d{b, 0.0, K.k2, K.bI, K.bFL, K.bDL, K.bT, K.bFL2, K.bDL2, {K.bJ2[0], K.bJ2[1]}};
      if constexpr (DRIVEN) {
        if (CMTJ_HAS(F_DYNH) || CMTJ_HAS(F_DYN)) {
          bool inwin = true;
          // step records are 0 outside [min t_start, max t_stop] (inclusive)
          if constexpr ((FM & F_KSTEP) != 0) inwin = ts >= win_lo && ts <= win_hi;
          if (inwin) {
#pragma unroll
            for (int r = 0; r < NR; ++r)
              if (ND >= 0 || r < g.ndyn)
                route(d, r, g.dmeta[r], rec_value(ft_tag, r, ts, stage),
                      DYNS ? coef((g.dmeta[r] >> 8) & 0xff, nbs) : K.g);
            for (int r = DREG; ND < 0 && !(FM & F_EXACT) && r < g.ndyn; ++r) {
              const DynRec rr = load_rec<FM>(g.dyn + (size_t)r * g.n + inst);
              constexpr bool FT = decltype(ft_tag)::value;
              const double v = wave_value<double, FT, FM>(g.dmeta[r] & 0xff, rr, g, ts, i, stage, sps);
              route(d, r, g.dmeta[r], feeds_lane(g.dmeta[r]) ? v : 0.0,
                    DYNS ? coef((g.dmeta[r] >> 8) & 0xff, nbs) : K.g);
            }
          }
        }
      }
      // a stack member's current is the stack's at every stage
      // (executeJunctionStep, core/stack.hpp:78-91)
      if constexpr (STK) d.I = K.stat_i ? ((stage == 0) ? sI[0] : (stage == 1) ? sI[1] : sI[2]) : 0.0;
      return d;
    };
    constexpr bool TERMS = DYNS || (FM & (F_IDMI | F_DIPOLE)) != 0;  // base_field in d.H
    auto start_field = [&](const Rot<double> (&nbs)[2]) __attribute__((always_inline)) -> double {
      double b = TERMS ? base_field(nbs) : K.hb;
      if constexpr (GW > 0) b += gH;
      return b;
    };
    // ---- what of the field a stage's m does not change, all components
    auto frozen = [&](const CLDrive& d, const Rot<double> (&nbs)[2]) __attribute__((always_inline)) -> Rot<double> {
      if constexpr ((SLOTW || (!DRIVEN && !TERMS)) && GW == 0) {
        // constant field and coupling: the neighbours' components are in the lane
        Rot<double> B{K.hb, K.hb1, K.hb2};
        if (CMTJ_HAS(F_IEC)) {
#pragma unroll
          for (int n = 0; n < NN; ++n)
            B = {fma(nbs[n].a, K.jn[n], B.a), fma(nbs[n].b, K.jn[n], B.b), fma(nbs[n].c, K.jn[n], B.c)};
        }
        return B;
      }
      double b = d.H;
      if constexpr (!TERMS) {
#pragma unroll
        for (int n = 0; n < NN; ++n)
          if (CMTJ_HAS(F_IEC)) b = fma(nbs[n].a, K.jn[n], b);
      }
      return rot3(b);
    };
    // ---- the field's matrix: the constant one, with the biquadratic
    // coupling's rank-one terms 2 J2 (nb . s) nb / (Ms t) of the frozen
    // neighbours
    auto matrix = [&](const CLDrive& d, const Rot<double> (&nbs)[2]) __attribute__((always_inline)) -> CLRows {
      CLRows A{K.A0, K.A1, K.A2};
      if (CMTJ_HAS(F_IEC2)) {
#pragma unroll
        for (int n = 0; n < NN; ++n) {
          const double w = d.J2[n];
          const Rot<double> v = nbs[n];
          const double wa = w * v.a, wb = w * v.b, wc = w * v.c;
          A.a = {fma(wa, v.a, A.a.a), fma(wa, v.b, A.a.b), fma(wa, v.c, A.a.c)};
          A.b = {fma(wb, v.a, A.b.a), fma(wb, v.b, A.b.b), fma(wb, v.c, A.b.c)};
          A.c = {fma(wc, v.a, A.c.a), fma(wc, v.b, A.c.b), fma(wc, v.c, A.c.c)};
        }
      }
      return A;
    };
    // ---- field at m = s (all three components; calculateHeffDipoleInjection,
    // core/junction.hpp:590-622), scaled by K.g
    auto field = [&](const Rot<double>& s, const CLDrive& d, const Rot<double>& B,
                     const CLRows& A) __attribute__((always_inline)) -> Rot<double> {
      auto along = [&](const Rot<double>& r, double x) {
        return fma(r.c, s.c, fma(r.b, s.b, fma(r.a, s.a, x)));
      };
      Rot<double> h;
      if constexpr (DG)
        h = {fma(A.a.a, s.a, B.a), GAUGE ? B.b : fma(A.b.b, s.b, B.b), fma(A.c.c, s.c, B.c)};
      else if constexpr (GAUGE && !(FM & F_IEC2))
        h = {along(A.a, B.a), fma(A.b.c, s.c, fma(A.b.a, s.a, B.b)), along(A.c, B.c)};
      else
        h = {along(A.a, B.a), along(A.b, B.b), along(A.c, B.c)};
      if constexpr ((FM & (F_DYN | F_ANIS2)) != 0) {
        if (CMTJ_HAS(F_ANIS2) || k_driven) {
          // calculateSecondOrderAnisotropy (:645-652): 4 K2 (anis . m)^3 / Ms,
          // and what drives add to the first order
          const double u = fma(K.an2, s.c, fma(K.an1, s.b, K.an0 * s.a));  // anis . m
          const double w = fma(d.k2, u * u, d.kd) * u;
          h = {fma(K.an0, w, h.a), fma(K.an1, w, h.b), fma(K.an2, w, h.c)};
        }
      }
      return h;
    };
    // ---- the spin torques of a stage time (:743-812): a p + b m x p over the
    // polarisers p, with a, b and p fixed for the stage, joins the field as
    // a p and the damping's alpha h as (b - alpha a) p, so that a torque costs
    // what it costs without them and one more (before: eight more; a step of a
    // spin-torque oscillator 161 -> 128 VALU instructions)
    auto polariser = [&](const Rot<double> (&nbs)[2]) __attribute__((always_inline)) -> Rot<double> {
      // the layer's reference vector: fixed, or the start-of-step top /
      // bottom neighbour
      Rot<double> p = K.pol;
      if (nb_pol) {
#pragma unroll
        for (int n = 0; n < NN; ++n)
          p = {fma(K.wp[n], nbs[n].a, p.a), fma(K.wp[n], nbs[n].b, p.b), fma(K.wp[n], nbs[n].c, p.c)};
      }
      return p;
    };
    const bool spin_on = CMTJ_HAS(F_STT) || CMTJ_HAS(F_SOT);
    auto spin = [&](const CLDrive& d, const Rot<double> (&nbs)[2], const Rot<double>& B) __attribute__((always_inline)) -> CLSpin {
      CLSpin r{B, {0.0, 0.0, 0.0}};
      if constexpr (SPC) {
        r.Q = Q0;
#pragma unroll
        for (int n = 0; n < NN; ++n) {
          r.B = {fma(swa[n], nbs[n].a, r.B.a), fma(swa[n], nbs[n].b, r.B.b), fma(swa[n], nbs[n].c, r.B.c)};
          r.Q = {fma(swb[n], nbs[n].a, r.Q.a), fma(swb[n], nbs[n].b, r.Q.b), fma(swb[n], nbs[n].c, r.Q.c)};
        }
      } else if constexpr ((FM & (F_STT | F_SOT)) != 0) {
        if (spin_on) {
          const Rot<double> p = polariser(nbs);
          double a = 0.0, b = 0.0;
          if (CMTJ_HAS(F_STT)) {
            // Slonczewski STT (:743-769) where eta is constant (else torque()
            // adds it)
            const double w = den_const ? d.I * K.wc : 0.0;
            a = K.sta * w;
            b = K.stb * w;
          }
          if (CMTJ_HAS(F_SOT)) {
            // SOT (:770-812): coefficients from the drivers, or static ones
            // scaling the current
            const double Hdl = fma(K.dlt, d.I, d.DL), Hfl = fma(K.flt, d.I, d.FL);
            a = fma(K.ga, Hfl, fma(-K.gaa, Hdl, a));
            b = fma(K.ga, Hdl, fma(K.gaa, Hfl, b));
          }
          const double w = fma(-K.alpha, a, b);
          r.B = {fma(a, p.a, B.a), fma(a, p.b, B.b), fma(a, p.c, B.c)};
          r.Q = {w * p.a, w * p.b, w * p.c};
          if (CMTJ_HAS(F_SOT2)) {
            // the secondary reference (dynamic SOT drivers only)
            const double a2 = fma(K.g2, d.FL2, -K.g2a * d.DL2), b2 = fma(K.g2, d.DL2, K.g2a * d.FL2);
            const double w2 = fma(-K.alpha, a2, b2);
            const Rot<double> p2 = K.ref2;
            r.B = {fma(a2, p2.a, r.B.a), fma(a2, p2.b, r.B.b), fma(a2, p2.c, r.B.c)};
            r.Q = {fma(w2, p2.a, r.Q.a), fma(w2, p2.b, r.Q.b), fma(w2, p2.c, r.Q.c)};
          }
        }
      }
      return r;
    };
    // ---- dm of a step at m = s (solveLLG, :716-815): m x (h + m x (alpha h)),
    // the spin torques in both.  As cross products throughout: the initial m
    // of a run need not have unit length.
    auto torque = [&](const Rot<double>& s, const CLDrive& d, const CLSpin& sp, const CLRows& A,
                      const Rot<double> (&nbs)[2]) __attribute__((always_inline)) -> double {
      Rot<double> h = field(s, d, sp.B, A);
      if constexpr ((FM & (F_STT | F_SOT)) != 0) {
        if (spin_on) {
          Rot<double> v{fma(K.alpha, h.a, sp.Q.a), fma(K.alpha, h.b, sp.Q.b), fma(K.alpha, h.c, sp.Q.c)};
          if (CMTJ_HAS(F_STT) && __builtin_expect(!den_const, 0)) {
            const Rot<double> p = polariser(nbs);
            const double mp = rdot(s, p);
            const double den = K.alt ? fma(K.lam, mp, 1.0) : fma(K.lam2 - 1.0, mp, K.lam2 + 1.0);
            const double w = d.I * (K.num / den);
            const double a = K.stt ? K.sta * w : 0.0, b = K.stt ? K.stb * w : 0.0;
            h = {fma(a, p.a, h.a), fma(a, p.b, h.b), fma(a, p.c, h.c)};
            v = {fma(b, p.a, v.a), fma(b, p.b, v.b), fma(b, p.c, v.c)};
          }
          return cross_a(s, fma(s.c, v.a, fma(-s.a, v.c, h.b)), fma(s.a, v.b, fma(-s.b, v.a, h.c)));
        }
      }
      return cross_a(s, fma(K.alpha, cross_b(s, h), h.b), fma(K.alpha, cross_c2(s, h), h.c));
    };
    constexpr std::integral_constant<bool, !F64> FTT{};  // binary32 path: single-precision transcendentals
    const double b0 = start_field(nb);
    const CLDrive d0 = drive(FTT, t, 0, b0, nb);
    const Rot<double> B0 = frozen(d0, nb);
    const CLRows M0 = matrix(d0, nb);
    const CLSpin S0 = spin(d0, nb, B0);
    if constexpr (F64 && SOLVER == CMTJ_RK4) {
      // rk4_step (core/junction.hpp:1017-1041) in binary64
      const double k1 = torque(m, d0, S0, M0, nb);
      CLDrive d1 = d0;
      Rot<double> B1 = B0;
      CLRows M1 = M0;
      CLSpin S1 = S0;
      auto stage_drives = [&](double ts, int stage) __attribute__((always_inline)) {
        if constexpr (DRIVEN || STK) {
          // (a KCL stack's current is the same at every stage time)
          if (STK && !DRIVEN && s_kcl) return;
          turn();
          d1 = drive(FTT, ts, stage, b0, nb);
          if (DRIVEN && (!DYNS || h_driven)) B1 = frozen(d1, nb);
          if (DYNS && j2_driven) M1 = matrix(d1, nb);
          S1 = spin(d1, nb, B1);
        }
      };
      stage_drives(t + 0.5 * dt, 1);
      const double k2 = torque(rot3(fma(0.5, k1, m.a)), d1, S1, M1, nb);
      const double k3 = torque(rot3(fma(0.5, k2, m.a)), d1, S1, M1, nb);
      stage_drives(t + dt, 2);
      const double k4 = torque(rot3(m.a + k3), d1, S1, M1, nb);
      mn = fma(fma(2.0, k2 + k3, k1 + k4), 1.0 / 6.0, m.a);
    } else if constexpr (F64) {
      // stochasticTorque (core/junction.hpp:824-831) with the layer's three
      // normals of the shared Philox stream: -gamma/(1 + a^2) m x (dW + a m x dW)
      // dW scaled by -gamma/(1 + a^2) and sqrt(dt), so this is the kick itself
      auto noise = [&](const Rot<double>& s, const Rot<double>& dW) __attribute__((always_inline)) -> double {
        return cross_a(s, fma(K.alpha, cross_b(s, dW), dW.b), fma(K.alpha, cross_c2(s, dW), dW.c));
      };
      const double f0 = torque(m, d0, S0, M0, nb);
      Rot<double> dW{0.0, 0.0, 0.0};
      double g0 = 0.0;
      if (CMTJ_HAS(F_THERMAL)) {
        const Rot<double> n = next_normals();
        double sg = K.sg0;
        if (t_driven) {
          double T = d0.T;
          asm volatile("" : "+v"(T));  // (a root taken only here: the compiler would take it at every step)
          sg = K.therm ? sqrt(K.sig2 * T) * K.kick : 0.0;
        }
        dW = {n.a * sg, n.b * sg, n.c * sg};
        g0 = noise(m, dW);
      }
      if constexpr (SOLVER == CMTJ_HEUN) {
        // heunSolverStep (core/junction.hpp:1756-1815): a predictor m + f dt
        // + g sqrt(dt), whose neighbours feed the corrector's second
        // evaluation at t + dt; the same dW in both
        const Rot<double> mN = rot3(m.a + f0 + g0);
        Rot<double> nN[2] = {nb[0], nb[1]};
        neighbours(nN, mN.a);
        turn();
        turn();
        const CLDrive d1 = drive(FTT, t + dt, 1, start_field(nN), nN);
        const double f1 = torque(mN, d1, spin(d1, nN, frozen(d1, nN)), matrix(d1, nN), nN);
        mn = m.a + (f0 + f1) * 0.5;
        if (CMTJ_HAS(F_THERMAL)) mn = fma(0.5, g0 + noise(mN, dW), mn);
      } else {
        // eulerHeunSolverStep (core/junction.hpp:1709-1754): drift at t, the
        // stochastic torque at m and at m + g sqrt(dt), one dW per step
        mn = m.a + f0;
        if (CMTJ_HAS(F_THERMAL)) mn = fma(0.5, g0 + noise(rot3(m.a + g0), dW), mn);
        turn();
        turn();
      }
    } else {
      // ---- anchor: dm/dt at (m, t) in binary64
      const Rot<double> h = field(m, d0, B0, M0);
      const double gb = fma(K.alpha, cross_b(m, h), h.b), gc = fma(K.alpha, cross_c2(m, h), h.c);
      const double k1 = cross_a(m, gb, gc);
      // ---- stages 2-4: binary32 increments about the anchor
      float dmid = 0.f, dend = 0.f;
      if constexpr (DRIVEN) {
        // drive increments against the start of the step
        const double u = PLAIN32 ? ig : 1.0;
        turn();
        dmid = (float)((drive(FTT, t + 0.5 * dt, 1, b0, nb).H - d0.H) * u);
        turn();
        dend = (float)((drive(FTT, t + dt, 2, b0, nb).H - d0.H) * u);
      }
      if constexpr (PLAIN32) {
        // unscaled, cross products expanded about the anchor: (m0 + d) x (H0 +
        // dH) - m0 x H0 = (m0 + d) x dH + d x H0, and the same for m x (m x H)
        const float m1 = (float)m.b, m2 = (float)m.c, H1 = (float)(h.b * ig), H2 = (float)(h.c * ig),
                    P1 = (float)(cross_b(m, h) * ig), P2 = (float)(cross_c2(m, h) * ig);
        auto cross32 = [&](float a1, float a2, float b) {
          return a1 * dpp_f<QP_ROT2>(b) - a2 * dpp_f<QP_ROT1>(b);
        };
        auto delta = [&](float d, float dd) __attribute__((always_inline)) -> float {
          const float d1 = dpp_f<QP_ROT1>(d), d2 = dpp_f<QP_ROT2>(d), s1 = m1 + d1, s2 = m2 + d2;
          float dH = fmaf(-p_nms, d, dd);
          if (CMTJ_HAS(F_ANIS)) dH = fmaf(p_ak, fmaf(p_an2, d2, fmaf(p_an1, d1, p_an * d)), dH);
          const float dP = cross32(s1, s2, dH) + fmaf(d1, H2, -d2 * H1);
          const float dQ = cross32(s1, s2, dP) + fmaf(d1, P2, -d2 * P1);
          return fmaf(dQ, p_al, dP) * p_g;
        };
        const float d2 = (float)(k1 * 0.5);
        float dk = delta(d2, dmid), acc = dk * 2.f;
        dk = delta(d2 + dk * 0.5f, dmid);
        acc = acc + dk * 2.f;
        acc = acc + delta((float)k1 + dk, dend);
        mn = m.a + k1 + (double)(acc * (float)(1.0 / 6.0));
      } else {
        const StageConst KF{(float)K.A0.a, (float)K.A0.b, (float)K.A0.c, (float)K.alpha};
        mn = m.a + fma((double)stage_increments<DG>(KF, (float)k1, m, h, gb, gc, dmid, dend), 1.0 / 6.0, k1);
      }
    }
    // ---- CVector::normalize (core/cvector.hpp:185-192).  Binary64: |m|^2 - 1
    // as a butterfly over the quad, (x^2 + y^2) + (z^2 - 1) in all its lanes,
    // which so scale by the same factor: every lane's copy of a component
    // equals its owner's.  Binary32 increments: each lane adds the squares it
    // holds in its own order (two instructions fewer, 46.7 -> 44.7 ms for the
    // 200,000 steps of the PIMM sweep), which may differ in the last bit
    // between lanes, a direction error of 1e-16 a step beside the increments'
    // 1e-9; the other components are then read from their owners.
    Rot<double> mnew = rot3(mn);
    double e;
    if constexpr (F64) {
      e = fma(mn, mn, unit);
      e = e + dpp_d<QP_SWAP1>(e);
      e = e + dpp_d<QP_SWAP2>(e);
    } else {
      e = fma(mnew.c, mnew.c, fma(mnew.b, mnew.b, fma(mn, mn, unit)));
    }
    if constexpr (SOLVER == CMTJ_RK4) {
      // (1 + e)^(-1/2) - 1 = -e/2 + 3/8 e^2 - 5/16 e^3 + 35/128 e^4
      const double p = e * fma(e, fma(e, fma(e, len4, len3), len2), -0.5);
      const Rot<double> ms = F64 ? Rot<double>{fma(mn, p, mn), fma(mnew.b, p, mnew.b), fma(mnew.c, p, mnew.c)}
                                 : rot3(fma(mn, p, mn));
      if constexpr (CHK) {
        const double ss = lact ? e + 1.0 : 0.0;
        const double len = (ss != 0.0) ? sqrt(ss) : 1.0;  // a zero vector stays
        const bool near = fabs(e) <= kUnitRange;
        if constexpr (F64)
          mnew = {near ? ms.a : mn / len, near ? ms.b : mnew.b / len, near ? ms.c : mnew.c / len};
        else
          mnew = rot3(near ? ms.a : mn / len);
      } else {
        dev = fma(e, e, dev);
        mnew = ms;
      }
    } else {
      // a stochastic step's length is off by the square of its kick: the
      // series within its range, the root and division beyond
      const double p = e * fma(e, fma(e, fma(e, len4, len3), len2), -0.5);
      mnew = {fma(mn, p, mn), fma(mnew.b, p, mnew.b), fma(mnew.c, p, mnew.c)};
      const bool near = fabs(e) <= kUnitRange;
      if (__builtin_expect(__ballot(!near) != 0ull, 0)) {
        const double ss = lact ? e + 1.0 : 0.0;
        const Rot<double> ex = rot3((ss != 0.0) ? mn / sqrt(ss) : mn);
        mnew = {near ? mnew.a : ex.a, near ? mnew.b : ex.b, near ? mnew.c : ex.c};
      }
    }
    // the reference updates layers in turn and stops at the first NaN
    // layer; layers up to and including it take the new value (RK4 only:
    // the Euler-Heun step of the reference has no such test)
    if constexpr (CHK) {
      const unsigned long long bad = __ballot(isnan(mnew.a)) & nan_lanes;
      hitb = bad;
      if constexpr (GW > 0) hitg = group_any(bad != 0ull);
      if (__builtin_expect((GW > 0) ? hitg : bad != 0ull, 0)) {
        // a NaN in the wave (rare): layers up to and including the instance's
        // first NaN layer take the new value; a member's NaN ends its stack's
        // or group's run (the reference throws), the other members take this
        // step and stop with it (selects, no per-lane branch: the whole test stays
        // wave-uniform)
        const uint32_t gb = (uint32_t)((bad >> gshift) & ((1ull << LPI) - 1));
        bool take = (gb != 0u) & (ly <= (int)(__builtin_ctz(gb | 0x80000000u) >> 2));
        if constexpr (STK) take = take | ((gb == 0u) & ((bad & s_mask) != 0ull));
        if constexpr (GW > 0) take = take | (gb == 0u);
        m.a = take ? mnew.a : m.a;
        return;
      }
    }
    // a step that goes on: new m, neighbours, log entry
    m = mnew;
    if (nb_step) neighbours(nb, m.a);
    if constexpr (LOGM == 3) {
      if (!nb_step) neighbours(nb, m.a);
      lv = lane_value();
    } else if (LOGM == 1 || (LOGM == 0 && (uint64_t)i == next_log)) {
      if (!nb_step) neighbours(nb, m.a);
      const double v = lane_value();
      if (wlog) log_put(f32log, pk, v);
      if (LOGF != 1 && strip) {
        // stripMagnetoResistance (:1835-1857), parallel sum of the layers
        double rx = 0.0, ry = 0.0;
        if (lact && c == 0) {
          const double Rx = sRx0 + sAMRX * (m.a * m.a) + sSMRX * (m.b * m.b);
          const double Ry = sRy0 + sAHE2 * m.c + sXY * m.a * m.b;
          rx = 1. / Rx;
          ry = 1. / Ry;
        }
#pragma unroll
        for (int o = 4; o < LPI; o <<= 1) {
          rx += __shfl_xor(rx, o, 64);
          ry += __shfl_xor(ry, o, 64);
        }
        if (own && q == 0) {
          log_put(f32log, pk - om + orr, 1 / rx);
          log_put(f32log, pk - om + orr + cs, 1 / ry);
        }
      }
      if constexpr (STK) {
        if (logging && own && q == 0) {  // the member's stack channels follow its junction channels
          const uint64_t nch = (uint64_t)log_channels(nl, g.mr_mode, g.log_mask);
          log_put(f32log, pk - om + nch * cs, sIlog);
          log_put(f32log, pk - om + (nch + 1) * cs, sClog);
        }
      }
      pk += esize;
      if constexpr (LOGM == 0) {
        ++k;
        next_log += W;
      }
    }
  };
  bool stopped = false;
  // Steps of one phase (the lane's steps below lim) in wave-uniform passes:
  // each pass runs the fewest steps any lane of the wave still has in the
  // phase on a scalar counter, so the loop needs no per-lane exit test;
  // lanes done with the phase sit out the passes that follow.  A NaN in any
  // lane ends the pass at that step, which no lane counts: the lanes of
  // the instances (stacks) it stops end their run there (steps done = i),
  // the others take the step again in the next pass (the same inputs: the
  // same result).
  //
  // A pass whose lanes all log with the same cadence, in step, finds the
  // logged steps on a scalar countdown.
  auto phase = [&](uint32_t lim, auto drv_tag) __attribute__((always_inline)) {
    using I0 = std::integral_constant<int, 0>;
    using I1 = std::integral_constant<int, 1>;
    using I2 = std::integral_constant<int, 2>;
    using I3 = std::integral_constant<int, 3>;
    for (;;) {
      const uint32_t n = (!stopped && i < lim) ? lim - i : 0u;
      const uint32_t seg = wave_min_nonzero(n);
      if (seg == 0u) break;
      if (n != 0u) {
        const uint32_t i0 = i;
        uint32_t end = seg;  // wave-uniform
        seek();
        pk = lpl + (uint64_t)k * esize;
        next_log = (uint64_t)k * W;
        // steps to the next entry, where every lane of the pass agrees on it
        // and on the cadence
        const uint32_t W0 = __builtin_amdgcn_readfirstlane(W);
        uint32_t cd = __builtin_amdgcn_readfirstlane((uint32_t)(next_log - i));
        const bool uni = __ballot(W != W0 || (uint32_t)(next_log - i) != cd || next_log < i) == 0ull;
        uint32_t slow = 0;  // blocks to run checked
        bool flagged = false;
        for (uint32_t u0 = 0; u0 < end;) {
          uint32_t ue = min(u0 + (uint32_t)CL_BLOCK, end);
          if constexpr (OSC) {
            // a block ends where a lane's phases are set again
            const uint32_t a = (i0 + u0) & (CL_BLOCK - 1), a0 = __builtin_amdgcn_readfirstlane(a);
            if (__ballot(a != a0) == 0ull)
              ue = min(u0 + (CL_BLOCK - a0), end);
            else
              ue = min(u0 + wave_min_nonzero(CL_BLOCK - a), end);
            i = i0 + u0;
            if (u0 != 0u && a == 0u) seek();
          }
          if constexpr (SOLVER != CMTJ_RK4) {
            set_lines(i0 + u0, i0 + ue - 1u);
            for (uint32_t u = u0; u < ue;) {
              draw(i0 + u);
              const uint32_t un = min(u + 4u, ue);
#pragma nounroll
              for (; u < un; ++u) {
                i = i0 + u;
                step(drv_tag, I0{}, std::false_type{});
              }
            }
          } else {
            // steps without a per-step NaN test; a block that meets a NaN or
            // a length outside the series' range is taken again from its
            // start, step by step with the test, up to the NaN step (the same
            // inputs: the same values; log entries a stopping instance wrote
            // past that step lie beyond its entries_done).  Where one block
            // after another needs that, the next ones are run checked at once.
            const double m_b = m.a;
            const uint32_t k_b = k, cd_b = cd;
            bool redo = slow != 0u;
            if (!redo) {
              dev = 0.0;
              if (!uni) {
                for (uint32_t u = u0; u < ue; ++u) {
                  i = i0 + u;
                  step(drv_tag, I0{}, std::false_type{});
                }
              } else if (W0 == 1u && cd == 0u && !strip && !STK) {
                // every step an entry: two steps to a store (half the
                // loop's branches and changes of the execution mask)
                uint32_t u = u0;
                for (; u + 1u < ue; u += 2u) {
                  i = i0 + u;
                  step(drv_tag, I3{}, std::false_type{});
                  const double v = lv;
                  i = i0 + u + 1u;
                  step(drv_tag, I3{}, std::false_type{});
                  if (wlog) {
                    if (f32log) {
                      struct __attribute__((packed, aligned(4))) F2 { float a, b; };
                      *(F2*)pk = F2{(float)v, (float)lv};
                    } else {
                      struct __attribute__((packed, aligned(8))) D2 { double a, b; };
                      *(D2*)pk = D2{v, lv};
                    }
                  }
                  pk += 2u * esize;
                }
                if (u < ue) {
                  i = i0 + u;
                  step(drv_tag, I1{}, std::false_type{});
                }
                k += ue - u0;
              } else {
                uint32_t ne = 0;
                for (uint32_t u = u0; u < ue;) {
                  const uint32_t us = min(ue - u, cd);  // steps without an entry
                  const uint32_t un = u + us;
                  for (; u + 1u < un; u += 2u) {
                    i = i0 + u;
                    step(drv_tag, I2{}, std::false_type{});
                    i = i0 + u + 1u;
                    step(drv_tag, I2{}, std::false_type{});
                  }
                  if (u < un) {
                    i = i0 + u;
                    step(drv_tag, I2{}, std::false_type{});
                    ++u;
                  }
                  cd -= us;
                  if (u < ue) {
                    i = i0 + u;
                    step(drv_tag, I1{}, std::false_type{});
                    ++u;
                    ++ne;
                    cd = W0 - 1u;
                  }
                }
                k += ne;
              }
              redo = __ballot(!(dev <= kUnitRange * kUnitRange)) != 0ull;
              if constexpr (GW > 0) redo = group_any(redo);
              slow = (redo && flagged) ? 31u : 0u;
              flagged = redo;
              if (redo) {
                m = rot3(m_b);
                neighbours(nb, m.a);
              }
            } else {
              --slow;
            }
            if (__builtin_expect(redo, 0)) {
              k = k_b;
              pk = lpl + (uint64_t)k * esize;
              next_log = (uint64_t)k * W;
              i = i0 + u0;
              seek();
              for (uint32_t u = u0; u < ue; ++u) {
                i = i0 + u;
                step(drv_tag, I0{}, std::true_type{});
                if ((GW > 0) ? hitg : hitb != 0ull) {
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
        if ((GW > 0) ? hitg : hitb != 0ull) {
          const uint32_t gb = (uint32_t)((hitb >> gshift) & ((1ull << LPI) - 1));
          bool stop = gb != 0u;
          if constexpr (STK) stop = stop || (hitb & s_mask) != 0ull;
          if constexpr (GW > 0) stop = true;
          if (gb) {
            nan_layer = __builtin_ctz(gb) >> 2;
            code = CMTJ_ERR_NAN;
          }
          // every lane whose NaN is in the ballot belongs to an instance
          // that stops here, so the pass makes progress; were none to stop,
          // the lanes would take the same step again for ever: end their
          // runs with the error instead
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
  auto run = [&](auto dg_tag) __attribute__((always_inline)) {
  constexpr int DG2 = decltype(dg_tag)::value ? 2 : 0;
  constexpr std::integral_constant<int, DG2> OFF{};
  constexpr std::integral_constant<int, DG2 + 1> ON{};
  if constexpr ((FM & F_KSTEP) != 0 && !(FM & F_TABLE)) {
    // steps [ia, ib) may meet a record's window [win_lo, win_hi]; every
    // stage time of a step before ia is below win_lo, of a step from ib on
    // above win_hi (one step of margin on each side)
    uint32_t ia = iend, ib = iend;
    if (win_lo <= win_hi) {
      const double a = floor(win_lo / dt) - 2.0, b = floor(win_hi / dt) + 2.0;
      ia = a <= (double)i ? i : (a >= (double)iend ? iend : (uint32_t)a);
      ib = b <= (double)ia ? ia : (b >= (double)iend ? iend : (uint32_t)b);
    }
    phase(ia, OFF);
    phase(ib, ON);
    phase(iend, OFF);
  } else {
    phase(iend, ON);
  }
  };
  if constexpr (DGSET) {
    if (diag)
      run(std::true_type{});
    else
      run(std::false_type{});
  } else {
    run(std::false_type{});
  }
  if (g.mag_out && live) g.mag_out[((size_t)jid * CMTJ_MAX_LAYERS + ly) * 3 + c] = m.a;
  if (g.status && own && q == 0) {
    cmtj_status s;
    s.code = code;
    s.steps_done = i;
    s.entries_done = k;
    s.nan_layer = nan_layer;
    g.status[jid] = s;
  }
  if (S) {
    if (live) S->m[ly][c] = m.a;
    if (own && q == 0) {
      S->step = i;
      S->entries = k;
      S->code = code;
      S->nan_layer = nan_layer;
    }
  }
}

}  // namespace cmtj
