// Net production rates for mechanisms whose one-lane-per-state program needs more than the registers of two waves per
// SIMD (hand-written frame; the host prepends the sizes and fills in one straight-line section of reactions per part).
//
// A team of PARTS waves owns 64 states, one lane per state in every wave, and shares in LDS what the reactions read:
// per species C_k, F_k = S E+_k C_k and E-_k / S (E+ = min(c+, e^g), E- = min(c-, 1/e^g), g = G°_k/RT), rows of 64
// states each. The power of two S keeps F of a trace species (C down to 1e-300) out of the subnormal numbers; it
// leaves a reaction's product of F and E- as S^Σν, which the factor (P0/RT)^(-Σν) takes back.
//   1. species k = p, p + PARTS, ..: amounts n_k = Y_k/W_k, Σn and Σ max(0, n) over the team (reaction.rs:362-373 on a
//      mass basis), C_k, and the NASA-7 piece's g_k (reaction.rs:78-110, 236-268)
//   2. part p's reactions (a wave-uniform branch): k_f, q = k_f (Π C^ν' - Π F Π E- (P0/RT)^(-Σν)), ω_k += ν_k q into
//      register sums (reaction.rs:113-327); a species on both sides multiplies both products by its concentration once
//   3. the parts' sums, in a fixed order: the upper half of the parts hands its sums to the lower half through LDS,
//      then every part adds the rows of its own species and writes them out
//
// Bound: FP64 VALU issue. Per 64 states of the 53-species mechanism it issues 17.5 k VALU instructions where the
// one-lane kernel issued 23.4 k (no accumulation-register moves, exponentials without clamps of their own and with
// a reduction of one rounding, one exponential per rate constant, one factor per product species) at one wave per
// SIMD; with two waves per SIMD and the parts' scalar constants and LDS reads beside the other wave's arithmetic, 2^20
// states take 0.86 ms against 1.18 ms (30 launches each on one card; 0.92 in the full benchmark run), and a single
// wavefront's worth of states 25 against 75 us (a quarter of the reactions per wave). What is left of it: two thirds of a
// block's cycles are the reactions (half of them issue), an eighth the Gibbs exponentials, a tenth its loads and a
// fourteenth the sums. Measured and not kept: six parts at three waves per SIMD (4 to 19 % longer: 168 registers spill),
// persistent blocks with the teams on barriers of their own (2 to 12 % longer: the loop's invariants spill), rows of
// independent instructions pinned by scheduling barriers (no gain, compile times of minutes).
// Rounding: 3.6e-15 of the state's largest rate on average (4096 states, against the program in 80-bit arithmetic), 4.7e-15
// for the one-lane kernel and 4.0e-15 with the library's functions.
// Required defines: NAME, K, KA (active species), PARTS (waves per team, even), TEAMS (teams per block), FAST (1: exp
// and ln on the FP32 cores; 0: FP64 polynomials).
// Tables: rcp_W[K], gibbs[KA][15] = the split temperature and the two 7-coefficient pieces of g (low first), in the
// basis 1, ln T, T, T², T³, T⁴, 1/T.

typedef const double __attribute__((address_space(4))) * table;  // read by scalar loads at wave-uniform indices

#define RGAS (1.380649e-23 * 6.02214076e23)
#define P0_R (101325.0 / RGAS)
#define FLT_MIN_D 1.1754943508222875e-38
#define FLT_MAX_D 3.4028234663852886e38
#define LN_FLT_MAX 0x1.62e42fefa39efp+6
#define SCALE 0x1p+100
#define COLS (64 * TEAMS)
#define KP ((K + PARTS - 1) / PARTS)
// Rows of part p's sums, over those of F and E- (and, with one team of eight parts, of C)
#define SUMS(p) (lds_v + (p) * KA * COLS + col)

// 1/b: v_rcp_f64 (relative error below 2^-24) and one Newton step (2.2e-15)
__device__ __forceinline__ double rcp64(double b) {
  double r = __builtin_amdgcn_rcp(b);
  { const double e = __builtin_fma(-b, r, 1.0);
    r = __builtin_fma(r, e, r); }
  return r;
}

// Several independent evaluations side by side.
#define ROW _Pragma("unroll") for (int i = 0; i < N; i++)
template <int N>
__device__ __forceinline__ void rcp64_rows(double* x) {
  double r[N], e[N];
  ROW r[i] = __builtin_amdgcn_rcp(x[i]);
  ROW e[i] = __builtin_fma(-x[i], r[i], 1.0);
  ROW x[i] = __builtin_fma(r[i], e[i], r[i]);
}

// exp64_rows: e^x. log_rows and pow_rows: the logarithm to a base of the kernel's own (FAST: e, else 2) and its inverse.
// log64: ln x.
#if FAST
// With FP32 cores: 2^n 2^f with the FP64 reduction x log2 e = n + f and v_exp_f32; the FP64 exponent and mantissa split and
// v_log_f32
template <int N>
__device__ __forceinline__ void exp64_rows(double* x) {
  double y[N], n[N];
  float f[N];
  ROW y[i] = x[i] * 1.4426950408889634;
  ROW n[i] = __builtin_rint(y[i]);
  ROW n[i] = __builtin_fmax(n[i], -1100.0);
  ROW n[i] = __builtin_fmin(n[i], 1100.0);
  ROW f[i] = (float)(y[i] - n[i]);
  ROW f[i] = __builtin_amdgcn_exp2f(f[i]);
  ROW x[i] = __builtin_ldexp((double)f[i], (int)n[i]);
}
template <int N>
__device__ __forceinline__ void pow_rows(double* x) {
  exp64_rows<N>(x);
}
template <int N>
__device__ __forceinline__ void log_rows(double* x) {
  ROW {
    const long long b = __double_as_longlong(x[i]);
    const int e = (int)((b >> 52) & 0x7FF) - 1023;
    const double m = __longlong_as_double((b & 0x000FFFFFFFFFFFFFLL) | 0x3FF0000000000000LL);
    x[i] = ((double)e + (double)__builtin_amdgcn_logf((float)m)) * 0.6931471805599453;
  }
}
__device__ __forceinline__ double log64(double x) {
  log_rows<1>(&x);
  return x;
}
#else
// 2^(t + r) with t an integer plus 1.5·2^52, of which the low word is read, and |r| <= 1/2: the Chebyshev interpolant of 2^r
// of degree 10 (exp_coefficients.py; relative error below 5e-16) and v_ldexp_f64, which gives 0 and +inf outside the FP64
// range
template <int N>
__device__ __forceinline__ void pow2_rows(double* y, const double* t, const double* r) {
  double p[N];
  ROW p[i] = __builtin_fma(0x1.e6063f7217bc6p-28, r[i], 0x1.b675bca4eeebbp-24);
  const double c[9] = {0x1.62bfd47773353p-20, 0x1.ffcb54062e698p-17, 0x1.430913096fd9fp-13, 0x1.5d87fe9d7a584p-10, 0x1.3b2ab6fba1ddap-7,
                       0x1.c6b08d703ce49p-5,  0x1.ebfbdff82c598p-3,  0x1.62e42fefa3a19p-1,  1.0};
#pragma unroll
  for (int j = 0; j < 9; j++) {
    ROW p[i] = __builtin_fma(p[i], r[i], c[j]);
  }
  ROW y[i] = __builtin_ldexp(p[i], (int)(unsigned)__double_as_longlong(t[i]));
}
// For |y| < 2^31: n = rint(y), r = y - n exactly: 14 instructions.
template <int N>
__device__ __forceinline__ void pow_rows(double* y) {
  double t[N], r[N];
  ROW t[i] = y[i] + 0x1.8p+52;
  ROW r[i] = t[i] - 0x1.8p+52;
  ROW r[i] = y[i] - r[i];
  pow2_rows<N>(y, t, r);
}
// For |x| < 2^30: n = rint(x log2 e), r = x log2 e - n in one rounding: 14 instructions too. The FP64 log2 e is off by 1.4e-17
// of itself, an eighth of the rounding that x comes with; scaling the exponents' coefficients by it beforehand costs a
// rounding of every coefficient (mean error of the rates 4.4e-15 instead of 3.6e-15).
template <int N>
__device__ __forceinline__ void exp64_rows(double* x) {
  double t[N], r[N];
  ROW t[i] = __builtin_fma(x[i], 0x1.71547652b82fep+0, 0x1.8p+52);
  ROW r[i] = t[i] - 0x1.8p+52;
  ROW r[i] = __builtin_fma(x[i], 0x1.71547652b82fep+0, -r[i]);
  pow2_rows<N>(x, t, r);
}
// log2 m for x = 2^e m > 0 with m in [sqrt(1/2), sqrt(2)): s P(s²) with s = (m-1)/(m+1) (the atanh series; P the
// Chebyshev interpolant of degree 7, exp_coefficients.py, relative error 1.4e-17)
template <int N>
__device__ __forceinline__ void mantissa_log_rows(const double* x, double* e, double* s, double* p) {
  double num[N], den[N], r[N], z[N];
  ROW {
    const double m = __builtin_amdgcn_frexp_mant(x[i]);
    const int low = m < 0x1.6a09e667f3bcdp-1;
    e[i] = (double)(__builtin_amdgcn_frexp_exp(x[i]) - low);
    num[i] = __builtin_ldexp(m, low);
    den[i] = r[i] = num[i] + 1.0;
    num[i] -= 1.0;
  }
  rcp64_rows<N>(r);
  ROW s[i] = num[i] * r[i];
  ROW z[i] = __builtin_fma(-s[i], den[i], num[i]);
  ROW s[i] = __builtin_fma(z[i], r[i], s[i]);
  ROW z[i] = s[i] * s[i];
  ROW p[i] = __builtin_fma(0x1.b592d3c48c41cp-3, z[i], 0x1.c46e1440404d7p-3);
  const double c[6] = {0x1.0ca160627dbfcp-2, 0x1.484afb7a67652p-2, 0x1.a61762d693934p-2,
                       0x1.2776c50ee39dcp-1, 0x1.ec709dc3a047dp-1, 0x1.71547652b82fep+1};
#pragma unroll
  for (int j = 0; j < 6; j++) {
    ROW p[i] = __builtin_fma(p[i], z[i], c[j]);
  }
}
template <int N>
__device__ __forceinline__ void log_rows(double* x) {
  double e[N], s[N], p[N];
  mantissa_log_rows<N>(x, e, s, p);
  ROW x[i] = __builtin_fma(s[i], p[i], e[i]);
}
// (one rounding at the size of the result: with ln 2 times log2 x the rates' mean error was 4.0e-15 instead of 3.6e-15)
__device__ __forceinline__ double log64(double x) {
  double e, s, p;
  mantissa_log_rows<1>(&x, &e, &s, &p);
  return __builtin_fma(e, 0x1.62e42fefa39efp-1, s * p * 0x1.62e42fefa39efp-1);
}
#endif
__device__ __forceinline__ double exp64(double x) {
  exp64_rows<1>(&x);
  return x;
}

extern "C" __global__ void __launch_bounds__(64 * PARTS * TEAMS)
NAME(const double* const* __restrict__ in, double* const* __restrict__ out, unsigned n, const double* __restrict__ rcp_W_,
     const double* __restrict__ gibbs_, double clamp_pos, double clamp_neg) {
  // rows of COLS states: F_k, then E-_k of the active species; at the end the parts' sums
  __shared__ double lds_v[@LDS_V@];
#if TEAMS > 1
  __shared__ double lds_c[K * COLS];
#else
  double* const lds_c = lds_v + 2 * KA * COLS;
#endif
  const table rcp_W = (table)rcp_W_, gibbs = (table)gibbs_;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int team = wave / PARTS, part = wave % PARTS;
  const unsigned col = 64 * team + (threadIdx.x & 63);
  const unsigned s = blockIdx.x * COLS + col;
  const bool valid = s < n;
  const unsigned sc = valid ? s : n - 1;  // states past n compute the last one again and write nothing

  // 1. concentrations and Gibbs exponentials
  const double T = in[0][sc], P = in[1][sc];
  double y[KP], sum = 0.0, positive = 0.0;
#pragma unroll
  for (int i = 0; i < KP; i++) y[i] = part + PARTS * i < K ? in[2 + part + PARTS * i][sc] * rcp_W[part + PARTS * i] : 0.0;
#pragma unroll
  for (int i = 0; i < KP; i++) {
    const int k = part + PARTS * i;
    sum += y[i];
    y[i] = __builtin_fmax(0.0, y[i]);
    if (k < K - 1) positive += y[i];
    if (k < K) lds_c[k * COLS + col] = y[i];
  }
  lds_v[part * COLS + col] = sum;
  lds_v[(PARTS + part) * COLS + col] = positive;
  // a second Newton step: 1/T stands in every exponent, tens of times over
  const double rT1 = rcp64(T), rcpT = __builtin_fma(rT1, __builtin_fma(-T, rT1, 1.0), rT1);
  const double L = log64(T), T2 = T * T, T3 = T * T2, T4 = T2 * T2;
  const double C_tot = P * (1.0 / RGAS) * rcpT;
  __syncthreads();
  sum = lds_v[col];
  positive = lds_v[PARTS * COLS + col];
#pragma unroll
  for (int p = 1; p < PARTS; p++) {
    sum += lds_v[p * COLS + col];
    positive += lds_v[(PARTS + p) * COLS + col];
  }
  const double density = C_tot * rcp64(sum);
  __syncthreads();
  // two species a turn, a loop rather than straight-line code: their coefficients are all that the scalar registers hold
#pragma unroll 1
  for (int k0 = part; k0 < K; k0 += 2 * PARTS) {
    double E[2], c[2];
#pragma unroll
    for (int i = 0; i < 2; i++) {
      const int k = k0 + i * PARTS, kc = k < K ? k : K - 1;
      const table a = gibbs + 15 * (k < KA ? k : KA - 1);
      c[i] = kc < K - 1 ? density * lds_c[kc * COLS + col] : C_tot - density * positive;
      const double lo = a[1] + (a[2] * L + a[3] * T + a[4] * T2 + a[5] * T3 + a[6] * T4 + a[7] * rcpT);
      const double hi = a[8] + (a[9] * L + a[10] * T + a[11] * T2 + a[12] * T3 + a[13] * T4 + a[14] * rcpT);
      E[i] = FAST ? (T <= a[0] ? lo : hi) : __builtin_fmax(T <= a[0] ? lo : hi, -1100.0);
    }
    exp64_rows<2>(E);
    double rE[2];
#pragma unroll
    for (int i = 0; i < 2; i++) rE[i] = E[i] = SCALE * __builtin_fmin(E[i], 0x1p+920);
    rcp64_rows<2>(rE);
#pragma unroll
    for (int i = 0; i < 2; i++) {
      const int k = k0 + i * PARTS;
      if (k < K) lds_c[k * COLS + col] = c[i];
      if (k < KA) {
        lds_v[k * COLS + col] = __builtin_fmin(SCALE * clamp_pos, E[i]) * c[i];
        lds_v[(KA + k) * COLS + col] = __builtin_fmin(clamp_neg / SCALE, rE[i]);
      }
    }
  }
  __syncthreads();

  // 2. the part's reactions
  const double* const c_ = lds_c + col;
  const double* const f_ = lds_v + col;
  const double* const e_ = lds_v + KA * COLS + col;
#define C(k) c_[(k) * COLS]
#define F(k) f_[(k) * COLS]
#define EN(k) e_[(k) * COLS]
  const double C0 = SCALE * P0_R * rcpT, rcpC0 = T * (1.0 / (SCALE * P0_R));
  const double rcpT2 = rcpT * rcpT;
#define LIMIT(x) __builtin_fmin(FLT_MAX_D, x)
#if FAST
#define KF(x) exp64(x)
#else
  // 1/T and ln T as the rate constants' exponents take them, kept where 2^30 bounds the exponents (below 1 mK and
  // outside the FP64 range every rate constant is 0 or FLT_MAX by then)
  const double rT = __builtin_fmin(rcpT, 1e3), LT = __builtin_fmin(__builtin_fmax(L, -760.0), 760.0);
#define KF(x) exp64(__builtin_fmin(LN_FLT_MAX, x))
#endif
@SECTIONS@
  // 3. sums over the parts
  __syncthreads();
  if (part >= PARTS / 2) {
    double* const row = SUMS(part - PARTS / 2);
@STORE@
  }
  __syncthreads();
  if (part < PARTS / 2) {
    double* const row = SUMS(part);
@ADD@
  }
  __syncthreads();
  if (!valid) return;
#pragma unroll
  for (int i = 0; i < (KA + PARTS - 1) / PARTS; i++) {
    const int k = part + PARTS * i;
    if (k < KA) {
      double w = lds_v[k * COLS + col];
#pragma unroll
      for (int p = 1; p < PARTS / 2; p++) w += SUMS(p)[k * COLS];
      out[k][s] = w;
    }
  }
}
