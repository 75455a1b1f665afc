// Mixture-averaged transport in FP64 for mechanisms of up to 64 species (hand-written frame; the host prepends the
// sizes and fills in each wave's straight-line share of the sums).
//
// A block of four waves owns 64 states, one lane per state in every wave; wave w owns species w, w + 4, .. With
// x_k = C_k and the fits in l = ln(T/T0) (transport.rs:125-136), v_k scaled by W_k^(-1/4):
//   λ = ½ √T (Σ x_k c_k / N + N / Σ x_k / c_k)                                    (transport.rs:141-146)
//   μ = √T Σ_k √W_k x_k v_k² / den_k, den_k = Σ_j x_j (1 + v_k/v_j)² √W_j / √8 / √(W_j + W_k)  (transport.rs:148-158)
//       = d0 + 2 v_k d1 + v_k² d2 with the moments d_m = Σ_j 1/√(W_k + W_j) · √(W_j/8) x_j v_j^(-m). The matrix
//       1/√(W_k + W_j) is positive definite and of low numerical rank: its pivoted Cholesky factor G (K×R, the host
//       stops when no entry is off by 2^-56 of its size) gives d_m = G (Gᵀ y_m), 6 K R products instead of 3 K².
//       The factors' products stay within a few per cent of the entries they sum to, so nothing cancels.
//   ρD_k = √T (Σ_j W_j x_j - W_k x_k) / (R S_k),  S_k = Σ_{j≠k} x_j / d_kj(l)       (transport.rs:162-177)
//       every pair once: the waves' species sets in turn against their own, the next wave's and, half each, the one
//       after that; a wave's own sums stay in registers, the others' go through LDS (one writer per row between
//       barriers). The fits normalised by their constant term, four reciprocals from one.
// Bound: FP64 VALU issue (22.0 k VALU instructions per 64 states of the 53-species mechanism, 14.3 k of them for its 1378
// pairs, where one lane per state took 26.2 k), at three waves per SIMD, which the 105 rows of LDS just allow (the bulk
// species' x stays in a register for that). 2^20 states of 53 species: 0.90 ms against 1.01 ms for one lane per state
// (VALU busy 83 % of the time); 64 states: 30 against 84 us. Measured and not kept: the sections' constants by scalar
// loads one block ahead instead of s_mov pairs (a third longer: every wait for one is a wait for all), two waves per
// SIMD (11 % longer), FP64 MFMA for the moments (v_mfma_f64_16x16x4 has the VALU's rate on this chip and does not overlap it).
// Required defines: K, R (rank), DD (fit length).
// Tables: rcp_W[K], W[K], fit_c[K][DD], fit_v[K][DD] (v scaled).

typedef const double __attribute__((address_space(4))) * table;  // read by scalar loads at wave-uniform indices

#define RGAS (1.380649e-23 * 6.02214076e23)
#define WAVES 4
#define KW ((K + WAVES - 1) / WAVES)  // species per wave
#define RW ((R + WAVES - 1) / WAVES)  // Cholesky columns per wave
#define ROWS_S (K > 3 * R ? K : 3 * R)

// 1/b: v_rcp_f64 (relative error below 2^-24) and one Newton step (2.2e-15)
__device__ __forceinline__ double rcp64(double b) {
  const double r = __builtin_amdgcn_rcp(b);
  return __builtin_fma(r, __builtin_fma(-b, r, 1.0), r);
}
// ln x for x > 0: x = 2^e m with m in [sqrt(1/2), sqrt(2)), log2 m = s P(s²) with s = (m-1)/(m+1) (the atanh series; P
// the Chebyshev interpolant of degree 7, relative error 1.4e-17)
__device__ __forceinline__ double log64(double x) {
  double m = __builtin_amdgcn_frexp_mant(x);
  int e = __builtin_amdgcn_frexp_exp(x);
  const int low = m < 0x1.6a09e667f3bcdp-1;
  m = __builtin_ldexp(m, low);
  e -= low;
  const double num = m - 1.0, den = m + 1.0;
  const double r = rcp64(den);
  double s = num * r;
  s = __builtin_fma(__builtin_fma(-s, den, num), r, s);
  const double z = s * s;
  double p = 0x1.b592d3c48c41cp-3;
  p = __builtin_fma(p, z, 0x1.c46e1440404d7p-3);
  p = __builtin_fma(p, z, 0x1.0ca160627dbfcp-2);
  p = __builtin_fma(p, z, 0x1.484afb7a67652p-2);
  p = __builtin_fma(p, z, 0x1.a61762d693934p-2);
  p = __builtin_fma(p, z, 0x1.2776c50ee39dcp-1);
  p = __builtin_fma(p, z, 0x1.ec709dc3a047dp-1);
  p = __builtin_fma(p, z, 0x1.71547652b82fep+1);
  return __builtin_fma(s, p, (double)e) * 0x1.62e42fefa39efp-1;
}

// (the first of two bounds on the waves per SIMD holds: three)
extern "C" __global__ void __attribute__((amdgpu_waves_per_eu(3))) __launch_bounds__(256, 2)
transport_fp64(const double* const* __restrict__ in, double* const* __restrict__ out, unsigned n, const double* __restrict__ rcp_W_,
               const double* __restrict__ W_, const double* __restrict__ fit_c_, const double* __restrict__ fit_v_, double rcp_T0) {
  __shared__ double lds_x[(K - 1) * 64];  // x_k without the bulk species'
  __shared__ double lds_s[ROWS_S * 64];  // 1/v_k, then Gᵀ y_m, then S_k
  const table rcp_W = (table)rcp_W_, W = (table)W_, fit_c = (table)fit_c_, fit_v = (table)fit_v_;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const unsigned lane = threadIdx.x & 63, s = blockIdx.x * 64 + lane;
  const unsigned sc = s < n ? s : n - 1;  // states past n compute the last one again and write nothing

  // 1. concentrations (amounts n_k = Y_k/W_k, C_k = max(0, n_k) C_tot/Σn, bulk C_tot - Σ), fits, conductivity sums
  const double T = in[0][sc], P = in[1][sc];
  double x[KW];
  double sum = 0.0, positive = 0.0, mass = 0.0;
#pragma unroll
  for (int i = 0; i < KW; i++) x[i] = wave + WAVES * i < K ? in[2 + wave + WAVES * i][sc] : 0.0;
#pragma unroll
  for (int i = 0; i < KW; i++) {
    const int k = wave + WAVES * i;
    const double y = x[i], a = k < K ? y * rcp_W[k] : 0.0;
    sum += a;
    x[i] = __builtin_fmax(0.0, a);
    if (k < K - 1) {
      positive += x[i];
      mass += __builtin_fmax(0.0, y);
    }
  }
  lds_s[wave * 64 + lane] = sum;
  lds_s[(WAVES + wave) * 64 + lane] = positive;
  lds_s[(2 * WAVES + wave) * 64 + lane] = mass;
  const double l = log64(T * rcp_T0), C_tot = P * (1.0 / RGAS) * rcp64(T);
  double pw[DD];
  pw[0] = 1.0;
#pragma unroll
  for (int d = 1; d < DD; d++) pw[d] = pw[d - 1] * l;
  __syncthreads();
  sum = lds_s[lane];
  positive = lds_s[WAVES * 64 + lane];
  mass = lds_s[2 * WAVES * 64 + lane];
#pragma unroll
  for (int w = 1; w < WAVES; w++) {
    sum += lds_s[w * 64 + lane];
    positive += lds_s[(WAVES + w) * 64 + lane];
    mass += lds_s[(2 * WAVES + w) * 64 + lane];
  }
  const double density = C_tot * rcp64(sum), bulk = C_tot - density * positive;
  const double WN = __builtin_fma(W[K - 1], bulk, density * mass);  // Σ W_k x_k
  __syncthreads();
  double v[KW], A = 0.0, B = 0.0;
#pragma unroll
  for (int i = 0; i < KW; i++) {
    const int k = wave + WAVES * i;
    if (k < K) {
      x[i] = k < K - 1 ? density * x[i] : bulk;
      double c = fit_c[k * DD], u = fit_v[k * DD];
#pragma unroll
      for (int d = 1; d < DD; d++) {
        c += fit_c[k * DD + d] * pw[d];
        u += fit_v[k * DD + d] * pw[d];
      }
      A += x[i] * c;
      B += x[i] * rcp64(c);
      v[i] = u;
      if (k < K - 1) lds_x[k * 64 + lane] = x[i];
      lds_s[k * 64 + lane] = rcp64(u);
    } else {
      x[i] = v[i] = 0.0;
    }
  }
  __syncthreads();

  // 2. viscosity: wave w's columns of Gᵀ y_m (rows 3 r + m), then its species' rows of G (Gᵀ y_m)
  const double* const x_ = lds_x + lane;
  double* const s_ = lds_s + lane;
#define X(k) ((k) < K - 1 ? x_[(k) * 64] : bulk)
#define S(k) s_[(k) * 64]
  double z[RW][3];
@COLUMNS@
  __syncthreads();
#pragma unroll
  for (int i = 0; i < RW; i++)
    if (wave + WAVES * i < R) {
      S(3 * (wave + WAVES * i)) = z[i][0];
      S(3 * (wave + WAVES * i) + 1) = z[i][1];
      S(3 * (wave + WAVES * i) + 2) = z[i][2];
    }
  __syncthreads();
  double d0[KW], d1[KW], d2[KW], mu = 0.0;  // the moments over √W_k
@ROWS@
  asm volatile("" ::: "memory");  // x from LDS again: its registers served the moments (three waves per SIMD)
#pragma unroll
  for (int i = 0; i < KW; i++) {
    const int k = wave + WAVES * i;
    if (k < K) {
      x[i] = X(k);
      const double den = __builtin_fma(v[i], __builtin_fma(v[i], d2[i], 2.0 * d1[i]), d0[i]);
      mu = __builtin_fma(x[i] * (v[i] * v[i]), rcp64(den), mu);
    }
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < KW; i++)
    if (wave + WAVES * i < K) S(wave + WAVES * i) = 0.0;

  // 3. diffusion: g[i] = the wave's own Σ_j x_j / d_kj, the others' species' terms added into S(j)
  double g[KW];
#pragma unroll
  for (int i = 0; i < KW; i++) g[i] = 0.0;
@PAIRS@
  __syncthreads();
#pragma unroll
  for (int i = 0; i < KW; i++)
    if (wave + WAVES * i < K) g[i] += S(wave + WAVES * i);
  // λ and μ of the four waves, over the x rows
  double* const p_ = lds_x + lane;
  p_[wave * 64] = A;
  p_[(WAVES + wave) * 64] = B;
  p_[(2 * WAVES + wave) * 64] = mu;
  __syncthreads();
  if (s >= n) return;
  const double root_T = __builtin_sqrt(T);
  if (wave == 0) {
#pragma unroll
    for (int w = 1; w < WAVES; w++) {
      A += p_[w * 64];
      B += p_[(WAVES + w) * 64];
    }
    out[0][s] = 0.5 * root_T * (A * rcp64(C_tot) + C_tot * rcp64(B));
  }
  if (wave == 1) {
    mu = p_[2 * WAVES * 64];
#pragma unroll
    for (int w = 1; w < WAVES; w++) mu += p_[(2 * WAVES + w) * 64];
    out[1][s] = root_T * mu;
  }
  const double scale = root_T * rcp64(RGAS * WN);
#pragma unroll
  for (int i = 0; i < KW; i++) {
    const int k = wave + WAVES * i;
    if (k < K) out[2 + k][s] = scale * (WN - W[k] * x[i]) * rcp64(g[i]);
  }
}
