// Mixture-averaged transport in FP64 for mechanisms of 65 to 160 species (hand-written; the host prepends the sizes).
//
// A block of WAVES waves owns 64 states, one lane per state in every wave; wave w owns species w, w + WAVES, ..
// (SW = ⌈K/WAVES⌉ slots). x_k and one array of sums fill the CU's LDS (2 K - 1 rows of 64 states: the bulk species' x is
// in a register of every wave). With x_k = C_k and the fits in l = ln(T/T0) (transport.rs:125-136), v_k scaled by
// W_k^(-1/4):
//   λ = ½ √T (Σ x_k c_k / N + N / Σ x_k / c_k)                                    (transport.rs:141-146)
//   μ = √T Σ_k √W_k x_k v_k² / den_k, den_k = d0 + 2 v_k d1 + v_k² d2             (transport.rs:148-158), the moments
//       d_m = Σ_j 1/√(W_k + W_j) · √(W_j/8) x_j v_j^(-m) by the pivoted Cholesky factor G (K×R) of 1/√(W_k + W_j):
//       d_m = G (Gᵀ y_m), exact to rounding at R = 19 of 160
//   ρD_k = √T (Σ_j W_j x_j - W_k x_k) / (R S_k),  S_k = Σ_{j≠k} x_j / d_kj(l)       (transport.rs:162-177)
//       every pair once: in phase p wave w takes its own species against those of wave w + p (phase 0: among its own;
//       phase WAVES/2: half of them, the opposite wave the other half), its own sums in registers, the others' through
//       LDS (one writer per row between barriers). The fits normalised by their constant term; the reciprocals of a
//       column's pairs from one or two reciprocals of their products.
// The pairs' constants are wave-uniform and used once: each wave streams its own through scalar loads, whose latency the
// other three waves of its SIMD cover.
//
// Bound: FP64 VALU issue and the constants' latency. 171 k VALU instructions per 64 states of 160 species, four waves per
// SIMD, VALU busy 63 % of the time (the waves wait 56 % of theirs, mostly for their constants): 2^17 states take 1.00 ms
// against 2.09 ms for transport_tiled, whose FP64 MFMA tiles have the VALU's rate on this chip and do not overlap it.
// Measured and not kept: half a column's constants fetched ahead of the other half's arithmetic (5 % longer: 106 scalar
// registers do not hold both).
// Rounding: 1.1e-16, 1.1e-16 and 1.9e-16 of λ, μ and ρD on average against the formulas in 80-bit arithmetic (160 species);
// transport_tiled 1.3e-16, 1.4e-16 and 2.1e-16. The reciprocals, quotients and the order of the sums below are for that: they
// took 4 % more instructions and 1.2 % of the time.
// Required defines: K, R (rank), DD (fit length), WAVES (a power of two).
// Tables: rcp_W[K], W[K], fit_c[K][DD], fit_v[K][DD] (v scaled), columns[R][KC] = √(W_j/8) G_jr (KC = K rounded up to 8),
// rows[WAVES][R][SW] = G_kr / √W_k, pairs[WAVES][..] = per wave its pairs' DD constants in the order of the phases
// (c_1/c_0, .., 1/c_0; a slot without species: 0, .., 0), offset[WAVES] into it.

typedef const double __attribute__((address_space(4))) * table;  // read by scalar loads at wave-uniform indices

#define RGAS (1.380649e-23 * 6.02214076e23)
#define SW ((K + WAVES - 1) / WAVES)
#define KC ((K + 7) / 8 * 8)
#define HALF (SW / 2)

// 1/b: v_rcp_f64 (r, relative error e below 2^-24) times 1 + e + e² (error e³: the last rounding is all there is). A Newton
// step, 1 + e, is always low, by 3e-16 on average, which the sums do not average out.
__device__ __forceinline__ double rcp64(double b) {
  const double r = __builtin_amdgcn_rcp(b), e = __builtin_fma(-b, r, 1.0);
  return __builtin_fma(r, __builtin_fma(e, e, e), r);
}
// a/b, rounded once or nearly
__device__ __forceinline__ double quotient(double a, double b) {
  const double r = rcp64(b), q = a * r;
  return __builtin_fma(__builtin_fma(-b, q, a), r, q);
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
  return __builtin_fma((double)e, 0x1.62e42fefa39efp-1, s * p * 0x1.62e42fefa39efp-1);
}

// 1/y of N values from one reciprocal of their product (prefix products, then back; the y are near 1)
template <int N>
__device__ __forceinline__ void rcp_all(double* y) {
  double prefix[N];
  prefix[0] = y[0];
#pragma unroll
  for (int i = 1; i < N; i++) prefix[i] = prefix[i - 1] * y[i];
  double q = rcp64(prefix[N - 1]);
#pragma unroll
  for (int i = N - 1; i > 0; i--) {
    const double r = q * prefix[i - 1];
    q *= y[i];
    y[i] = r;
  }
  y[0] = q;
}

// R_i = 1/d of the N pairs whose constants start at t
template <int N>
__device__ __forceinline__ void reciprocals(const double* t, const double* pw, double* r) {
#pragma unroll
  for (int i = 0; i < N; i++) {
    double y = 1.0;
#pragma unroll
    for (int d = 1; d < DD; d++) y = __builtin_fma(t[i * DD + d - 1], pw[d], y);
    r[i] = y;
  }
  rcp_all<N>(r);
#pragma unroll
  for (int i = 0; i < N; i++) r[i] *= t[i * DD + DD - 1];
}

// Column j (another wave's species) against the wave's slots [0, N), in two batches.
template <int N>
__device__ __forceinline__ void column(table& t, const double* pw, double xj, double* sj, const double* x, double* g) {
  constexpr int A = (N + 1) / 2, B = N - A;
  double c[N * DD], ra[A];
#pragma unroll
  for (int i = 0; i < N * DD; i++) c[i] = t[i];
  t += N * DD;
  double s = 0.0;  // the column's own sum first: a chain of all the pairs of j would round at the size of S_j each time
  reciprocals<A>(c, pw, ra);
#pragma unroll
  for (int i = 0; i < A; i++) {
    g[i] = __builtin_fma(xj, ra[i], g[i]);
    s = i ? __builtin_fma(x[i], ra[i], s) : x[i] * ra[i];
  }
  if constexpr (B > 0) {
    double rb[B];
    reciprocals<B>(c + A * DD, pw, rb);
#pragma unroll
    for (int i = 0; i < B; i++) {
      g[A + i] = __builtin_fma(xj, rb[i], g[A + i]);
      s = __builtin_fma(x[A + i], rb[i], s);
    }
  }
  *sj += s;
}

// The waves' values in the rows p[64 w], added in pairs
__device__ __forceinline__ double waves_sum(const double* p) {
  double v[WAVES];
#pragma unroll
  for (int w = 0; w < WAVES; w++) v[w] = p[64 * w];
#pragma unroll
  for (int n = WAVES / 2; n > 0; n /= 2) {
#pragma unroll
    for (int w = 0; w < n; w++) v[w] += v[w + n];
  }
  return v[0];
}

extern "C" __global__ void __launch_bounds__(64 * WAVES)
transport_tiled(const double* const* __restrict__ in, double* const* __restrict__ out, unsigned n, const double* __restrict__ rcp_W_,
                const double* __restrict__ W_, const double* __restrict__ fit_c_, const double* __restrict__ fit_v_,
                const double* __restrict__ columns_, const double* __restrict__ rows_, const double* __restrict__ pairs_,
                const unsigned* __restrict__ offset, double T0) {
  __shared__ double lds_x[(K - 1) * 64];  // x_k without the bulk species'
  __shared__ double lds_s[K * 64];        // 1/v_k, then Gᵀ y_m, then S_k
  const table rcp_W = (table)rcp_W_, W = (table)W_, fit_c = (table)fit_c_, fit_v = (table)fit_v_;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const unsigned lane = threadIdx.x & 63, s = blockIdx.x * 64 + lane;
  const unsigned sc = s < n ? s : n - 1;  // states past n compute the last one again and write nothing
  const double* const x_ = lds_x + lane;
  double* const s_ = lds_s + lane;

  // 1. concentrations (amounts n_k = Y_k/W_k, C_k = max(0, n_k) C_tot/Σn, bulk C_tot - Σ), fits, conductivity sums
  const double T = in[0][sc], P = in[1][sc];
  double x[SW];
  double sum = 0.0, positive = 0.0, mass = 0.0;
#pragma unroll
  for (int i = 0; i < SW; i++) x[i] = wave + WAVES * i < K ? in[2 + wave + WAVES * i][sc] : 0.0;
#pragma unroll
  for (int i = 0; i < SW; i++) {
    const int k = wave + WAVES * i;
    const double y = x[i], a = k < K ? y * rcp_W[k] : 0.0;
    sum += a;
    x[i] = __builtin_fmax(0.0, a);
    if (k < K - 1) {
      positive += x[i];
      mass += __builtin_fmax(0.0, y);
    }
  }
  s_[wave * 64] = sum;
  s_[(WAVES + wave) * 64] = positive;
  s_[(2 * WAVES + wave) * 64] = mass;
  const double l = log64(T / T0), C_tot = quotient(quotient(P, RGAS), T);
  double pw[DD];
  pw[0] = 1.0;
#pragma unroll
  for (int d = 1; d < DD; d++) pw[d] = pw[d - 1] * l;
  __syncthreads();
  sum = waves_sum(s_);
  positive = waves_sum(s_ + WAVES * 64);
  mass = waves_sum(s_ + 2 * WAVES * 64);
  const double density = quotient(C_tot, sum), bulk = C_tot - density * positive;
  const double WN = density * mass + W[K - 1] * bulk;  // Σ W_k x_k
  __syncthreads();
  double v[SW], A = 0.0, B = 0.0;
#pragma unroll
  for (int i = 0; i < SW; i++) {
    const int k = wave + WAVES * i;
    x[i] = k < K - 1 ? density * x[i] : k < K ? bulk : 0.0;
    v[i] = 1.0;
    if (k < K) {
      double c = fit_c[k * DD], u = fit_v[k * DD];
#pragma unroll
      for (int d = 1; d < DD; d++) {
        c += fit_c[k * DD + d] * pw[d];
        u += fit_v[k * DD + d] * pw[d];
      }
      A += x[i] * c;
      B += quotient(x[i], c);
      v[i] = u;
      if (k < K - 1) lds_x[k * 64 + lane] = x[i];
      s_[k * 64] = rcp64(u);
    }
  }
  __syncthreads();

  // 2. viscosity: Gᵀ y_m for the columns r = wave, wave + WAVES, .., then the wave's species' rows of G (Gᵀ y_m)
  constexpr int RW = (R + WAVES - 1) / WAVES;
  double z[RW][3];
#pragma unroll
  for (int q = 0; q < RW; q++) {
    z[q][0] = z[q][1] = z[q][2] = 0.0;
    const int r = wave + WAVES * q;
    if (r < R) {
      const table c = (table)columns_ + r * KC;
#pragma unroll 1
      for (int j0 = 0; j0 < K; j0 += 8) {
        double part[3];  // eight species first, for the same reason as a column's sum
#pragma unroll
        for (int j = 0; j < 8; j++) {
          // past the species: a constant of zero, and the bulk's concentration
          const int k = j0 + j < K ? j0 + j : K - 1;
          const double xj = k < K - 1 ? x_[k * 64] : bulk, u = s_[k * 64], y1 = xj * u;
          part[0] = j ? __builtin_fma(c[j0 + j], xj, part[0]) : c[j0] * xj;
          part[1] = j ? __builtin_fma(c[j0 + j], y1, part[1]) : c[j0] * y1;
          part[2] = j ? __builtin_fma(c[j0 + j], y1 * u, part[2]) : c[j0] * (y1 * u);
        }
#pragma unroll
        for (int m = 0; m < 3; m++) z[q][m] += part[m];
      }
    }
  }
  __syncthreads();
#pragma unroll
  for (int q = 0; q < RW; q++) {
    const int r = wave + WAVES * q;
    if (r < R) {
#pragma unroll
      for (int m = 0; m < 3; m++) s_[(3 * r + m) * 64] = z[q][m];
    }
  }
  __syncthreads();
  double mu = 0.0;
  {
    double d0[SW], d1[SW], d2[SW];  // the moments over √W_k
#pragma unroll
    for (int i = 0; i < SW; i++) d0[i] = d1[i] = d2[i] = 0.0;
    const table c = (table)rows_ + wave * R * SW;
#pragma unroll 1
    for (int r = 0; r < R; r++) {
      const double z0 = s_[3 * r * 64], z1 = s_[(3 * r + 1) * 64], z2 = s_[(3 * r + 2) * 64];
#pragma unroll
      for (int i = 0; i < SW; i++) {
        const double G = c[r * SW + i];
        d0[i] = __builtin_fma(G, z0, d0[i]);
        d1[i] = __builtin_fma(G, z1, d1[i]);
        d2[i] = __builtin_fma(G, z2, d2[i]);
      }
    }
    asm volatile("" ::: "memory");  // x from LDS again: its registers served the moments
#pragma unroll
    for (int i = 0; i < SW; i++) {
      const int k = wave + WAVES * i;
      x[i] = k < K - 1 ? x_[k * 64] : k < K ? bulk : 0.0;
    }
#pragma unroll
    for (int i = 0; i < SW; i++)
      if (wave + WAVES * i < K) mu += quotient(x[i] * (v[i] * v[i]), d0[i] + v[i] * (2.0 * d1[i] + v[i] * d2[i]));
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < SW; i++)
    if (wave + WAVES * i < K) s_[(wave + WAVES * i) * 64] = 0.0;

  // 3. diffusion
  double g[SW];
#pragma unroll
  for (int i = 0; i < SW; i++) g[i] = 0.0;
  table t = (table)pairs_ + __builtin_amdgcn_readfirstlane(offset[wave]);
#pragma unroll
  for (int a = 1; a < SW; a++) {  // phase 0: slot a against the slots below it
    constexpr int M = 4;
#pragma unroll
    for (int b0 = 0; b0 < a; b0 += M) {
      const int N = a - b0 < M ? a - b0 : M;
      double r[M], c[M * DD];
#pragma unroll
      for (int i = 0; i < M * DD; i++) c[i] = i < N * DD ? t[i] : 0.0;  // past the row: 1/1, times zero
      t += N * DD;
      reciprocals<M>(c, pw, r);
#pragma unroll
      for (int i = 0; i < M; i++)
        if (i < N) {
          g[a] = __builtin_fma(x[b0 + i], r[i], g[a]);
          g[b0 + i] = __builtin_fma(x[a], r[i], g[b0 + i]);
        }
    }
  }
  __syncthreads();
#pragma unroll 1
  for (int p = 1; p < WAVES / 2; p++) {
    const int other = (wave + p) % WAVES;
#pragma unroll 1
    for (int j = other; j < K; j += WAVES) column<SW>(t, pw, j < K - 1 ? x_[j * 64] : bulk, s_ + j * 64, x, g);
    __syncthreads();
  }
  if (wave < WAVES / 2) {  // the lower slots against all of the opposite wave's species
#pragma unroll 1
    for (int j = wave + WAVES / 2; j < K; j += WAVES) column<HALF>(t, pw, j < K - 1 ? x_[j * 64] : bulk, s_ + j * 64, x, g);
  } else {  // all slots against the opposite wave's upper ones
#pragma unroll 1
    for (int j = wave - WAVES / 2 + WAVES * HALF; j < K; j += WAVES) column<SW>(t, pw, j < K - 1 ? x_[j * 64] : bulk, s_ + j * 64, x, g);
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < SW; i++)
    if (wave + WAVES * i < K) g[i] += s_[(wave + WAVES * i) * 64];

  // 4. outputs; λ's and μ's sums over the waves through the x rows
  double* const p_ = lds_x + lane;
  p_[wave * 64] = A;
  p_[(WAVES + wave) * 64] = B;
  p_[(2 * WAVES + wave) * 64] = mu;
  __syncthreads();
  if (s >= n) return;
  const double root_T = __builtin_sqrt(T);
  if (wave == 0) {
    A = waves_sum(p_);
    B = waves_sum(p_ + WAVES * 64);
    out[0][s] = 0.5 * root_T * (quotient(A, C_tot) + quotient(C_tot, B));
  }
  if (wave == 1) {
    out[1][s] = root_T * waves_sum(p_ + 2 * WAVES * 64);
  }
  const double scale = quotient(root_T, RGAS * WN);
#pragma unroll
  for (int i = 0; i < SW; i++) {
    const int k = wave + WAVES * i;
    if (k < K) out[2 + k][s] = quotient(scale * (WN - W[k] * x[i]), g[i]);
  }
}
