// Dense layers of the transport surrogate (training): BF16 operands, FP32 accumulation on v_mfma_f32_16x16x16bf16_1k.
// Three kernels carry a training step, whatever the number of layers; every dimension is a multiple of 64 (the host pads
// features), the number of states is any:
//   mlp_forward   all layers: a block takes 64 states through the whole network, their activations in LDS
//   mlp_backward  the gradients by the pre-activations of two layers, likewise 64 states a block
//   mlp_weights   the weight and bias gradients of those two layers, split over ranges of states
// All three are bound by what must go through memory: the pre-activations (FP32) and activations (BF16) that the backward
// pass needs. 2^14 states of a 55-256-256-256-55 network: a step (forward, backward, Adam) takes
// 116 us in 8 launches, against 407 in 28 launches layer by layer.
// Networks whose widest layer is above 576 take mlp_gemm layer by layer (two activation tiles of 64 states no longer fit
// the 160 KB of LDS).

typedef short bf16x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef unsigned short u16;

#define LDSK 40  // 32 k plus 8 of padding per row

__device__ __forceinline__ u16 to_bf16(float x) {
  unsigned u = __float_as_uint(x);
  u += 0x7FFFu + ((u >> 16) & 1u);
  return (u16)(u >> 16);
}
__device__ __forceinline__ float from_bf16(u16 b) { return __uint_as_float((unsigned)b << 16); }
__device__ __forceinline__ float sigmoid(float z) { return __builtin_amdgcn_rcpf(1.f + __builtin_amdgcn_exp2f(-z * 1.4426950408889634f)); }

__device__ __forceinline__ float silu_derivative_times(float c, float z) {
  const float s = sigmoid(z);
  return c * s * (1.f + z * (1.f - s));
}
__device__ __forceinline__ unsigned pair(float a, float b) { return (unsigned)to_bf16(a) | (unsigned)to_bf16(b) << 16; }

#define ROWS 64  // states per block

// The network on 64 states a block: activations alternate between two LDS tiles (row length ld = the widest layer + 16
// BF16: rows 8 banks apart, so that the 32 lanes of half a ds_read_b64 use all 64 banks), weights come from L2. A wave
// computes 64 states × 32 outputs. A lane reads 16 bytes of a weight row, 8 of 32 k, the lanes of the second and third 16
// each other's; one v_permlane16_swap a dword then gives the fragments of the two products over 16 k. The weights are the
// first operand, so that a lane ends with 8 consecutive outputs of one state (row 4Q + r of tile t is output 8Q + 2r + t):
// whole 16-byte stores of z and h. The products run over k in mlp_gemm's order, with the same rounding points.
// 32 us for 2^14 states of 55-256-256-256-55 (84 MB written), 128 registers a lane so that two blocks share a CU when
// there are more than 256; four products of mlp_gemm took 85. Measured and not kept: weights read 8 bytes a lane (38), 32
// states a block (52: twice the weight reads), weights through LDS, 64 k of 256 outputs at a time (43).
extern "C" __global__ void __launch_bounds__(512, 4)
mlp_forward(const float* __restrict__ x, const float* __restrict__ params, const u16* __restrict__ params16, long n, int in, int width,
            int out, int depth, int ld, u16* __restrict__ h0, float* __restrict__ z0, u16* __restrict__ h1, long layer_bytes,
            float* __restrict__ y) {
  extern __shared__ __attribute__((aligned(16))) u16 act[];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, c = lane & 15, q = lane >> 4;
  const long m0 = (long)blockIdx.x * ROWS;
  u16 *cur = act, *next = act + ROWS * ld;
  const int quads = in >> 2;
  for (int i = tid; i < ROWS * quads; i += 512) {
    const int row = i / quads, col = (i - row * quads) * 4;
    uint2 v = {0u, 0u};
    if (m0 + row < n) {
      const float4 f = *(const float4*)(x + (m0 + row) * in + col);
      v = {pair(f.x, f.y), pair(f.z, f.w)};
      *(uint2*)(h0 + (m0 + row) * in + col) = v;
    }
    *(uint2*)(cur + row * ld + col) = v;
  }
  __syncthreads();
  const u16* w16 = params16;
  const float* w32 = params;
  int K = in;
  for (int l = 0; l <= depth; l++) {
    const int N = l == depth ? out : width;
    const float* bias = w32 + (long)N * K;
    float* z = (float*)((char*)z0 + l * layer_bytes);
    u16* h = (u16*)((char*)h1 + l * layer_bytes);
    for (int nb = wave * 32; nb < N; nb += 256) {
      const u16* wrow = w16 + (long)(nb + 2 * c) * K + 8 * (q == 1 ? 2 : q == 2 ? 1 : q);
      f32x4 acc[4][2];
      uint4 w[2][2], ahead[2][2];  // [32 k][tile]
#pragma unroll
      for (int i = 0; i < 4; i++)
#pragma unroll
        for (int t = 0; t < 2; t++) acc[i][t] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int i = 0; i < 2; i++)
#pragma unroll
        for (int t = 0; t < 2; t++) {
          ahead[i][t] = *(const uint4*)(wrow + t * K + 32 * i);
        }
      for (int k0 = 0; k0 < K; k0 += 64) {
#pragma unroll
        for (int i = 0; i < 2; i++)
#pragma unroll
          for (int t = 0; t < 2; t++) {
            w[i][t] = ahead[i][t];
            if (k0 + 64 < K) ahead[i][t] = *(const uint4*)(wrow + t * K + k0 + 64 + 32 * i);
          }
#pragma unroll
        for (int kk = 0; kk < 2; kk++) {
          bf16x4 b[2][2];
#pragma unroll
          for (int t = 0; t < 2; t++) {
            const auto p = __builtin_amdgcn_permlane16_swap(w[kk][t].x, w[kk][t].z, false, false);
            const auto r = __builtin_amdgcn_permlane16_swap(w[kk][t].y, w[kk][t].w, false, false);
            b[0][t] = __builtin_bit_cast(bf16x4, (uint2){p[0], r[0]});
            b[1][t] = __builtin_bit_cast(bf16x4, (uint2){p[1], r[1]});
          }
#pragma unroll
          for (int u = 0; u < 2; u++) {
            bf16x4 a[4];
#pragma unroll
            for (int i = 0; i < 4; i++) a[i] = *(const bf16x4*)(cur + (16 * i + c) * ld + k0 + 32 * kk + 16 * u + 4 * q);
#pragma unroll
            for (int i = 0; i < 4; i++)
#pragma unroll
              for (int t = 0; t < 2; t++) acc[i][t] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(b[u][t], a[i], acc[i][t], 0, 0, 0);
          }
        }
      }
      const int col = nb + 8 * q;
      float bs[8];
#pragma unroll
      for (int j = 0; j < 8; j++) bs[j] = bias[col + j];
#pragma unroll
      for (int i = 0; i < 4; i++) {
        const int row = 16 * i + c;
        const bool in_batch = m0 + row < n;
        float v[8];
#pragma unroll
        for (int r = 0; r < 4; r++)
#pragma unroll
          for (int t = 0; t < 2; t++) v[2 * r + t] = acc[i][t][r] + bs[2 * r + t];
        float* to = (l == depth ? y : z) + (m0 + row) * N + col;
        if (in_batch) {
          *(float4*)to = (float4){v[0], v[1], v[2], v[3]};
          *(float4*)(to + 4) = (float4){v[4], v[5], v[6], v[7]};
        }
        if (l < depth) {
#pragma unroll
          for (int j = 0; j < 8; j++) v[j] = v[j] * sigmoid(v[j]);
          const uint4 p = {pair(v[0], v[1]), pair(v[2], v[3]), pair(v[4], v[5]), pair(v[6], v[7])};
          *(uint4*)(next + row * ld + col) = p;
          if (in_batch) *(uint4*)(h + (m0 + row) * N + col) = p;
        }
      }
    }
    __syncthreads();
    u16* const swap = cur;
    cur = next;
    next = swap;
    w16 += (long)N * K + N;
    w32 += (long)N * K + N;
    K = N;
  }
}

// One layer back: g = (cur W) · SiLU'(z) for 64 states, W [K][width] row-major, into next (unless the last) and out. W is
// read along its rows, 128 bytes per 16 lanes and four rows a lane, and the 4×4 values transposed in registers: tile t of a
// wave's 64 columns takes columns 4c + t, and a lane ends with 16 consecutive columns (row 4Q + r of tile t is column
// 16Q + 4r + t). A wave computes 32 states × 64 columns. z is requested before the products. 12 us per layer of 256 × 256
// for 2^14 states (25 MB), where mlp_gemm took 30.
__device__ __forceinline__ void layer_back(const u16* __restrict__ cur, u16* __restrict__ next, int ld, const u16* __restrict__ W, int K,
                                           int width, const float* __restrict__ z, u16* __restrict__ out, long m0, long n) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, c = lane & 15, q = lane >> 4, rows = (wave & 1) * 32;
  for (int nb = (wave >> 1) * 64; nb < width; nb += 256) {
    const u16* from = W + (long)(4 * q) * width + nb + 4 * c;
    uint2 w[4][4], ahead[4][4];  // [16 k][row 4q + r]
    f32x4 acc[2][4], zv[2][4];
#pragma unroll
    for (int i = 0; i < 4; i++)
#pragma unroll
      for (int r = 0; r < 4; r++) ahead[i][r] = *(const uint2*)(from + (long)(16 * i + r) * width);
#pragma unroll
    for (int i = 0; i < 2; i++) {
      const long m = m0 + rows + 16 * i + c;
#pragma unroll
      for (int r = 0; r < 4; r++) {
        acc[i][r] = (f32x4){0.f, 0.f, 0.f, 0.f};
        zv[i][r] = m < n ? *(const f32x4*)(z + m * width + nb + 16 * q + 4 * r) : (f32x4){0.f, 0.f, 0.f, 0.f};
      }
    }
    for (int k0 = 0; k0 < K; k0 += 64) {
#pragma unroll
      for (int i = 0; i < 4; i++)
#pragma unroll
        for (int r = 0; r < 4; r++) {
          w[i][r] = ahead[i][r];
          if (k0 + 64 < K) ahead[i][r] = *(const uint2*)(from + (long)(k0 + 64 + 16 * i + r) * width);
        }
#pragma unroll
      for (int kk = 0; kk < 4; kk++) {
        bf16x4 a[2];
#pragma unroll
        for (int i = 0; i < 2; i++) a[i] = *(const bf16x4*)(cur + (rows + 16 * i + c) * ld + k0 + 16 * kk + 4 * q);
#pragma unroll
        for (int t = 0; t < 4; t++) {
          const unsigned sel = t & 1 ? 0x07060302u : 0x05040100u;
          uint2 p;
          p.x = t < 2 ? __builtin_amdgcn_perm(w[kk][1].x, w[kk][0].x, sel) : __builtin_amdgcn_perm(w[kk][1].y, w[kk][0].y, sel);
          p.y = t < 2 ? __builtin_amdgcn_perm(w[kk][3].x, w[kk][2].x, sel) : __builtin_amdgcn_perm(w[kk][3].y, w[kk][2].y, sel);
          const bf16x4 b = __builtin_bit_cast(bf16x4, p);
#pragma unroll
          for (int i = 0; i < 2; i++) acc[i][t] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(b, a[i], acc[i][t], 0, 0, 0);
        }
      }
    }
#pragma unroll
    for (int i = 0; i < 2; i++) {
      const int row = rows + 16 * i + c, col = nb + 16 * q;
      float v[16];
#pragma unroll
      for (int r = 0; r < 4; r++)
#pragma unroll
        for (int t = 0; t < 4; t++) v[4 * r + t] = silu_derivative_times(acc[i][t][r], zv[i][r][t]);
#pragma unroll
      for (int j = 0; j < 2; j++) {
        const uint4 p = {pair(v[8 * j], v[8 * j + 1]), pair(v[8 * j + 2], v[8 * j + 3]), pair(v[8 * j + 4], v[8 * j + 5]),
                         pair(v[8 * j + 6], v[8 * j + 7])};
        if (next) *(uint4*)(next + row * ld + col + 8 * j) = p;
        if (m0 + row < n) *(uint4*)(out + (m0 + row) * width + col + 8 * j) = p;
      }
    }
  }
}

// The gradients by the pre-activations of layer `hi` (into ghi) and, unless it is layer 0, of layer hi - 1 (into glo), for
// 64 states a block. The output layer's comes from the loss, mean((y - target)²) over the first `valid` outputs (zero on
// padding); the others from the layer above, which glo holds from the launch before (a block reads and later writes its own
// 64 rows). wabove and whi are the weights of layers hi + 1 and hi, zhi and zlo the pre-activations.
extern "C" __global__ void __launch_bounds__(512)
mlp_backward(const float* __restrict__ y, const float* __restrict__ target, long n, int out, int valid, int from_loss, int width,
             const u16* __restrict__ wabove, const u16* __restrict__ whi, const float* __restrict__ zhi, const float* __restrict__ zlo,
             u16* ghi, u16* glo, int ld) {
  extern __shared__ __attribute__((aligned(16))) u16 act[];
  const long m0 = (long)blockIdx.x * ROWS;
  u16 *cur = act, *next = act + ROWS * ld;
  int K = out;
  if (from_loss) {
    const int quads = out >> 2;
    const float count = (float)(n * (long)valid);
    for (int i = threadIdx.x; i < ROWS * quads; i += 512) {
      const int row = i / quads, col = (i - row * quads) * 4;
      uint2 v = {0u, 0u};
      if (m0 + row < n) {
        const float4 a = *(const float4*)(y + (m0 + row) * out + col), b = *(const float4*)(target + (m0 + row) * out + col);
        const float f[4] = {col < valid ? 2.f * (a.x - b.x) / count : 0.f, col + 1 < valid ? 2.f * (a.y - b.y) / count : 0.f,
                            col + 2 < valid ? 2.f * (a.z - b.z) / count : 0.f, col + 3 < valid ? 2.f * (a.w - b.w) / count : 0.f};
        v = {pair(f[0], f[1]), pair(f[2], f[3])};
        *(uint2*)(ghi + (m0 + row) * out + col) = v;
      }
      *(uint2*)(cur + row * ld + col) = v;
    }
    __syncthreads();
  } else {
    K = width;
    const int octets = width >> 3;
    for (int i = threadIdx.x; i < ROWS * octets; i += 512) {
      const int row = i / octets, col = (i - row * octets) * 8;
      uint4 v = {0u, 0u, 0u, 0u};
      if (m0 + row < n) v = *(const uint4*)(glo + (m0 + row) * width + col);
      *(uint4*)(cur + row * ld + col) = v;
    }
    __syncthreads();
    layer_back(cur, zlo ? next : nullptr, ld, wabove, K, width, zhi, ghi, m0, n);
    __syncthreads();
    u16* const swap = cur;
    cur = next;
    next = swap;
  }
  if (zlo) layer_back(cur, nullptr, ld, whi, K, width, zlo, glo, m0, n);
}

// Reads 4 states × 4 columns of a row-major BF16 matrix, zero from state `end` on.
__device__ __forceinline__ void read_4x4(uint2 (&v)[4], const u16* __restrict__ src, long ld, long s, long end) {
#pragma unroll
  for (int r = 0; r < 4; r++) v[r] = s + r < end ? *(const uint2*)(src + (s + r) * ld) : (uint2){0u, 0u};
}

#define WK 72  // 64 states plus 8 of padding per column: 16 columns of a fragment read use all 64 banks
// ... and writes them transposed: four states of a column are one fragment.
__device__ __forceinline__ void write_4x4(u16 (*dst)[WK], const uint2 (&v)[4], int col, int s) {
#pragma unroll
  for (int t = 0; t < 4; t++) {
    const unsigned sel = t & 1 ? 0x07060302u : 0x05040100u;
    uint2 p;
    p.x = t < 2 ? __builtin_amdgcn_perm(v[1].x, v[0].x, sel) : __builtin_amdgcn_perm(v[1].y, v[0].y, sel);
    p.y = t < 2 ? __builtin_amdgcn_perm(v[3].x, v[2].x, sel) : __builtin_amdgcn_perm(v[3].y, v[2].y, sel);
    *(uint2*)&dst[col + t][s] = p;
  }
}

// Weight gradients of two layers, dW[o][i] = Σ_states g[o] h[i], and their bias gradients Σ_states g[o]: a block takes a
// 64×64 tile of one layer over one of `parts` ranges of states; its four groups of four waves (each wave a 32×32 quarter)
// take 64 states each at a time, the next in flight, and their sums are added in order at the end. (One group: 21 us for two
// layers at 2^14 states, bound by the latency of the loads; four: 18. Layer by layer with mlp_gemm and the column sums: 60.) Both operands have the states as their slow index; they are transposed 4×4 in registers on the way
// to LDS. The tiles of a layer's first columns also take the bias sums, as products with ones. Ranges are interleaved over
// consecutive blocks, so that the tiles of a range mostly share an XCD's L2. `to` is laid out as the parameters from the
// lower layer's weights on, one copy of `size` values per range.
#define GROUPS 4
struct MlpLayerGradient {
  const u16 *g, *h;
  int rows, cols;   // outputs and inputs of the layer
  long w, b;        // offsets of its weights and biases in `to`
};
extern "C" __global__ void __launch_bounds__(1024)
mlp_weights(MlpLayerGradient hi, MlpLayerGradient lo, long n, int parts, long range, float* __restrict__ to, long size) {
  __shared__ __attribute__((aligned(16))) u16 tiles[GROUPS][2][64][WK];
  const int group = threadIdx.x >> 8;
  u16 (*const G)[WK] = tiles[group][0], (*const H)[WK] = tiles[group][1];
  const int part = blockIdx.x % parts;
  int tile = blockIdx.x / parts;
  const int hi_tiles = (hi.rows >> 6) * (hi.cols >> 6);
  const bool second = tile >= hi_tiles;
  if (second) tile -= hi_tiles;
  const u16 *g = second ? lo.g : hi.g, *h = second ? lo.h : hi.h;
  const int rows = second ? lo.rows : hi.rows, cols = second ? lo.cols : hi.cols;
  const int across = cols >> 6, o0 = tile / across * 64, i0 = tile % across * 64;
  const int lane = threadIdx.x & 63, wave = (threadIdx.x >> 6) & 3, c = lane & 15, q = lane >> 4, wo = (wave >> 1) * 32, wi = (wave & 1) * 32;
  const bool bias = i0 == 0 && wi == 0;
  const long begin = part * range, end = begin + range < n ? begin + range : n;
  // 16 × 16 groups of 4 × 4 (columns, states): a wave reads 8 × 8 of them, 64 bytes of a row at a time
  const int col = ((wave & 1) * 8 + (lane & 7)) * 4, st = ((wave >> 1) * 8 + (lane >> 3)) * 4;
  const u16 *gp = g + o0 + col, *hp = h + i0 + col;
  f32x4 acc[2][2], sums[2];
#pragma unroll
  for (int i = 0; i < 2; i++) {
    sums[i] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int j = 0; j < 2; j++) acc[i][j] = (f32x4){0.f, 0.f, 0.f, 0.f};
  }
  const short one = 0x3F80;
  const bf16x4 ones = {one, one, one, one};
  uint2 gv[4], hv[4];
  read_4x4(gv, gp, rows, begin + 64 * group + st, end);
  read_4x4(hv, hp, cols, begin + 64 * group + st, end);
  for (long s = begin; s < end; s += 64 * GROUPS) {
    write_4x4(G, gv, col, st);
    write_4x4(H, hv, col, st);
    __syncthreads();
    if (s + 64 * GROUPS < end) {
      read_4x4(gv, gp, rows, s + 64 * (GROUPS + group) + st, end);
      read_4x4(hv, hp, cols, s + 64 * (GROUPS + group) + st, end);
    }
#pragma unroll
    for (int k = 0; k < 64; k += 16) {
      bf16x4 a[2], b[2];
#pragma unroll
      for (int i = 0; i < 2; i++) {
        a[i] = *(const bf16x4*)&G[wo + 16 * i + c][k + 4 * q];
        b[i] = *(const bf16x4*)&H[wi + 16 * i + c][k + 4 * q];
      }
#pragma unroll
      for (int i = 0; i < 2; i++) {
#pragma unroll
        for (int j = 0; j < 2; j++) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a[i], b[j], acc[i][j], 0, 0, 0);
        if (bias) sums[i] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a[i], ones, sums[i], 0, 0, 0);
      }
    }
    __syncthreads();
  }
  // the groups' sums in order: 4096 products and 64 bias sums each
  float* const sum = (float*)tiles;
  float* const mine = sum + group * (4096 + 64);
#pragma unroll
  for (int i = 0; i < 2; i++)
#pragma unroll
    for (int r = 0; r < 4; r++) {
      const int o = wo + 16 * i + 4 * q + r;
#pragma unroll
      for (int j = 0; j < 2; j++) mine[o * 64 + wi + 16 * j + c] = acc[i][j][r];
      if (bias && c == 0) mine[4096 + o] = sums[i][r];
    }
  __syncthreads();
  float* w = to + part * size + (second ? lo.w : hi.w);
  float* b = to + part * size + (second ? lo.b : hi.b);
  for (int e = threadIdx.x; e < 4096 + (i0 == 0 ? 64 : 0); e += 64 * 4 * GROUPS) {
    float v = sum[e];
#pragma unroll
    for (int k = 1; k < GROUPS; k++) v += sum[k * (4096 + 64) + e];
    if (e < 4096)
      w[(long)(o0 + (e >> 6)) * cols + i0 + (e & 63)] = v;
    else
      b[o0 + e - 4096] = v;
  }
}

// Loads rows [r0, r0+64) × k [k0, k0+32) of a strided BF16 matrix into dst[row][k], zero outside [0, R) × [klo, khi).
__device__ __forceinline__ void load_tile(u16 (*dst)[LDSK], const u16* __restrict__ src, long sr, long sk, long r0, long R,
                                          long k0, long klo, long khi) {
  const int t = threadIdx.x;
  if (sk == 1) {
    const int row = t >> 2, kc = (t & 3) * 8;
    const long r = r0 + row, k = k0 + kc;
    u16 v[8];
    if (r < R && k >= klo && k + 8 <= khi) {
      const uint4 q = *(const uint4*)(src + r * sr + k);
      __builtin_memcpy(v, &q, 16);
    } else {
      for (int i = 0; i < 8; i++) v[i] = (r < R && k + i >= klo && k + i < khi) ? src[r * sr + k + i] : (u16)0;
    }
    for (int i = 0; i < 8; i++) dst[row][kc + i] = v[i];
  } else {  // sr == 1: 8 consecutive rows at one k
    const int kc = t >> 3, row = (t & 7) * 8;
    const long k = k0 + kc, r = r0 + row;
    u16 v[8];
    if (k >= klo && k < khi && r + 8 <= R) {
      const uint4 q = *(const uint4*)(src + r + k * sk);
      __builtin_memcpy(v, &q, 16);
    } else {
      for (int i = 0; i < 8; i++) v[i] = (k >= klo && k < khi && r + i < R) ? src[r + i + k * sk] : (u16)0;
    }
    for (int i = 0; i < 8; i++) dst[row + i][kc] = v[i];
  }
}

// 64×64 output tiles per 256-thread block (each wave a 32×32 quarter), k in steps of 32 staged through LDS. One kernel
// serves the forward product, the backward data product and the weight gradient: C[m][n] = Σ_k A(m, k) B(n, k), with
// A(m, k) = A[m sam + k sak] and B(n, k) = B[n sbn + k sbk], so transposed operands are strides, and the epilogue is chosen
// by `mode`:
//   0  hidden layer forward: z = C + bias[n] (FP32 out) and h = SiLU(z) (BF16 out)
//   1  output layer forward: z = C + bias[n] (FP32 out)
//   2  backward data: g = C · SiLU'(zprev[m][n]) (BF16 out), the previous layer's pre-activation gradient
//   3  weight gradient: C over the k range [kz·kchunk, (kz+1)·kchunk) of blockIdx.z, FP32 out into partial[kz][m][n]
// M is guarded.
extern "C" __global__ void __launch_bounds__(256)
mlp_gemm(int mode, long M, long N, long Kd, const u16* __restrict__ A, long sam, long sak, const u16* __restrict__ B, long sbn,
         long sbk, const float* __restrict__ bias, const float* __restrict__ zprev, float* __restrict__ zout,
         u16* __restrict__ hout, long ldc, float* __restrict__ partial, long kchunk) {
  __shared__ u16 As[64][LDSK], Bs[64][LDSK];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int wm = wave >> 1, wn = wave & 1;
  const long m0 = (long)blockIdx.x * 64, n0 = (long)blockIdx.y * 64;
  long klo = 0, khi = Kd;
  if (mode == 3) {
    klo = (long)blockIdx.z * kchunk;
    khi = klo + kchunk < Kd ? klo + kchunk : Kd;
  }
  f32x4 acc[2][2];
  for (int i = 0; i < 2; i++)
    for (int j = 0; j < 2; j++) acc[i][j] = (f32x4){0.f, 0.f, 0.f, 0.f};
  for (long k0 = klo & ~31L; k0 < khi; k0 += 32) {
    load_tile(As, A, sam, sak, m0, M, k0, klo, khi);
    load_tile(Bs, B, sbn, sbk, n0, N, k0, klo, khi);
    __syncthreads();
    for (int kk = 0; kk < 32; kk += 16) {
      bf16x4 a[2], b[2];
      for (int i = 0; i < 2; i++) a[i] = *(const bf16x4*)&As[wm * 32 + i * 16 + (lane & 15)][kk + 4 * (lane >> 4)];
      for (int j = 0; j < 2; j++) b[j] = *(const bf16x4*)&Bs[wn * 32 + j * 16 + (lane & 15)][kk + 4 * (lane >> 4)];
      for (int i = 0; i < 2; i++)
        for (int j = 0; j < 2; j++) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a[i], b[j], acc[i][j], 0, 0, 0);
    }
    __syncthreads();
  }
  for (int i = 0; i < 2; i++)
    for (int j = 0; j < 2; j++)
      for (int r = 0; r < 4; r++) {
        const long m = m0 + wm * 32 + i * 16 + 4 * (lane >> 4) + r, n = n0 + wn * 32 + j * 16 + (lane & 15);
        if (m >= M || n >= N) continue;
        const float c = acc[i][j][r];
        if (mode == 0) {
          const float z = c + bias[n];
          zout[m * ldc + n] = z;
          hout[m * ldc + n] = to_bf16(z * sigmoid(z));
        } else if (mode == 1) {
          zout[m * ldc + n] = c + bias[n];
        } else if (mode == 2) {
          const float z = zprev[m * ldc + n], s = sigmoid(z);
          hout[m * ldc + n] = to_bf16(c * s * (1.f + z * (1.f - s)));
        } else {
          partial[((long)blockIdx.z * M + m) * N + n] = c;
        }
      }
}

// out[i] = Σ_z partial[z][i] (z in order: deterministic).
extern "C" __global__ void mlp_reduce(const float* __restrict__ partial, long n, int parts, float* __restrict__ out) {
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  float s = 0.f;
  for (int z = 0; z < parts; z++) s += partial[(long)z * n + i];
  out[i] = s;
}

// Partial column sums of dz (BF16 gradients, FP32 sums) over the row chunk [z·chunk, (z+1)·chunk) of blockIdx.z:
// a 256-thread block takes 64 columns (the lane) and 4 interleaved row streams (the wave), combined in LDS in wave
// order, into partial[z][c]; mlp_reduce then adds the chunks in order (a fixed summation order for every run).
extern "C" __global__ void __launch_bounds__(256)
mlp_column_sum(const u16* __restrict__ dz, long M, long ld, long cols, long chunk, float* __restrict__ partial) {
  __shared__ float part[4][64];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const long c = (long)blockIdx.x * 64 + lane;
  const long m0 = (long)blockIdx.z * chunk, m1 = m0 + chunk < M ? m0 + chunk : M;
  float s = 0.f;
  if (c < cols)
#pragma unroll 8
    for (long m = m0 + wave; m < m1; m += 4) s += from_bf16(dz[m * ld + c]);
  part[wave][lane] = s;
  __syncthreads();
  if (wave == 0 && c < cols) partial[(long)blockIdx.z * cols + c] = ((part[0][lane] + part[1][lane]) + part[2][lane]) + part[3][lane];
}

// x (FP32) -> BF16, elementwise.
extern "C" __global__ void mlp_to_bf16(const float* __restrict__ x, long n, u16* __restrict__ out) {
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) out[i] = to_bf16(x[i]);
}

// Mean squared error over the first `valid` of ld outputs: dz = 2 (y - t) / (M valid) as BF16 (zero on padding).
extern "C" __global__ void mlp_mse_grad(const float* __restrict__ y, const float* __restrict__ t, long M, long ld, long valid,
                                        u16* __restrict__ dz) {
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= M * ld) return;
  const long c = i % ld;
  dz[i] = c < valid ? to_bf16(2.f * (y[i] - t[i]) / (float)(M * valid)) : (u16)0;
}

// Adam (Kingma & Ba 2015) on FP32 master parameters, refreshing their BF16 copies.
extern "C" __global__ void mlp_adam(float* __restrict__ p, u16* __restrict__ p16, const float* __restrict__ g, float* __restrict__ m1,
                                    float* __restrict__ m2, long n, float lr, float beta1, float beta2, float eps, float c1,
                                    float c2) {
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const float gi = g[i];
  const float a = beta1 * m1[i] + (1.f - beta1) * gi;
  const float b = beta2 * m2[i] + (1.f - beta2) * gi * gi;
  m1[i] = a;
  m2[i] = b;
  const float q = p[i] - lr * (a / c1) / (__builtin_sqrtf(b / c2) + eps);
  p[i] = q;
  p16[i] = to_bf16(q);
}
