// The potential surrogate: an MLP of 6 symmetry-adapted features -> 128 -> 128 -> 128 -> 1 with SiLU, trained and
// evaluated on the device. The two 128 x 128 hidden layers run on the matrix cores (v_mfma_f32_16x16x16_bf16:
// operands rounded to bf16, round to nearest even, products accumulated in FP32) in the forward pass and in both
// backward products (dW = A^T dZ, dA = dZ W^T); the 6 -> 128 input and 128 -> 1 output layers, the SiLU, the loss
// and Adam run in FP32 on the vector units. Rows are processed in tiles of 16 (the row count is a multiple of 16).
//
// A training step is two kernels. mlp_pass_kernel takes 16 rows through all layers, forward and back, with the
// activations in registers and their bf16 operands in LDS, and leaves what the gradient sums over the rows; every
// value is stored in the matrix cores' result layout (fragments of 16 rows x 16 units, lane l holding the rows
// 4 (l / 16) + 0 .. 3 of unit l % 16), which is the operand layout of the product A^T dZ, so nothing is transposed.
// mlp_update_kernel gives each 16 x 16 tile of a hidden layer's weights one wavefront, which runs its products over
// all rows in order and applies Adam to its tile, and each column of the other parameters one thread group. The
// weights are kept a second time as bf16 fragments, so that the passes read their operands as they are.
// A step of 4096 rows is 0.8 GFLOP, under a microsecond of matrix-core time: what it costs is launches and latency.
// As 16 kernels with the activations going through HBM it took 310 us on MI355X, of which the weight products (64
// wavefronts, four strided loads per operand) and the strided column sums were most; as two it takes 68 us.
#pragma once

#include <hip/hip_runtime.h>

namespace spo_dev {

constexpr int kMlpIn = 6;
constexpr int kMlpWidth = 128;
// Offsets of the parameter vector: W1 (6 x 128, row k), b1, W2 (128 x 128), b2, W3, b3, W4 (128), b4
constexpr int kMlpW1 = 0;
constexpr int kMlpB1 = kMlpW1 + kMlpIn * kMlpWidth;
constexpr int kMlpW2 = kMlpB1 + kMlpWidth;
constexpr int kMlpB2 = kMlpW2 + kMlpWidth * kMlpWidth;
constexpr int kMlpW3 = kMlpB2 + kMlpWidth;
constexpr int kMlpB3 = kMlpW3 + kMlpWidth * kMlpWidth;
constexpr int kMlpW4 = kMlpB3 + kMlpWidth;
constexpr int kMlpB4 = kMlpW4 + kMlpWidth;
constexpr int kMlpParams = kMlpB4 + 1;

constexpr int kMlpRows = 16;                 // rows of a tile
constexpr int kMlpTiles = kMlpWidth / 16;    // 16-unit tiles of a layer
constexpr int kMlpFragment = 64 * 4;         // values of a 16 x 16 fragment
// bf16 weight fragments [layer][direction][column tile][k step]: forward (B = W) and backward (B = W^T).
constexpr int kMlpWeightFragments = kMlpTiles * kMlpTiles * kMlpFragment;
constexpr int kMlpFragments = 4 * kMlpWeightFragments;

typedef short mlp_bf16x4 __attribute__((ext_vector_type(4)));
typedef float mlp_f32x4 __attribute__((ext_vector_type(4)));

__device__ inline short mlp_bf16(float f) {  // round to nearest even (finite inputs)
  unsigned u = __float_as_uint(f);
  u += 0x7FFFu + ((u >> 16) & 1u);
  return static_cast<short>(u >> 16);
}

__device__ inline float mlp_sigmoid(float z) { return 1.0f / (1.0f + __expf(-z)); }
__device__ inline float mlp_silu(float z) { return z * mlp_sigmoid(z); }
__device__ inline float mlp_silu_slope(float z) {
  const float s = mlp_sigmoid(z);
  return s * (1.0f + z * (1.0f - s));
}

// Writes weight (k, j) of hidden layer `layer` (0, 1) into its two fragments.
__device__ inline void mlp_put_weight(short* frag, int layer, int k, int j, float value) {
  short* f = frag + layer * 2 * kMlpWeightFragments;
  const short b = mlp_bf16(value);
  f[((j / 16) * kMlpTiles + k / 16) * kMlpFragment + ((k % 16) / 4 * 16 + j % 16) * 4 + k % 4] = b;
  f += kMlpWeightFragments;
  f[((k / 16) * kMlpTiles + j / 16) * kMlpFragment + ((j % 16) / 4 * 16 + k % 16) * 4 + j % 4] = b;
}

// The fragments of a whole parameter vector; one thread per weight of W2 and W3.
__global__ inline __launch_bounds__(256) void mlp_fragment_kernel(const float* p, short* frag) {
  const int e = blockIdx.x * 256 + threadIdx.x;
  if (e >= 2 * kMlpWidth * kMlpWidth) return;
  const int layer = e / (kMlpWidth * kMlpWidth), i = e % (kMlpWidth * kMlpWidth);
  mlp_put_weight(frag, layer, i / kMlpWidth, i % kMlpWidth, p[(layer ? kMlpW3 : kMlpW2) + i]);
}

// ---- one tile of 16 rows; four wavefronts, wavefront w owning the units 32 w + 16 tj + lane % 16 (tj = 0, 1) and in
// each of them the rows 4 (lane / 16) + v ------------------------------------------------------------------------
constexpr int kMlpLd = kMlpWidth + 8;  // operand rows in LDS: 16 lanes' reads at one k fall on distinct banks

struct MlpTile {
  float v[2][4];  // [tj][v]
};
__device__ inline int mlp_unit(int tj) { return 32 * (threadIdx.x / 64) + 16 * tj + threadIdx.x % 16; }
__device__ inline int mlp_row(int v) { return 4 * (threadIdx.x % 64 / 16) + v; }

// The wavefront's weight fragments of one layer (0, 1) and direction (0 forward, 1 backward).
struct MlpWeights {
  mlp_bf16x4 f[2][kMlpTiles];
};
__device__ inline MlpWeights mlp_weights(const short* frag, int layer, int backward) {
  MlpWeights out;
  const short* f = frag + (2 * layer + backward) * kMlpWeightFragments + 4 * (threadIdx.x % 64);
#pragma unroll
  for (int tj = 0; tj < 2; ++tj)
#pragma unroll
    for (int k = 0; k < kMlpTiles; ++k)
      out.f[tj][k] = *reinterpret_cast<const mlp_bf16x4*>(
          f + ((2 * (threadIdx.x / 64) + tj) * kMlpTiles + k) * kMlpFragment);
  return out;
}

// The rows of `left` (bf16, LDS) times the weights.
__device__ inline MlpTile mlp_product(const short* left, const MlpWeights& w) {
  const int lane = threadIdx.x % 64;
  mlp_f32x4 acc[2] = {};
#pragma unroll
  for (int k = 0; k < kMlpTiles; ++k) {
    const mlp_bf16x4 a = *reinterpret_cast<const mlp_bf16x4*>(left + (lane % 16) * kMlpLd + 16 * k + 4 * (lane / 16));
#pragma unroll
    for (int tj = 0; tj < 2; ++tj) acc[tj] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, w.f[tj][k], acc[tj], 0, 0, 0);
  }
  MlpTile out;
#pragma unroll
  for (int tj = 0; tj < 2; ++tj)
#pragma unroll
    for (int v = 0; v < 4; ++v) out.v[tj][v] = acc[tj][v];
  return out;
}

// A tile's values as the left operand of the next product, and (fragments not NULL) as the tile's fragments.
__device__ inline void mlp_store_operand(const MlpTile& a, short* rows, short* fragments) {
#pragma unroll
  for (int tj = 0; tj < 2; ++tj) {
    mlp_bf16x4 b;
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      b[v] = mlp_bf16(a.v[tj][v]);
      rows[mlp_row(v) * kMlpLd + mlp_unit(tj)] = b[v];
    }
    if (fragments)
      *reinterpret_cast<mlp_bf16x4*>(fragments + (2 * (threadIdx.x / 64) + tj) * kMlpFragment + 4 * (threadIdx.x % 64)) = b;
  }
}
__device__ inline void mlp_store_fragments(const MlpTile& a, float* fragments) {
#pragma unroll
  for (int tj = 0; tj < 2; ++tj)
    *reinterpret_cast<mlp_f32x4*>(fragments + (2 * (threadIdx.x / 64) + tj) * kMlpFragment + 4 * (threadIdx.x % 64)) =
        mlp_f32x4{a.v[tj][0], a.v[tj][1], a.v[tj][2], a.v[tj][3]};
}

// z1 = x W1 + b1 (xs: [row][6] in LDS)
__device__ inline MlpTile mlp_input_layer(const float* xs, const float* p) {
  MlpTile z;
#pragma unroll
  for (int tj = 0; tj < 2; ++tj) {
    const int n = mlp_unit(tj);
    float w[kMlpIn];
#pragma unroll
    for (int k = 0; k < kMlpIn; ++k) w[k] = p[kMlpW1 + k * kMlpWidth + n];
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      float s = p[kMlpB1 + n];
#pragma unroll
      for (int k = 0; k < kMlpIn; ++k) s += xs[mlp_row(v) * kMlpIn + k] * w[k];
      z.v[tj][v] = s;
    }
  }
  return z;
}

__device__ inline MlpTile mlp_hidden_layer(const short* left, const MlpWeights& w, const float* bias) {
  MlpTile z = mlp_product(left, w);
#pragma unroll
  for (int tj = 0; tj < 2; ++tj)
#pragma unroll
    for (int v = 0; v < 4; ++v) z.v[tj][v] = z.v[tj][v] + bias[mlp_unit(tj)];
  return z;
}

__device__ inline MlpTile mlp_silu_tile(const MlpTile& z) {
  MlpTile a;
#pragma unroll
  for (int tj = 0; tj < 2; ++tj)
#pragma unroll
    for (int v = 0; v < 4; ++v) a.v[tj][v] = mlp_silu(z.v[tj][v]);
  return a;
}

// y = a3 W4 + b4 of row threadIdx.x < 16 (act: [row][129] in LDS), summed in the units' order.
constexpr int kMlpLdOut = kMlpWidth + 1;
__device__ inline void mlp_park_output(const MlpTile& a, float* act) {
#pragma unroll
  for (int tj = 0; tj < 2; ++tj)
#pragma unroll
    for (int v = 0; v < 4; ++v) act[mlp_row(v) * kMlpLdOut + mlp_unit(tj)] = a.v[tj][v];
}
__device__ inline float mlp_output_layer(const float* act, const float* p) {
  float s = p[kMlpB4];
#pragma unroll 16
  for (int n = 0; n < kMlpWidth; ++n) s += act[threadIdx.x * kMlpLdOut + n] * p[kMlpW4 + n];
  return s;
}

// y of `rows` rows (any count). The wavefronts keep their weights in registers over the tiles of a workgroup.
__global__ inline __launch_bounds__(256) void mlp_predict_kernel(const float* x, const float* p, const short* frag,
                                                                 long rows, float* y) {
  __shared__ __align__(16) short left[2][kMlpRows * kMlpLd];
  __shared__ float act[kMlpRows * kMlpLdOut];
  __shared__ float xs[kMlpRows * kMlpIn];
  const int tid = threadIdx.x;
  const MlpWeights w2 = mlp_weights(frag, 0, 0), w3 = mlp_weights(frag, 1, 0);
  const long tiles = (rows + kMlpRows - 1) / kMlpRows;
  for (long tile = blockIdx.x; tile < tiles; tile += gridDim.x) {
    const long row0 = tile * kMlpRows;
    const int n = static_cast<int>(rows - row0 < kMlpRows ? rows - row0 : kMlpRows);
    if (tid < kMlpRows * kMlpIn) xs[tid] = tid < n * kMlpIn ? x[row0 * kMlpIn + tid] : 0.0f;
    __syncthreads();
    mlp_store_operand(mlp_silu_tile(mlp_input_layer(xs, p)), left[0], nullptr);
    __syncthreads();
    mlp_store_operand(mlp_silu_tile(mlp_hidden_layer(left[0], w2, p + kMlpB2)), left[1], nullptr);
    __syncthreads();
    mlp_park_output(mlp_silu_tile(mlp_hidden_layer(left[1], w3, p + kMlpB3)), act);
    __syncthreads();
    if (tid < n) y[row0 + tid] = mlp_output_layer(act, p);
  }
}

// What a training pass leaves for the gradient's sums over the rows, [row tile][unit tile][64][4]: bf16 operands and
// FP32 values, and per row the error d = y - t and dL/dy.
struct MlpTape {
  short* a1;
  short* a2;
  short* dz2;
  short* dz3;
  float* dz1_f;
  float* dz2_f;
  float* dz3_f;
  float* a3_f;
  float* d;
  float* dy;
};

// Forward and backward of the mean squared error over `rows` rows; one workgroup per tile.
__global__ inline __launch_bounds__(256) void mlp_pass_kernel(const float* x, const float* t, long rows, const float* p,
                                                              const short* frag, MlpTape tape) {
  __shared__ __align__(16) short left[2][kMlpRows * kMlpLd];
  __shared__ float act[kMlpRows * kMlpLdOut];
  __shared__ float xs[kMlpRows * kMlpIn];
  __shared__ float dys[kMlpRows];
  const int tid = threadIdx.x;
  const long row0 = static_cast<long>(blockIdx.x) * kMlpRows;
  const long at = static_cast<long>(blockIdx.x) * kMlpTiles * kMlpFragment;
  if (tid < kMlpRows * kMlpIn) xs[tid] = x[row0 * kMlpIn + tid];
  const MlpWeights w2 = mlp_weights(frag, 0, 0), w3 = mlp_weights(frag, 1, 0);
  __syncthreads();
  const MlpTile z1 = mlp_input_layer(xs, p);
  mlp_store_operand(mlp_silu_tile(z1), left[0], tape.a1 + at);
  __syncthreads();
  const MlpTile z2 = mlp_hidden_layer(left[0], w2, p + kMlpB2);
  mlp_store_operand(mlp_silu_tile(z2), left[1], tape.a2 + at);
  __syncthreads();
  const MlpTile z3 = mlp_hidden_layer(left[1], w3, p + kMlpB3);
  const MlpTile a3 = mlp_silu_tile(z3);
  mlp_park_output(a3, act);
  mlp_store_fragments(a3, tape.a3_f + at);
  const MlpWeights b3 = mlp_weights(frag, 1, 1), b2 = mlp_weights(frag, 0, 1);
  __syncthreads();
  if (tid < kMlpRows) {
    const float d = mlp_output_layer(act, p) - t[row0 + tid];
    const float dy = 2.0f * d / static_cast<float>(rows);
    dys[tid] = dy;
    tape.d[row0 + tid] = d;
    tape.dy[row0 + tid] = dy;
  }
  __syncthreads();
  // dZ3 = (dy W4^T) SiLU'(z3)
  MlpTile d;
#pragma unroll
  for (int tj = 0; tj < 2; ++tj)
#pragma unroll
    for (int v = 0; v < 4; ++v)
      d.v[tj][v] = dys[mlp_row(v)] * p[kMlpW4 + mlp_unit(tj)] * mlp_silu_slope(z3.v[tj][v]);
  mlp_store_fragments(d, tape.dz3_f + at);
  mlp_store_operand(d, left[0], tape.dz3 + at);
  __syncthreads();
  // dA2 = dZ3 W3^T, dZ2 = dA2 SiLU'(z2)
  d = mlp_product(left[0], b3);
#pragma unroll
  for (int tj = 0; tj < 2; ++tj)
#pragma unroll
    for (int v = 0; v < 4; ++v) d.v[tj][v] = d.v[tj][v] * mlp_silu_slope(z2.v[tj][v]);
  mlp_store_fragments(d, tape.dz2_f + at);
  mlp_store_operand(d, left[1], tape.dz2 + at);
  __syncthreads();
  // dA1 = dZ2 W2^T, dZ1 = dA1 SiLU'(z1)
  d = mlp_product(left[1], b2);
#pragma unroll
  for (int tj = 0; tj < 2; ++tj)
#pragma unroll
    for (int v = 0; v < 4; ++v) d.v[tj][v] = d.v[tj][v] * mlp_silu_slope(z1.v[tj][v]);
  mlp_store_fragments(d, tape.dz1_f + at);
}

// Where a gradient entry goes: into Adam (bias-corrected) or, with grad not NULL, there.
struct MlpAdam {
  float* p;
  float* m;
  float* v;
  float* grad;
  float lr, beta1, beta2, eps, c1, c2;
  // Returns the parameter after the update.
  __device__ inline float apply(int i, float gi) const {
    if (grad) {
      grad[i] = gi;
      return p[i];
    }
    const float mi = beta1 * m[i] + (1.0f - beta1) * gi, vi = beta2 * v[i] + (1.0f - beta2) * gi * gi;
    m[i] = mi;
    v[i] = vi;
    const float value = p[i] - lr * (mi / c1) / (sqrtf(vi / c2) + eps);
    p[i] = value;
    return value;
  }
};

// Sums over the rows of a column tile's fragments, as 256 interleaved running sums (rows r, r + 256, ...) added
// pairwise at distances 128, 64, ... 1. Thread (wavefront w, lane l) holds the running sums of the rows
// 16 (w + 4 s) + 4 (l / 16) + v of unit l % 16: the distances 128 and 64 are its own s, 32 and 16 go over the
// wavefronts, 8 and 4 over the lanes, 2 and 1 are its own v. Every lane of wavefront 0 returns its unit's sum.
__device__ inline float mlp_fold(float (&s)[4][4], float* shared) {
  const int lane = threadIdx.x % 64, w = threadIdx.x / 64;
  float a[4];
#pragma unroll
  for (int v = 0; v < 4; ++v) a[v] = (s[0][v] + s[2][v]) + (s[1][v] + s[3][v]);
  __syncthreads();  // the last use of `shared`
#pragma unroll
  for (int v = 0; v < 4; ++v) shared[(w * 64 + lane) * 4 + v] = a[v];
  __syncthreads();
  float out[4];
#pragma unroll
  for (int v = 0; v < 4; ++v) {
    const float* c = shared + lane * 4 + v;
    float b = (c[0] + c[512]) + (c[256] + c[768]);
    b += __shfl_xor(b, 32);
    b += __shfl_xor(b, 16);
    out[v] = b;
  }
  return (out[0] + out[2]) + (out[1] + out[3]);
}

// The gradient's sums over the rows and the update of every parameter; blocks:
//   0 .. 127: a 16 x 16 tile of W2 or W3 (one wavefront; products over the rows in order);
//   128 .. 135: W1 and b1 of one unit tile; 136 .. 143: b2; 144 .. 151: b3; 152 .. 159: W4 (152 also b4 and the loss).
constexpr int kMlpUpdateBlocks = 2 * kMlpTiles * kMlpTiles + 4 * kMlpTiles;
__global__ inline __launch_bounds__(256) void mlp_update_kernel(MlpAdam adam, short* frag, MlpTape tape, const float* x,
                                                                long rows, float* loss) {
  __shared__ float shared[1024];
  const int tid = threadIdx.x, lane = tid % 64, w = tid / 64;
  const int row_tiles = static_cast<int>(rows / kMlpRows);
  const int stride = kMlpTiles * kMlpFragment;  // values of a row tile
  int block = blockIdx.x;
  if (block < 2 * kMlpTiles * kMlpTiles) {
    if (w > 0) return;
    const int layer = block / (kMlpTiles * kMlpTiles), ti = block / kMlpTiles % kMlpTiles, tj = block % kMlpTiles;
    const mlp_bf16x4* a = reinterpret_cast<const mlp_bf16x4*>((layer ? tape.a2 : tape.a1) + ti * kMlpFragment) + lane;
    const mlp_bf16x4* b = reinterpret_cast<const mlp_bf16x4*>((layer ? tape.dz3 : tape.dz2) + tj * kMlpFragment) + lane;
    mlp_f32x4 acc = {};
    // The operands of the next DEPTH row tiles are in flight while these are multiplied.
    constexpr int DEPTH = 16;
    mlp_bf16x4 av[DEPTH], bv[DEPTH];
#pragma unroll
    for (int i = 0; i < DEPTH; ++i)
      if (i < row_tiles) {
        av[i] = a[static_cast<long>(i) * (stride / 4)];
        bv[i] = b[static_cast<long>(i) * (stride / 4)];
      }
    for (int r0 = 0; r0 < row_tiles; r0 += DEPTH) {
      mlp_bf16x4 an[DEPTH], bn[DEPTH];
#pragma unroll
      for (int i = 0; i < DEPTH; ++i)
        if (r0 + DEPTH + i < row_tiles) {
          an[i] = a[static_cast<long>(r0 + DEPTH + i) * (stride / 4)];
          bn[i] = b[static_cast<long>(r0 + DEPTH + i) * (stride / 4)];
        }
#pragma unroll
      for (int i = 0; i < DEPTH; ++i)
        if (r0 + i < row_tiles) acc = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(av[i], bv[i], acc, 0, 0, 0);
#pragma unroll
      for (int i = 0; i < DEPTH; ++i) {
        av[i] = an[i];
        bv[i] = bn[i];
      }
    }
    const int j = 16 * tj + lane % 16;
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      const int k = 16 * ti + 4 * (lane / 16) + c;
      const float value = adam.apply((layer ? kMlpW3 : kMlpW2) + k * kMlpWidth + j, acc[c]);
      if (!adam.grad) mlp_put_weight(frag, layer, k, j, value);
    }
    return;
  }
  block -= 2 * kMlpTiles * kMlpTiles;
  const int what = block / kMlpTiles, tj = block % kMlpTiles, unit = 16 * tj + lane % 16;
  const float* src = (what == 0 ? tape.dz1_f : what == 1 ? tape.dz2_f : what == 2 ? tape.dz3_f : tape.a3_f) +
                     tj * kMlpFragment + 4 * lane;
  float s[4][4] = {}, sx[kMlpIn][4][4] = {};
  for (int r0 = w; r0 < row_tiles; r0 += 16) {
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int r = r0 + 4 * q;
      if (r >= row_tiles) break;
      const mlp_f32x4 f = *reinterpret_cast<const mlp_f32x4*>(src + static_cast<long>(r) * stride);
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const long row = static_cast<long>(r) * kMlpRows + 4 * (lane / 16) + v;
        s[q][v] += f[v] * (what == 3 ? tape.dy[row] : 1.0f);
        if (what == 0) {
#pragma unroll
          for (int k = 0; k < kMlpIn; ++k) sx[k][q][v] += x[row * kMlpIn + k] * f[v];
        }
      }
    }
  }
  const float sum = mlp_fold(s, shared);
  const bool owner = tid < 16;
  if (owner) adam.apply((what == 0 ? kMlpB1 : what == 1 ? kMlpB2 : what == 2 ? kMlpB3 : kMlpW4) + unit, sum);
  if (what == 0) {
#pragma unroll
    for (int k = 0; k < kMlpIn; ++k) {
      const float g = mlp_fold(sx[k], shared);
      if (owner) adam.apply(kMlpW1 + k * kMlpWidth + unit, g);
    }
  }
  if (what == 3 && tj == 0) {  // b4 and the loss, over every lane's copy of its row (the units of a row agree)
    float sd[4][4] = {}, sl[4][4] = {};
    for (int r0 = w; r0 < row_tiles; r0 += 16) {
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int r = r0 + 4 * q;
        if (r >= row_tiles) break;
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          const long row = static_cast<long>(r) * kMlpRows + 4 * (lane / 16) + v;
          const float d = tape.d[row];
          sd[q][v] += tape.dy[row] * 1.0f;
          sl[q][v] += d * d;
        }
      }
    }
    const float g = mlp_fold(sd, shared), l = mlp_fold(sl, shared);
    if (tid == 0) {
      adam.apply(kMlpB4, g);
      if (loss) *loss = l / static_cast<float>(rows);
    }
  }
}

}  // namespace spo_dev
