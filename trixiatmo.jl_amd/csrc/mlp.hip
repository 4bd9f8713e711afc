// gfx950 kernels of the small MLP (3 -> 32 -> 32 -> 2, tanh, FP32) that seeds
// the rainy-Euler saturation solve: batched forward, loss and gradient, and
// Adam.
//
// A wave takes tiles of 16 samples, its weights in registers.  The hidden
// layers, their transposes and the weight gradients are products on the matrix
// cores (v_mfma_f32_16x16x4f32, FP32 throughout).  With g = lane / 16 and c =
// lane % 16 that instruction reads A[row c][k = g] and B[k = g][column c] and
// returns rows 4 g + r (r = 0..3) of column c.  Columns are samples: a lane
// holds neurons 16 T + 4 g + r (T = 0, 1) of sample c, and since a sum over k
// may run in any order, result register r of tile T is the next layer's B
// operand for the four neurons 16 T + 4 g + r as it stands.  The gradients sum
// over samples instead, so activations and deltas pass once through LDS to be
// read by sample.  Gradients stay in registers over all tiles of a wave; one
// partial per workgroup is written, and a second kernel sums the partials in a
// fixed order, so a gradient is bit-reproducible, and applies Adam.
//
// Measured on MI355X (before: one lane per sample, weights broadcast from LDS,
// one partial per 64 samples summed by one thread per parameter; calls as the
// host sees them): loss and gradient over 524,288 samples 97 against 2,145 us,
// a training step of 4,096 samples 10 against 45 us (three dependent kernels
// of 64 one-wave workgroups before, two now: 7.2 and 4.1 us, latency), the
// forward pass over 524,288 samples 44 against 46 us, where the tanh of the
// vector units (64 per sample, two transcendental operations each) sets the
// time.
#include <hip/hip_runtime.h>

#include <type_traits>

#include "rainy_kernels.hpp"

namespace atmo {

namespace {

constexpr int H = kMlpHidden, I = kMlpIn, O = kMlpOut, P = kMlpParams;
constexpr int oW1 = 0, ob1 = oW1 + H * I, oW2 = ob1 + H, ob2 = oW2 + H * H, oW3 = ob2 + H,
              ob3 = oW3 + O * H;
constexpr int kPartial = P + 1;  // gradient + loss
constexpr int kTile = 16;        // samples per wave and pass
constexpr int kWaves = 4;        // waves per workgroup
constexpr int kMaxBlocks = 512;  // workgroups of a launch: two waves per SIMD

typedef float floatx4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ floatx4 mfma(float a, float b, floatx4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

// the weights a lane needs of the forward pass: W1 with b1 as its fourth
// column, W2 as the A operand, and b2, W3 of the lane's own neurons
struct Weights {
  float w1[2], w2[2][8], b2[8], w3[O][8], b3[O];
  float mean, scale;  // of the lane's input component (the fourth is the constant 1)
};

__device__ __forceinline__ void load_weights(const float* params, const float* norm, int g, int c,
                                             Weights& w) {
#pragma unroll
  for (int T = 0; T < 2; ++T) {
    const int row = 16 * T + c;
    w.w1[T] = g < I ? params[oW1 + row * I + g] : params[ob1 + row];
#pragma unroll
    for (int q = 0; q < 8; ++q)  // k = 16 (q / 4) + 4 g + q % 4
      w.w2[T][q] = params[oW2 + row * H + 16 * (q / 4) + 4 * g + q % 4];
  }
#pragma unroll
  for (int q = 0; q < 8; ++q) {
    const int j = 16 * (q / 4) + 4 * g + q % 4;
    w.b2[q] = params[ob2 + j];
#pragma unroll
    for (int o = 0; o < O; ++o) w.w3[o][q] = params[oW3 + o * H + j];
  }
#pragma unroll
  for (int o = 0; o < O; ++o) w.b3[o] = params[ob3 + o];
  w.mean = g < I ? norm[g] : 0.0f;
  w.scale = g < I ? norm[3 + g] : 1.0f;
}

// hidden activations of the lane's neurons for sample c, and the normalised
// outputs of sample c (on every lane of its column); x: the lane's normalised
// input component
__device__ __forceinline__ void forward(const Weights& w, float x, float* h1, float* h2, float* y) {
#pragma unroll
  for (int T = 0; T < 2; ++T) {
    const floatx4 z = mfma(w.w1[T], x, floatx4{0.0f, 0.0f, 0.0f, 0.0f});
#pragma unroll
    for (int r = 0; r < 4; ++r) h1[4 * T + r] = mlp_tanh(z[r]);
  }
#pragma unroll
  for (int T = 0; T < 2; ++T) {
    floatx4 z = {w.b2[4 * T], w.b2[4 * T + 1], w.b2[4 * T + 2], w.b2[4 * T + 3]};
#pragma unroll
    for (int q = 0; q < 8; ++q) z = mfma(w.w2[T][q], h1[q], z);
#pragma unroll
    for (int r = 0; r < 4; ++r) h2[4 * T + r] = mlp_tanh(z[r]);
  }
#pragma unroll
  for (int o = 0; o < O; ++o) {
    float a = 0.0f;
#pragma unroll
    for (int q = 0; q < 8; ++q) a += w.w3[o][q] * h2[q];
    a += __shfl_xor(a, 16, 64);
    a += __shfl_xor(a, 32, 64);
    y[o] = a + w.b3[o];
  }
}

// sum over the 16 lanes of a row (lanes that share g) by row rotations
__device__ __forceinline__ float row_sum(float v) {
  auto ror = [](float x, auto ctrl) {
    return __int_as_float(
        __builtin_amdgcn_update_dpp(0, __float_as_int(x), decltype(ctrl)::value, 0xf, 0xf, false));
  };
  v += ror(v, std::integral_constant<int, 0x128>{});  // row_ror:8
  v += ror(v, std::integral_constant<int, 0x124>{});  // row_ror:4
  v += ror(v, std::integral_constant<int, 0x122>{});  // row_ror:2
  v += ror(v, std::integral_constant<int, 0x121>{});  // row_ror:1
  return v;
}

}  // namespace

// partial[block][P + 1]: gradient and loss of the samples [offset, offset +
// count) (through `perm` when given) that the block's waves take
__global__ __launch_bounds__(64 * kWaves) void mlp_loss_grad_kernel(
    const float* params, const float* norm, const float* x, const float* y, const int* perm,
    int64_t offset, int64_t count, float inv_count, float* partial) {
  // per wave h1, h2 deltas and inputs by [neuron][sample]; the gradients of the
  // waves follow in the same memory
  constexpr int S = kTile + 1;
  constexpr int kStage = (3 * H + I + 1) * S;
  constexpr int kShared = kWaves * (kStage > kPartial ? kStage : kPartial);
  __shared__ float smem[kShared];
  const int wave = threadIdx.x >> 6, l = threadIdx.x & 63, g = l >> 4, c = l & 15;
  float* sh1 = smem + wave * kStage;
  float* sd1 = sh1 + H * S;
  float* sd2 = sd1 + H * S;
  float* sx = sd2 + H * S;
  Weights w;
  load_weights(params, norm, g, c, w);
  float w2t[2][8];  // W2 transposed as the A operand
#pragma unroll
  for (int T = 0; T < 2; ++T)
#pragma unroll
    for (int q = 0; q < 8; ++q)
      w2t[T][q] = params[oW2 + (16 * (q / 4) + 4 * g + q % 4) * H + 16 * T + c];
  float ymean[O], yscale[O];
#pragma unroll
  for (int o = 0; o < O; ++o) {
    ymean[o] = norm[6 + o];
    yscale[o] = norm[8 + o];
  }
  floatx4 gw2[2][2] = {}, gw1[2] = {};
  float gb2[8] = {}, gw3[O][8] = {}, gb3[O] = {}, loss = 0.0f;

  const int64_t tiles = (count + kTile - 1) / kTile;
  const int64_t stride = (int64_t)gridDim.x * kWaves;
  // every wave of a workgroup makes the same number of passes (barriers inside)
  const int64_t first = (int64_t)blockIdx.x * kWaves;
  for (int64_t t0 = first; t0 < tiles; t0 += stride) {
    const int64_t b = (t0 + wave) * kTile + c;
    const bool valid = b < count;
    const int64_t at = valid ? b : 0;
    const int64_t src = perm ? (int64_t)perm[offset + at] : offset + at;
    const float xin = g < I ? x[I * src + g] : 1.0f;
    float yt[O];
#pragma unroll
    for (int o = 0; o < O; ++o) yt[o] = (y[O * src + o] - ymean[o]) / yscale[o];
    const float xn = (xin - w.mean) / w.scale;
    float h1[8], h2[8], out[O], dy[O];
    forward(w, xn, h1, h2, out);
#pragma unroll
    for (int o = 0; o < O; ++o) {
      const float d = valid ? out[o] - yt[o] : 0.0f;
      loss += d * d * inv_count;
      dy[o] = 2.0f * d * inv_count;
      gb3[o] += dy[o];
    }
    // deltas of the pre-activations
    float d2[8], d1[8];
#pragma unroll
    for (int q = 0; q < 8; ++q) {
      float a = 0.0f;
#pragma unroll
      for (int o = 0; o < O; ++o) {
        a += dy[o] * w.w3[o][q];
        gw3[o][q] += dy[o] * h2[q];
      }
      d2[q] = a * (1.0f - h2[q] * h2[q]);
      gb2[q] += d2[q];
    }
#pragma unroll
    for (int T = 0; T < 2; ++T) {
      floatx4 z = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
      for (int q = 0; q < 8; ++q) z = mfma(w2t[T][q], d2[q], z);
#pragma unroll
      for (int r = 0; r < 4; ++r) d1[4 * T + r] = z[r] * (1.0f - h1[4 * T + r] * h1[4 * T + r]);
    }
    __syncthreads();  // the tile before has been read
#pragma unroll
    for (int q = 0; q < 8; ++q) {
      const int j = 16 * (q / 4) + 4 * g + q % 4;
      sh1[j * S + c] = h1[q];
      sd1[j * S + c] = d1[q];
      sd2[j * S + c] = d2[q];
    }
    sx[g * S + c] = xn;
    __syncthreads();
    // sums over the samples 4 q + g
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int s = 4 * q + g;
      const float a0 = sd2[c * S + s], a1 = sd2[(16 + c) * S + s];
      const float b0 = sh1[c * S + s], b1 = sh1[(16 + c) * S + s];
      gw2[0][0] = mfma(a0, b0, gw2[0][0]);
      gw2[0][1] = mfma(a0, b1, gw2[0][1]);
      gw2[1][0] = mfma(a1, b0, gw2[1][0]);
      gw2[1][1] = mfma(a1, b1, gw2[1][1]);
      const float xs = c <= I ? sx[(c <= I ? c : 0) * S + s] : 0.0f;
      gw1[0] = mfma(sd1[c * S + s], xs, gw1[0]);
      gw1[1] = mfma(sd1[(16 + c) * S + s], xs, gw1[1]);
    }
  }
  // the per-sample sums over the wave's 16 columns
#pragma unroll
  for (int q = 0; q < 8; ++q) {
    gb2[q] = row_sum(gb2[q]);
#pragma unroll
    for (int o = 0; o < O; ++o) gw3[o][q] = row_sum(gw3[o][q]);
  }
#pragma unroll
  for (int o = 0; o < O; ++o) gb3[o] = row_sum(gb3[o]);
  loss = row_sum(loss);
  __syncthreads();
  float* out = smem + wave * kPartial;
#pragma unroll
  for (int T = 0; T < 2; ++T)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int j = 16 * T + 4 * g + r;
      out[oW2 + j * H + c] = gw2[T][0][r];
      out[oW2 + j * H + 16 + c] = gw2[T][1][r];
      if (c < I) out[oW1 + j * I + c] = gw1[T][r];
      if (c == I) out[ob1 + j] = gw1[T][r];
      if (c == 0) {
        out[ob2 + j] = gb2[4 * T + r];
#pragma unroll
        for (int o = 0; o < O; ++o) out[oW3 + o * H + j] = gw3[o][4 * T + r];
      }
    }
  if (l == 0) {
#pragma unroll
    for (int o = 0; o < O; ++o) out[ob3 + o] = gb3[o];
    out[P] = loss;
  }
  __syncthreads();
  for (int i = threadIdx.x; i < kPartial; i += 64 * kWaves) {
    float a = smem[i];
#pragma unroll
    for (int k = 1; k < kWaves; ++k) a += smem[k * kPartial + i];
    partial[(size_t)blockIdx.x * kPartial + i] = a;
  }
}

struct AdamStep {
  float *params, *m, *v;  // params NULL: the gradient only
  float lr, beta1, beta2, eps, bc1, bc2;
};

// grad_loss[P + 1] = sum over the blocks' partials in a fixed order: 32 entries
// per workgroup, its eight groups of 32 lanes taking every eighth block; then
// Adam on the parameters
__global__ __launch_bounds__(256) void mlp_reduce_kernel(const float* partial, int blocks,
                                                         float* grad_loss, AdamStep adam) {
  __shared__ float s[8][32];
  const int k = threadIdx.x & 31, part = threadIdx.x >> 5;
  const int i = blockIdx.x * 32 + k;
  float acc = 0.0f;
  if (i < kPartial) {
#pragma unroll 8
    for (int b = part; b < blocks; b += 8) acc += partial[(size_t)b * kPartial + i];
  }
  s[part][k] = acc;
  __syncthreads();
  if (part != 0 || i >= kPartial) return;
  float g = s[0][k];
#pragma unroll
  for (int p = 1; p < 8; ++p) g += s[p][k];
  grad_loss[i] = g;
  if (!adam.params || i >= P) return;
  const float mi = adam.beta1 * adam.m[i] + (1.0f - adam.beta1) * g;
  const float vi = adam.beta2 * adam.v[i] + (1.0f - adam.beta2) * g * g;
  adam.m[i] = mi;
  adam.v[i] = vi;
  adam.params[i] -= adam.lr * (mi / adam.bc1) / (sqrtf(vi / adam.bc2) + adam.eps);
}

// y[2 n] = network(x[3 n]) in physical units; lanes past n evaluate the
// normalisation means and write nothing
__global__ __launch_bounds__(64 * kWaves) void mlp_forward_kernel(const float* params,
                                                                  const float* norm,
                                                                  const float* x, float* y,
                                                                  int64_t n) {
  const int wave = threadIdx.x >> 6, l = threadIdx.x & 63, g = l >> 4, c = l & 15;
  Weights w;
  load_weights(params, norm, g, c, w);
  const int64_t tiles = (n + kTile - 1) / kTile, stride = (int64_t)gridDim.x * kWaves;
  for (int64_t t = (int64_t)blockIdx.x * kWaves + wave; t < tiles; t += stride) {
    const int64_t q = t * kTile + c;
    const bool valid = q < n;
    const float xin = g < I ? (valid ? x[I * q + g] : w.mean) : 1.0f;
    float h1[8], h2[8], out[O];
    forward(w, (xin - w.mean) / w.scale, h1, h2, out);
    // lane g writes output g
    const float v = g == 0 ? out[0] : out[1];
    if (valid && g < O) y[O * q + g] = v * norm[8 + g] + norm[6 + g];
  }
}

int mlp_grad_blocks(int64_t count) {
  const int64_t blocks = (count + kTile * kWaves - 1) / (kTile * kWaves);
  return (int)(blocks < kMaxBlocks ? blocks : kMaxBlocks);
}

int mlp_launch_loss_grad(const float* params, const float* norm, const float* x, const float* y,
                         const int* perm, int64_t offset, int64_t count, float* partial,
                         hipStream_t s) {
  const int blocks = mlp_grad_blocks(count);
  hipLaunchKernelGGL(mlp_loss_grad_kernel, dim3(blocks), dim3(64 * kWaves), 0, s, params, norm, x,
                     y, perm, offset, count, 1.0f / (float)count, partial);
  return blocks;
}

void mlp_launch_reduce(const float* partial, int blocks, float* grad_loss, hipStream_t s) {
  hipLaunchKernelGGL(mlp_reduce_kernel, dim3((kPartial + 31) / 32), dim3(256), 0, s, partial,
                     blocks, grad_loss, AdamStep{});
}

void mlp_launch_reduce_adam(const float* partial, int blocks, float* grad_loss, float* params,
                            float* m, float* v, float lr, float beta1, float beta2, float eps,
                            int step, hipStream_t s) {
  const float bc1 = 1.0f - powf(beta1, (float)step), bc2 = 1.0f - powf(beta2, (float)step);
  hipLaunchKernelGGL(mlp_reduce_kernel, dim3((kPartial + 31) / 32), dim3(256), 0, s, partial,
                     blocks, grad_loss, AdamStep{params, m, v, lr, beta1, beta2, eps, bc1, bc2});
}

void mlp_launch_forward(const float* params, const float* norm, const float* x, float* y,
                        int64_t n, hipStream_t s) {
  // four waves per SIMD at most, each over many tiles
  const int64_t blocks = (n + kTile * kWaves - 1) / (kTile * kWaves);
  hipLaunchKernelGGL(mlp_forward_kernel, dim3((unsigned)(blocks < 1024 ? blocks : 1024)),
                     dim3(64 * kWaves), 0, s, params, norm, x, y, n);
}

}  // namespace atmo
