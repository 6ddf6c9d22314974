// Learned block proposal network: HIP kernels for gfx950.
//
// No counterpart in lacker/seticore. A small convolutional network scores
// 4096-channel blocks of a 16-row coarse channel from a frequency-pooled,
// noise-normalised tile; only blocks it flags are searched with the full tree
// (the plain search is the fallback and the judge of its recall).
//
// Network (23,393 parameters; weights and activations stored as BF16,
// products accumulated in FP32):
//   input  z [16][1024]           pooled power, z = 2 (sum of 4 channels -
//                                 median/4) / std (column-sum statistics),
//                                 clamped to [-4, 32]
//   conv1  1 -> 16, 3x5, stride (1,2), pad (1,2), ReLU   -> h1 [16][512][16]
//   conv2 16 -> 32, 3x5, stride (2,2), pad (1,2), ReLU   -> h2 [ 8][256][32]
//   conv3 32 -> 32, 3x5, stride (2,2), pad (1,2), ReLU   -> h3 [ 4][128][32]
//   head   1x1 32 -> 1 (FP32 weights), max over the 512 positions -> logit
// Activations are NHWC (channels innermost). The convolutions run on the
// matrix cores (v_mfma_f32_16x16x16_bf16) as implicit GEMMs: rows = output
// positions, columns = output channels, K = (tap, input channel).
//
// Training: weighted binary cross-entropy on the block logit. The max makes
// the backward pass sparse - only the receptive field of each block's argmax
// position carries gradient (3x5 positions of h2, 7x13 of h1) - so one
// workgroup per block computes that block's whole parameter gradient, and a
// second kernel sums the per-block gradients in a fixed order
// (deterministic). Adam updates FP32 master weights, then the BF16 copies are
// refreshed.

#include <hip/hip_runtime.h>
#include <math.h>
#include <stdint.h>

#include "dd_internal.h"
#include "pn_internal.h"

namespace sc {
namespace pn {

namespace {

typedef short bf16x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

// Round-to-nearest-even float -> bfloat16 bits (inputs are finite).
__device__ __forceinline__ unsigned short f2bf(float f) {
  unsigned u = __float_as_uint(f);
  u += 0x7FFFu + ((u >> 16) & 1u);
  return (unsigned short)(u >> 16);
}
__device__ __forceinline__ float bf2f(unsigned short h) {
  return __uint_as_float((unsigned)h << 16);
}

// Where the BF16 copy of weight (co, tap t, ci) of a 3x5 convolution with CIN
// input channels lies: in the order of the matrix-core operands, so that a
// wave's operand is one 512-byte load (as rows of an output channel it touched
// 16 cache lines, which bound the forward pass).
template <int CIN>
__device__ __forceinline__ int weight_index(int co, int t, int ci) {
  return ((((co / 16) * 15 + t) * (CIN / 16) + ci / 16) * 64 + co % 16 + 16 * (ci % 16 / 4)) * 4 +
         ci % 4;
}

// Four ReLU outputs to BF16 (v_cvt_pk_bf16_f32, round to nearest even as f2bf).
__device__ __forceinline__ bf16x4 relu_bf16(const f32x4& acc, const float (&bias)[4]) {
  typedef float f32x2 __attribute__((ext_vector_type(2)));
  typedef __bf16 bf2 __attribute__((ext_vector_type(2)));
  const bf2 lo = __builtin_convertvector(
      (f32x2{fmaxf(acc[0] + bias[0], 0.0f), fmaxf(acc[1] + bias[1], 0.0f)}), bf2);
  const bf2 hi = __builtin_convertvector(
      (f32x2{fmaxf(acc[2] + bias[2], 0.0f), fmaxf(acc[3] + bias[3], 0.0f)}), bf2);
  typedef unsigned u32x2 __attribute__((ext_vector_type(2)));
  return __builtin_bit_cast(bf16x4,
                            (u32x2{__builtin_bit_cast(unsigned, lo), __builtin_bit_cast(unsigned, hi)}));
}

// ---------------------------------------------------------------------------
// Pooling: z[blk][t][j] from the 4 channels 4096*blk + 4j .. +3 of row t.
template <typename In>
__device__ __forceinline__ float load_f32(const In* p);
template <>
__device__ __forceinline__ float load_f32<float>(const float* p) { return *p; }
template <>
__device__ __forceinline__ float load_f32<unsigned short>(const unsigned short* p) {
  return bf2f(*p);
}
template <>
__device__ __forceinline__ float load_f32<_Float16>(const _Float16* p) { return (float)*p; }

template <typename In>
__device__ __forceinline__ void pool_body(const In* __restrict__ x, long stride, int nblk,
                                          const float* __restrict__ stats,
                                          unsigned short* __restrict__ z) {
  const long i = blockIdx.x * 256L + threadIdx.x;  // over nblk * 16 * 1024
  if (i >= (long)nblk * kRows * kPooled) return;
  const int j = (int)(i % kPooled);
  const int t = (int)((i / kPooled) % kRows);
  const long blk = i / ((long)kPooled * kRows);
  const In* p = x + t * stride + blk * kBlockChannels + 4L * j;
  // The four samples in one load, at any element alignment.
  struct __attribute__((packed, aligned(sizeof(In)))) In4 {
    In v[4];
  };
  const In4 q = *(const In4*)p;
  const float s = (load_f32<In>(&q.v[0]) + load_f32<In>(&q.v[1])) +
                  (load_f32<In>(&q.v[2]) + load_f32<In>(&q.v[3]));
  const float median = stats[0], sd = stats[1];
  float v = 2.0f * (s - 0.25f * median) / sd;
  v = fminf(fmaxf(v, kZMin), kZMax);
  z[i] = f2bf(v);
}

template <typename In>
__global__ void __launch_bounds__(256)
    pool_kernel(const In* __restrict__ x, long stride, int nblk, const float* __restrict__ stats,
                unsigned short* __restrict__ z) {
  pool_body<In>(x, stride, nblk, stats, z);
}

// Several channels (grid.y = channel), channel c's tiles at z + c * nblk tiles.
template <typename In>
__global__ void __launch_bounds__(256)
    pool_set_kernel(FrontSet fs, long stride, int nblk, unsigned short* __restrict__ z) {
  const int c = blockIdx.y;
  pool_body<In>((const In*)fs.x[c], stride, nblk, fs.stats_out[c],
                z + (long)c * nblk * kRows * kPooled);
}

// ---------------------------------------------------------------------------
// The three convolutions of a column tile in one workgroup, on the matrix
// cores, with the activations passed through LDS.
//
// Lane layout of v_mfma_f32_16x16x16_bf16: A[row][k] sits in lane
// row + 16*(k/4), element k%4; B[k][col] in lane col + 16*(k/4), element k%4;
// D[row][col] in lane col + 16*(row/4), element row%4. The products are formed
// transposed, D[channel][position] = W[channel][k] * X[k][position], so each
// lane ends with 4 consecutive channels of one position: one 8-byte store.
//
// A workgroup takes kTile3 = 16 columns of h3 of one block: 35 columns of h2
// and 80 of h1 (73 needed, in whole groups of 16 so that a group lies in one
// row), halo included, 63.5 KB of LDS, two workgroups (16 waves) per CU. Columns
// outside the maps and the row above them are zero in LDS, so the products
// need no bounds tests. A stride-2 convolution reads every second column, so
// columns are stored split by parity, and each group of four channels (a
// lane's share of an operand) is a plane of its own: 16 lanes read 128
// consecutive bytes, and the planes of a 32-lane half lie 32 banks apart. (With
// a position's channels together, two thirds of the LDS cycles were bank
// conflicts: 74 / 529 us at 256 / 2048 blocks.) conv2 takes positions 16 at a time across row ends. Each sum runs
// over (tap, channel) in the order of the separate convolutions this replaces,
// so logits are bit-identical to theirs.
//
// Separate kernels wrote and re-read every activation through memory and
// gathered their operands from L1/L2: 108 / 868 us for 256 / 2048 blocks, with
// the head; 60 / 479 us now, 15 instead of 46 for one. What bounds this one is
// vector work around the products (conv1 above all: an operand's taps, bias,
// ReLU, rounding and addresses for one product per 16 positions) and, with the
// activations kept, writing 416 KB per block. h1, h2 may be null (not kept).
constexpr int kTile3 = 16;
constexpr int kCols2 = 2 * kTile3 + 3, kCols1 = (4 * kTile3 + 9 + 15) / 16 * 16;
constexpr int kHalf2 = (kCols2 + 1) / 2, kHalf1 = kCols1 / 2;  // per column parity
constexpr int kPitchZ = 2 * kCols1 + 4;
constexpr int kPlane1 = (kH1 + 1) * 2 * kHalf1, kPlane2 = (kH2 + 1) * 2 * kHalf2 + 12;
static_assert(kPlane1 * 2 % 64 == 32 && kPlane2 * 2 % 64 == 32, "planes half the banks apart");
constexpr int kForwardThreads = 512;
constexpr int kForwardWaves = kForwardThreads / 64;

__global__ void __launch_bounds__(kForwardThreads, 4)
    forward_kernel(const unsigned short* __restrict__ z, const unsigned short* __restrict__ w1b,
                   const unsigned short* __restrict__ w2b, const unsigned short* __restrict__ w3b,
                   const float* __restrict__ params, unsigned short* __restrict__ h1,
                   unsigned short* __restrict__ h2, unsigned short* __restrict__ h3) {
  __shared__ __attribute__((aligned(16))) bf16x4 h1s[4][kPlane1];
  __shared__ __attribute__((aligned(16))) bf16x4 h2s[2][4][kPlane2];
  // z is done with when h2 is first written.
  unsigned short* zs = (unsigned short*)h2s;
  static_assert((kRows + 2) * kPitchZ * 2 <= sizeof(h2s), "z fits");
  static_assert(sizeof(h1s) + sizeof(h2s) <= 64 * 1024, "LDS of a workgroup");
  constexpr int kTiles = kW3 / kTile3;
  const int tid = threadIdx.x, lane = tid % 64, wave = tid / 64;
  const int r = lane % 16, g = lane / 16;
  const int a3 = blockIdx.x % kTiles * kTile3;  // first column in h3
  const int x2o = 2 * a3 - 2, x1o = 4 * a3 - 6, zo = 8 * a3 - 14;
  const long b = blockIdx.x / kTiles;

  // z rows -1 .. 16 (zo is even and the map 1024 wide: pairs of columns lie
  // inside or outside together); the zero rows above h1 and h2.
  for (int y = wave; y < kRows + 2; y += kForwardWaves) {
    const unsigned* row = (const unsigned*)(z + (b * kRows + y - 1) * kPooled + zo);
    for (int c = lane; c < kPitchZ / 2; c += 64) {
      const int x = zo + 2 * c;
      const bool ok = y >= 1 && y <= kRows && x >= 0 && x < kPooled;
      ((unsigned*)zs)[y * (kPitchZ / 2) + c] = ok ? row[c] : 0u;
    }
  }
  for (int e = tid; e < 4 * 2 * kHalf1; e += kForwardThreads)
    h1s[e / (2 * kHalf1)][e % (2 * kHalf1)] = bf16x4{0, 0, 0, 0};

  const bf16x4 w1 = *(const bf16x4*)(w1b + r * 16 + 4 * g);
  float bias1[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) bias1[i] = params[kOffB1 + 4 * g + i];
  // conv2: this wave's 16 output channels.
  const int n = wave % 2;
  bf16x4 w2[15];
#pragma unroll
  for (int t = 0; t < 15; ++t)
    w2[t] = ((const bf16x4*)w2b)[(n * 15 + t) * 64 + lane];
  __syncthreads();

  // conv1: position (y, c) reads z rows y .. y+2, columns 2c .. 2c+4; this
  // lane's four taps are 4g .. 4g+3 (15 does not exist). Two rows per wave.
  int tap[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int k = min(4 * g + i, 14);
    tap[i] = k / 5 * kPitchZ + k % 5 + 2 * r;
  }
  static_assert(kH1 == 2 * kForwardWaves, "conv1 rows");
#pragma unroll
  for (int yy = 0; yy < 2; ++yy) {
    const int y = 2 * wave + yy;
    const unsigned short* zrow = zs + y * kPitchZ;
    bf16x4* dst = h1s[g] + ((y + 1) * 2 + (r & 1)) * kHalf1 + (r >> 1);
    unsigned short* keep = h1 ? h1 + ((b * kH1 + y) * kW1 + x1o) * kC1 : nullptr;
    // All products of the row first, then the stores.
    bf16x4 v[kCols1 / 16];
#pragma unroll
    for (int u = 0; u < kCols1 / 16; ++u) {
      bf16x4 a;
#pragma unroll
      for (int i = 0; i < 4; ++i) a[i] = (short)zrow[tap[i] + 32 * u];
      if (g == 3) a[3] = 0;
      const f32x4 acc =
          __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(w1, a, f32x4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
      v[u] = relu_bf16(acc, bias1);
      const int x = x1o + 16 * u + r;
      if (x < 0 || x >= kW1) v[u] = bf16x4{0, 0, 0, 0};
    }
#pragma unroll
    for (int u = 0; u < kCols1 / 16; ++u) dst[8 * u] = v[u];
    if (keep) {
#pragma unroll
      for (int u = 0; u < kCols1 / 16; ++u) {
        const int c = 16 * u + r;
        if (c >= 6 && c < 6 + 4 * kTile3) *(bf16x4*)(keep + c * kC1 + 4 * g) = v[u];
      }
    }
  }
  __syncthreads();

  // conv2: position (y, c) reads h1 rows 2y .. 2y+2 (row 0 is the zero row),
  // columns 2c .. 2c+4. Waves of one channel half take every fourth group.
  for (int e = tid; e < 8 * 2 * kHalf2; e += kForwardThreads)
    h2s[e / (8 * kHalf2)][e / (2 * kHalf2) % 4][e % (2 * kHalf2)] = bf16x4{0, 0, 0, 0};
  float bias2[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) bias2[i] = params[kOffB2 + n * 16 + 4 * g + i];
  unsigned short* keep2 = h2 ? h2 + b * kH2 * kW2 * kC2 : nullptr;
  for (int u = wave / 2; u < (kH2 * kCols2 + 15) / 16; u += kForwardWaves / 2) {
    const int p = 16 * u + r, pc = min(p, kH2 * kCols2 - 1);
    const int y = pc / kCols2, c = pc % kCols2, x = x2o + c;
    const bf16x4* src = h1s[g] + 2 * y * 2 * kHalf1 + c;
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int t = 0; t < 15; ++t) {
      const int ty = t / 5, tx = t % 5;
      const bf16x4 a = src[(ty * 2 + (tx & 1)) * kHalf1 + (tx >> 1)];
      acc = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(w2[t], a, acc, 0, 0, 0);
    }
    bf16x4 v = relu_bf16(acc, bias2);
    if (x < 0 || x >= kW2) v = bf16x4{0, 0, 0, 0};
    if (p < kH2 * kCols2) {
      h2s[n][g][((y + 1) * 2 + (c & 1)) * kHalf2 + (c >> 1)] = v;
      if (keep2 && c >= 2 && c < 2 + 2 * kTile3)
        *(bf16x4*)(keep2 + (y * kW2 + x) * kC2 + n * 16 + 4 * g) = v;
    }
  }
  // conv3: one (row, channel half) per wave.
  static_assert(kForwardWaves == 2 * kH3, "conv3 units");
  const int y3 = wave / 2;
  bf16x4 w3[15][2];
#pragma unroll
  for (int t = 0; t < 15; ++t)
#pragma unroll
    for (int s = 0; s < 2; ++s) w3[t][s] = ((const bf16x4*)w3b)[((n * 15 + t) * 2 + s) * 64 + lane];
  float bias3[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) bias3[i] = params[kOffB3 + n * 16 + 4 * g + i];
  __syncthreads();
  f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int t = 0; t < 15; ++t) {
    const int ty = t / 5, tx = t % 5;
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      const bf16x4 a =
          h2s[s][g][((2 * y3 + ty) * 2 + (tx & 1)) * kHalf2 + r + (tx >> 1)];
      acc = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(w3[t][s], a, acc, 0, 0, 0);
    }
  }
  *(bf16x4*)(h3 + ((b * kH3 + y3) * kW3 + a3 + r) * kC3 + n * 16 + 4 * g) = relu_bf16(acc, bias3);
}

// Head: logit[b] = max over positions of (bh + sum_c h3[pos][c] * wh[c]);
// argmax = lowest position attaining it.
__global__ void __launch_bounds__(256)
    head_kernel(const unsigned short* __restrict__ h3, const float* __restrict__ params,
                float* __restrict__ logits, int* __restrict__ argmax) {
  __shared__ float sv[256];
  __shared__ int si[256];
  const long b = blockIdx.x;
  const float* wh = params + kOffWH;
  const float bh = params[kOffBH];
  float best = -INFINITY;
  int bi = 0;
  for (int pos = threadIdx.x; pos < kH3 * kW3; pos += 256) {
    const unsigned short* h = h3 + (b * kH3 * kW3 + pos) * kC3;
    float s = bh;
#pragma unroll
    for (int c = 0; c < kC3; ++c) s += bf2f(h[c]) * wh[c];
    if (s > best) {
      best = s;
      bi = pos;
    }
  }
  sv[threadIdx.x] = best;
  si[threadIdx.x] = bi;
  __syncthreads();
  for (int w = 128; w > 0; w >>= 1) {
    if ((int)threadIdx.x < w) {
      const float o = sv[threadIdx.x + w];
      const int oi = si[threadIdx.x + w];
      if (o > sv[threadIdx.x] || (o == sv[threadIdx.x] && oi < si[threadIdx.x])) {
        sv[threadIdx.x] = o;
        si[threadIdx.x] = oi;
      }
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    logits[b] = sv[0];
    if (argmax) argmax[b] = si[0];
  }
}

// ---------------------------------------------------------------------------
// Training.

// Weighted BCE: per block w*(max(z,0) - z*y + log1p(exp(-|z|))), w = pos_weight
// for y = 1; dz = w*(sigmoid(z) - y)/B; loss = mean (one workgroup, fixed order).
__global__ void __launch_bounds__(256)
    loss_kernel(const float* __restrict__ logits, const float* __restrict__ labels, int B,
                float pos_weight, float* __restrict__ dz, float* __restrict__ loss) {
  __shared__ double part[256];
  double acc = 0.0;
  for (int b = threadIdx.x; b < B; b += 256) {
    const float z = logits[b], y = labels[b];
    const float w = y > 0.5f ? pos_weight : 1.0f;
    const float l = fmaxf(z, 0.0f) - z * y + log1pf(expf(-fabsf(z)));
    const float p = 1.0f / (1.0f + expf(-z));
    dz[b] = w * (p - y) / (float)B;
    acc += (double)(w * l);
  }
  part[threadIdx.x] = acc;
  __syncthreads();
  for (int w = 128; w > 0; w >>= 1) {
    if ((int)threadIdx.x < w) part[threadIdx.x] += part[threadIdx.x + w];
    __syncthreads();
  }
  if (threadIdx.x == 0 && loss) loss[0] = (float)(part[0] / B);
}

// One workgroup per block: the whole parameter gradient of that block's loss
// term into gpart[b][kNumParams] (every entry written). Everything the block's
// argmax position depends on - 3x5 positions of h2, 7x13 of h1, 9x29 of z and
// conv2's weights - is first brought into LDS, zero outside the maps, so the
// sums below are free of bounds tests and of memory latency: at 256 blocks
// (one workgroup per CU) 127 us with global loads inside the sums on 256
// threads, 21 us now.
constexpr int kBackThreads = 512;
constexpr int kR1H = 7, kR1W = 13, kR1 = kR1H * kR1W;  // receptive field in h1
constexpr int kRZH = kR1H + 2, kRZW = 2 * kR1W + 3;    // and in z
__global__ void __launch_bounds__(kBackThreads)
    backward_kernel(const unsigned short* __restrict__ z, const unsigned short* __restrict__ h1,
                    const unsigned short* __restrict__ h2, const unsigned short* __restrict__ h3,
                    const int* __restrict__ argmax, const float* __restrict__ dz,
                    const float* __restrict__ params, float* __restrict__ gpart) {
  const long b = blockIdx.x;
  const int tid = threadIdx.x;
  float* g = gpart + b * (long)kNumParams;
  __shared__ float dY3[kC3];
  __shared__ float h2s[15][kC2];
  __shared__ __attribute__((aligned(16))) float dY2[15][kC2];  // conv2 outputs at conv3's taps
  __shared__ float h1s[kR1][kC1];
  __shared__ float dY1[kR1][kC1];
  __shared__ float zs[kRZH][kRZW];
  __shared__ unsigned short w2s[kC2 * 15 * kC1];

  const int pos = argmax[b];
  const int y3 = pos / kW3, x3 = pos % kW3;
  const float d = dz[b];

  // Tap t of conv3 reads h2 at (2 y3 + t/5 - 1, 2 x3 + t%5 - 2); tap t2 of
  // conv2 at conv3's tap j reads cell (2 (j/5) + t2/5, 2 (j%5) + t2%5) of the
  // h1 field, whose corner is (4 y3 - 3, 4 x3 - 6); tap t of conv1 at an h1
  // cell (y, x) reads cell (y + t/5, 2 x + t%5) of the z field.
  const int y1o = 4 * y3 - 3, x1o = 4 * x3 - 6;
  if (tid < 15 * kC2) {
    const int t = tid / kC2, yy = 2 * y3 + t / 5 - 1, xx = 2 * x3 + t % 5 - 2;
    const bool ok = yy >= 0 && yy < kH2 && xx >= 0 && xx < kW2;
    h2s[t][tid % kC2] = ok ? bf2f(h2[((b * kH2 + yy) * kW2 + xx) * kC2 + tid % kC2]) : 0.0f;
  }
  for (int e = tid; e < kR1 * kC1; e += kBackThreads) {
    const int cell = e / kC1, yy = y1o + cell / kR1W, xx = x1o + cell % kR1W;
    const bool ok = yy >= 0 && yy < kH1 && xx >= 0 && xx < kW1;
    h1s[cell][e % kC1] = ok ? bf2f(h1[((b * kH1 + yy) * kW1 + xx) * kC1 + e % kC1]) : 0.0f;
  }
  if (tid < kRZH * kRZW) {
    const int zy = y1o - 1 + tid / kRZW, zx = 2 * x1o - 2 + tid % kRZW;
    const bool ok = zy >= 0 && zy < kRows && zx >= 0 && zx < kPooled;
    zs[tid / kRZW][tid % kRZW] = ok ? bf2f(z[(b * kRows + zy) * kPooled + zx]) : 0.0f;
  }
  // The BF16 weights the forward pass used, rounded again from the master copy
  // (whose order suits these sums).
  for (int e = tid; e < kC2 * 15 * kC1; e += kBackThreads) w2s[e] = f2bf(params[kOffW2 + e]);

  // Head and conv3 bias.
  if (tid < kC3) {
    const float a = bf2f(h3[((b * kH3 + y3) * kW3 + x3) * kC3 + tid]);
    g[kOffWH + tid] = d * a;
    const float dh = d * params[kOffWH + tid];
    const float dy = a > 0.0f ? dh : 0.0f;
    dY3[tid] = dy;
    g[kOffB3 + tid] = dy;
  }
  if (tid == 0) g[kOffBH] = d;
  __syncthreads();

  // conv3 weights: dW3[co][t][ci] = dY3[co] * h2[p2(t)][ci].
  for (int e = tid; e < kC3 * 15 * kC2; e += kBackThreads)
    g[kOffW3 + e] = dY3[e / (kC2 * 15)] * h2s[(e / kC2) % 15][e % kC2];
  // Gradient at the 15 conv2 outputs, through the ReLU.
  if (tid < 15 * kC2) {
    const int ci = tid % kC2, t = tid / kC2;
    float s = 0.0f;
#pragma unroll
    for (int co = 0; co < kC3; ++co) s += dY3[co] * bf2f(f2bf(params[kOffW3 + (co * 15 + t) * kC2 + ci]));
    dY2[t][ci] = h2s[t][ci] > 0.0f ? s : 0.0f;
  }
  __syncthreads();

  // conv2 bias and weights: dW2[co][t2][ci] = sum_j dY2[j][co] * h1[cell(j, t2)][ci],
  // 16 output channels per thread.
  if (tid < kC2) {
    float s = 0.0f;
    for (int j = 0; j < 15; ++j) s += dY2[j][tid];
    g[kOffB2 + tid] = s;
  }
  if (tid < 2 * 15 * kC1) {
    const int e = tid % (15 * kC1), co0 = 16 * (tid / (15 * kC1));
    const int ci = e % kC1, t2 = e / kC1;
    const int c0 = t2 / 5 * kR1W + t2 % 5;
    float acc[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) acc[i] = 0.0f;
#pragma unroll
    for (int j = 0; j < 15; ++j) {
      const float h = h1s[c0 + j / 5 * 2 * kR1W + j % 5 * 2][ci];
#pragma unroll
      for (int i = 0; i < 16; ++i) acc[i] += dY2[j][co0 + i] * h;
    }
#pragma unroll
    for (int i = 0; i < 16; ++i) g[kOffW2 + (co0 + i) * 15 * kC1 + e] = acc[i];
  }
  // Gradient at the h1 field, through the ReLU.
  for (int e = tid; e < kR1 * kC1; e += kBackThreads) {
    const int ci = e % kC1, cell = e / kC1, cy = cell / kR1W, cx = cell % kR1W;
    float s = 0.0f;
    for (int j = 0; j < 15; ++j) {
      const int ty = cy - j / 5 * 2, tx = cx - j % 5 * 2;
      if (ty < 0 || ty >= 3 || tx < 0 || tx >= 5) continue;
      const unsigned short* w = w2s + (ty * 5 + tx) * kC1 + ci;
#pragma unroll
      for (int co = 0; co < kC2; ++co) s += dY2[j][co] * bf2f(w[co * 15 * kC1]);
    }
    dY1[cell][ci] = h1s[cell][ci] > 0.0f ? s : 0.0f;
  }
  __syncthreads();

  // conv1 bias and weights: dW1[co][t] = sum_cells dY1[cell][co] * z[cell(y, x, t)].
  if (tid < kC1 * 15) {
    const int co = tid / 15, t = tid % 15;
    float s = 0.0f;
    for (int cy = 0; cy < kR1H; ++cy)
#pragma unroll
      for (int cx = 0; cx < kR1W; ++cx)
        s += dY1[cy * kR1W + cx][co] * zs[cy + t / 5][2 * cx + t % 5];
    g[kOffW1 + co * 15 + t] = s;
  } else if (tid >= kBackThreads - kC1) {
    const int co = tid - (kBackThreads - kC1);
    float s = 0.0f;
    for (int cell = 0; cell < kR1; ++cell) s += dY1[cell][co];
    g[kOffB1 + co] = s;
  }
}

// grad[p] = sum over b of gpart[b][p]: 64 parameters per workgroup, each of
// its four waves sums a quarter of the blocks in ascending order with 16 loads
// in flight, then the quarters are added in order (one thread per parameter
// with a load at a time took 62 us at 256 blocks, 6 us now).
__global__ void __launch_bounds__(256)
    reduce_grad_kernel(const float* __restrict__ gpart, int B, float* __restrict__ grad) {
  __shared__ float part[4][64];
  const int lane = threadIdx.x % 64, wave = threadIdx.x / 64;
  const int p = blockIdx.x * 64 + lane;
  const int per = (B + 3) / 4, b1 = min(B, (wave + 1) * per);
  float s = 0.0f;
  if (p < kNumParams) {
    int b = wave * per;
    for (; b + 16 <= b1; b += 16) {
      float v[16];
#pragma unroll
      for (int i = 0; i < 16; ++i) v[i] = gpart[(long)(b + i) * kNumParams + p];
#pragma unroll
      for (int i = 0; i < 16; ++i) s += v[i];
    }
    for (; b < b1; ++b) s += gpart[(long)b * kNumParams + p];
  }
  part[wave][lane] = s;
  __syncthreads();
  if (wave == 0 && p < kNumParams)
    grad[p] = (part[0][lane] + part[1][lane]) + (part[2][lane] + part[3][lane]);
}

__global__ void __launch_bounds__(256)
    adam_kernel(float* __restrict__ params, float* __restrict__ m, float* __restrict__ v,
                const float* __restrict__ grad, float lr, float beta1, float beta2, float eps,
                float c1, float c2) {
  const int p = blockIdx.x * 256 + threadIdx.x;
  if (p >= kNumParams) return;
  const float gr = grad[p];
  const float mm = beta1 * m[p] + (1.0f - beta1) * gr;
  const float vv = beta2 * v[p] + (1.0f - beta2) * gr * gr;
  m[p] = mm;
  v[p] = vv;
  params[p] -= lr * (mm / c1) / (sqrtf(vv / c2) + eps);
}

// BF16 copies of the convolution weights in the matrix-core layouts:
// w1b[co][16] (tap 15 = 0), w2b and w3b by weight_index.
__global__ void __launch_bounds__(256)
    pack_kernel(const float* __restrict__ params, unsigned short* __restrict__ w1b,
                unsigned short* __restrict__ w2b, unsigned short* __restrict__ w3b) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i < kC1 * 16) {
    const int co = i / 16, k = i % 16;
    w1b[i] = k < 15 ? f2bf(params[kOffW1 + co * 15 + k]) : 0;
  }
  if (i < kC2 * 15 * kC1)
    w2b[weight_index<kC1>(i / (15 * kC1), i / kC1 % 15, i % kC1)] = f2bf(params[kOffW2 + i]);
  if (i < kC3 * 15 * kC2)
    w3b[weight_index<kC2>(i / (15 * kC2), i / kC2 % 15, i % kC2)] = f2bf(params[kOffW3 + i]);
}

// ---------------------------------------------------------------------------
// Gating: the channel tiles of the search that overlap a flagged block, in
// ascending order (one workgroup; list[0..*count)).
__device__ __forceinline__ void tile_list_body(const float* __restrict__ logits, int nblk,
                                               float threshold, int N, int tile_width,
                                               int* __restrict__ list, int* __restrict__ count,
                                               int* __restrict__ flagged, int* sums) {
  const int ntiles = (N + tile_width - 1) / tile_width;
  const int per = (ntiles + 1023) / 1024;
  const int t0 = threadIdx.x * per;
  int n = 0;
  for (int t = t0; t < min(ntiles, t0 + per); ++t) {
    const long c0 = (long)t * tile_width, c1 = min((long)N, c0 + tile_width) - 1;
    const int b0 = (int)(c0 / kBlockChannels), b1 = (int)min((long)nblk - 1, c1 / kBlockChannels);
    bool f = false;
    for (int bb = b0; bb <= b1; ++bb) f = f || (logits[bb] > threshold);
    n += f;
  }
  sums[threadIdx.x] = n;
  __syncthreads();
  for (int off = 1; off < 1024; off <<= 1) {
    const int v = (int)threadIdx.x >= off ? sums[threadIdx.x - off] : 0;
    __syncthreads();
    sums[threadIdx.x] += v;
    __syncthreads();
  }
  int w = sums[threadIdx.x] - n;
  for (int t = t0; t < min(ntiles, t0 + per); ++t) {
    const long c0 = (long)t * tile_width, c1 = min((long)N, c0 + tile_width) - 1;
    const int b0 = (int)(c0 / kBlockChannels), b1 = (int)min((long)nblk - 1, c1 / kBlockChannels);
    bool f = false;
    for (int bb = b0; bb <= b1; ++bb) f = f || (logits[bb] > threshold);
    if (f) list[w++] = t;
  }
  if (threadIdx.x == 1023) count[0] = sums[1023];
  if (flagged) {
    __syncthreads();
    if (threadIdx.x == 0) {
      int nf = 0;
      for (int bb = 0; bb < nblk; ++bb) nf += logits[bb] > threshold;
      flagged[0] = nf;
    }
  }
}

__global__ void __launch_bounds__(1024)
    tile_list_kernel(const float* __restrict__ logits, int nblk, float threshold, int N,
                     int tile_width, int* __restrict__ list, int* __restrict__ count,
                     int* __restrict__ flagged) {
  __shared__ int sums[1024];
  tile_list_body(logits, nblk, threshold, N, tile_width, list, count, flagged, sums);
}

// Several channels (one workgroup each; channel c's logits at logits + c * nblk).
__global__ void __launch_bounds__(1024)
    tile_list_set_kernel(const float* __restrict__ logits, int nblk, float threshold, int N,
                         int tile_width, FrontSet fs) {
  __shared__ int sums[1024];
  const int c = blockIdx.x;
  tile_list_body(logits + (long)c * nblk, nblk, threshold, N, tile_width, fs.list[c],
                 fs.count[c], fs.count[c] + 1, sums);
}

}  // namespace

hipError_t launch_pool(const void* x, int dtype, long stride, int nblk, const float* stats,
                       unsigned short* z, hipStream_t stream) {
  const long n = (long)nblk * kRows * kPooled;
  const dim3 grid((unsigned)((n + 255) / 256)), block(256);
  switch (dtype) {
    case 0:
      hipLaunchKernelGGL(pool_kernel<float>, grid, block, 0, stream, (const float*)x, stride,
                         nblk, stats, z);
      break;
    case 1:
      hipLaunchKernelGGL(pool_kernel<_Float16>, grid, block, 0, stream, (const _Float16*)x,
                         stride, nblk, stats, z);
      break;
    case 2:
      hipLaunchKernelGGL(pool_kernel<unsigned short>, grid, block, 0, stream,
                         (const unsigned short*)x, stride, nblk, stats, z);
      break;
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

hipError_t launch_pool_set(const FrontSet& fs, int n, int dtype, long stride, int nblk,
                           unsigned short* z, hipStream_t stream) {
  if (n < 1 || n > kMaxFusedSet) return hipErrorInvalidValue;
  const long per = (long)nblk * kRows * kPooled;
  const dim3 grid((unsigned)((per + 255) / 256), n), block(256);
  switch (dtype) {
    case 0:
      hipLaunchKernelGGL(pool_set_kernel<float>, grid, block, 0, stream, fs, stride, nblk, z);
      break;
    case 1:
      hipLaunchKernelGGL(pool_set_kernel<_Float16>, grid, block, 0, stream, fs, stride, nblk, z);
      break;
    case 2:
      hipLaunchKernelGGL(pool_set_kernel<unsigned short>, grid, block, 0, stream, fs, stride,
                         nblk, z);
      break;
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

hipError_t launch_forward(const Weights& w, const unsigned short* z, int B, Acts& a,
                          float* logits, int* argmax, hipStream_t stream) {
  hipLaunchKernelGGL(forward_kernel, dim3(kW3 / kTile3 * B), dim3(kForwardThreads), 0, stream, z,
                     w.w1b, w.w2b, w.w3b, w.params, a.h1, a.h2, a.h3);
  hipLaunchKernelGGL(head_kernel, dim3(B), dim3(256), 0, stream, a.h3, w.params, logits, argmax);
  return hipGetLastError();
}

hipError_t launch_gradient(const Weights& w, const unsigned short* z, const float* labels, int B,
                           float pos_weight, Acts& a, float* logits, int* argmax, float* dz,
                           float* gpart, float* grad, float* loss, hipStream_t stream) {
  hipError_t e = launch_forward(w, z, B, a, logits, argmax, stream);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(loss_kernel, dim3(1), dim3(256), 0, stream, logits, labels, B, pos_weight,
                     dz, loss);
  hipLaunchKernelGGL(backward_kernel, dim3(B), dim3(kBackThreads), 0, stream, z, a.h1, a.h2, a.h3, argmax,
                     dz, w.params, gpart);
  hipLaunchKernelGGL(reduce_grad_kernel, dim3((kNumParams + 63) / 64), dim3(256), 0, stream,
                     gpart, B, grad);
  return hipGetLastError();
}

hipError_t launch_adam(Weights& w, float* m, float* v, const float* grad, float lr, int step,
                       hipStream_t stream) {
  const float b1 = 0.9f, b2 = 0.999f;
  const float c1 = 1.0f - powf(b1, (float)step), c2 = 1.0f - powf(b2, (float)step);
  hipLaunchKernelGGL(adam_kernel, dim3((kNumParams + 255) / 256), dim3(256), 0, stream, w.params,
                     m, v, grad, lr, b1, b2, 1e-8f, c1, c2);
  return launch_pack(w, stream);
}

hipError_t launch_pack(Weights& w, hipStream_t stream) {
  hipLaunchKernelGGL(pack_kernel, dim3((kC3 * 15 * kC2 + 255) / 256), dim3(256), 0, stream,
                     w.params, w.w1b, w.w2b, w.w3b);
  return hipGetLastError();
}

hipError_t launch_tile_list_set(const float* logits, int nblk, float threshold, int N,
                                int tile_width, const FrontSet& fs, int n, hipStream_t stream) {
  if (n < 1 || n > kMaxFusedSet) return hipErrorInvalidValue;
  hipLaunchKernelGGL(tile_list_set_kernel, dim3(n), dim3(1024), 0, stream, logits, nblk,
                     threshold, N, tile_width, fs);
  return hipGetLastError();
}

hipError_t launch_tile_list(const float* logits, int nblk, float threshold, int N, int tile_width,
                            int* list, int* count, int* flagged, hipStream_t stream) {
  hipLaunchKernelGGL(tile_list_kernel, dim3(1), dim3(1024), 0, stream, logits, nblk, threshold,
                     N, tile_width, list, count, flagged);
  return hipGetLastError();
}

}  // namespace pn
}  // namespace sc
