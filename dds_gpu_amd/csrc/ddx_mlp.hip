// The trick-count net: an MLP that predicts NS tricks for (deal, strain, leader), used to seed
// the null-window search (DDX_SEED_CERT). Trained and evaluated on gfx950 by the kernels here:
// BF16 weights and activations, FP32 accumulation on the matrix cores
// (v_mfma_f32_16x16x16bf16_1k), FP32 master weights and Adam.
//
// Input (217 features, padded to 224): one-hot owner (4) of each of the 52 cards, one-hot
// strain (5), one-hot leader (4). Hidden: 256 ReLU, 256 ReLU. Output: 14 logits (padded to
// 16; the pad logits are masked) for NS tricks 0..13. 125,198 trained parameters.
//
// Parameter vector (FP32, this order; weights stored out x in, row-major):
//   W1t [256][224] | b1 [256] | W2t [256][256] | b2 [256] | W3t [16][256] | b3 [16]
// Input columns 217..223 and output rows 14..15 stay zero.
#include <hip/hip_runtime.h>
#include <math.h>
#include <stdio.h>
#include <string.h>

#include <algorithm>
#include <new>
#include <random>
#include <vector>

#include "ddx.h"
#include "ddx_dispatch.h"
#include "ddx_init.h"
#include "ddx_internal.h"
#include "ddx_resident.h"

#define HIPCHECK(x)                                                                 \
  do {                                                                              \
    hipError_t e_ = (x);                                                            \
    if (e_ != hipSuccess) {                                                         \
      ddx_set_error("%s:%d %s: %s", __FILE__, __LINE__, #x, hipGetErrorString(e_)); \
      return DDX_E_HIP;                                                             \
    }                                                                               \
  } while (0)

namespace {

constexpr int IN = 224, IN_USED = 217, H = 256, OUT = 16, OUT_USED = 14;
constexpr size_t OFF_W1 = 0, OFF_B1 = OFF_W1 + (size_t)H * IN, OFF_W2 = OFF_B1 + H,
                 OFF_B2 = OFF_W2 + (size_t)H * H, OFF_W3 = OFF_B2 + H, OFF_B3 = OFF_W3 + (size_t)OUT * H,
                 NPARAM = OFF_B3 + OUT;

typedef unsigned short bf16;
typedef short v4s __attribute__((ext_vector_type(4)));
typedef float v4f __attribute__((ext_vector_type(4)));

// Round to nearest even (v_cvt_pk_bf16_f32).
typedef __bf16 v2b __attribute__((ext_vector_type(2)));
typedef float v2f __attribute__((ext_vector_type(2)));
__device__ inline unsigned two_bf16(float a, float b) {
  union {
    v2b b;
    unsigned u;
  } x;
  x.b = __builtin_convertvector((v2f{a, b}), v2b);
  return x.u;
}
__device__ inline bf16 to_bf16(float f) { return (bf16)two_bf16(f, 0.f); }

// ---------------------------------------------------------------------------------------
// Data layout. Every layer is computed transposed, D = W * Y^T, with 16x16 tiles of
// v_mfma_f32_16x16x16_bf16 (wave64, q = lane / 16): lane l holds A[l%16][4q..4q+3],
// B[4q..4q+3][l%16] and D[4q+r][l%16], r = 0..3. A tile of D -- four consecutive neurons of one
// sample per lane -- is therefore already the next layer's B operand: activations go from layer
// to layer in registers or through LDS as 8-byte fragments, with no transposition.
//
// A unit of work is 16 deals x one strain: its four declarers' samples are four tiles of 16
// columns, one deal per column, so that the last 16 inputs (strain and leader, the only ones that
// differ between a deal's 20 samples) are the same for a whole tile. The cards' part of the first
// layer is summed once per 16 deals and finished per tile by one more MFMA: the k order of every
// sum is that of a plain matrix product, so results do not depend on the path.
//
// Weights are kept as fragments ("packed", below): fragment (mt, kc) of a matrix is 64 lanes x 4
// elements, one coalesced 512-byte load.
constexpr int KC1 = IN / 16, KCH = H / 16;  // k chunks of the first and of the hidden layers
constexpr size_t PK1 = 0, PK2 = PK1 + (size_t)H * IN, PK3 = PK2 + (size_t)H * H, PK2T = PK3 + (size_t)OUT * H,
                 PK3T = PK2T + (size_t)H * H, NPACK = PK3T + (size_t)H * OUT;

// Position of element (row, k) in the packed form of a matrix of `chunks` k chunks.
__device__ inline size_t packed(int row, int k, int chunks) {
  return ((size_t)((row >> 4) * chunks + (k >> 4)) * 64 + (row & 15) + 16 * ((k >> 2) & 3)) * 4 + (k & 3);
}

__device__ inline v4s as_v4s(uint2 u) {
  union {
    uint2 u;
    v4s s;
  } x;
  x.u = u;
  return x.s;
}
__device__ inline v4f mfma16(uint2 a, uint2 b, v4f c) {
  return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(as_v4s(a), as_v4s(b), c, 0, 0, 0);
}
__device__ inline uint2 pack4(float a, float b, float c, float d) {
  return make_uint2(two_bf16(a, b), two_bf16(c, d));
}
__device__ inline uint2 frag(const bf16* w, size_t matrix, int index, int lane) {
  return ((const uint2*)(w + matrix))[(size_t)index * 64 + lane];
}
// bf16 of relu(z + bias), the next layer's operand.
__device__ inline uint2 relu_frag(v4f z, float4 bias) {
  const float a = z[0] + bias.x, b = z[1] + bias.y, c = z[2] + bias.z, d = z[3] + bias.w;
  return pack4(a > 0.f ? a : 0.f, b > 0.f ? b : 0.f, c > 0.f ? c : 0.f, d > 0.f ? d : 0.f);
}
// bf16 of the gradient g where the activation y (bf16) is not zero.
__device__ inline uint2 mask_frag(v4f g, uint2 y) {
  return pack4(y.x & 0xFFFFu ? g[0] : 0.f, y.x >> 16 ? g[1] : 0.f, y.y & 0xFFFFu ? g[2] : 0.f, y.y >> 16 ? g[3] : 0.f);
}

// One-hot owners of card 4 * kc + q, the B fragment of input chunk kc < 13, from the deal's hands.
__device__ inline uint2 card_frag(const uint64_t h[4], int kc, int q) {
  const int c = 4 * kc + q, at = 16 * (c / 13) + c % 13;
  return make_uint2((unsigned)((h[0] >> at) & 1) * 0x3F80u | (unsigned)((h[1] >> at) & 1) * 0x3F800000u,
                    (unsigned)((h[2] >> at) & 1) * 0x3F80u | (unsigned)((h[3] >> at) & 1) * 0x3F800000u);
}
// One-hot strain (inputs 208..212) and leader (213..216) of a declarer: input chunk 13.
__device__ inline uint2 strain_frag(int strain, int decl, int q) {
  const int i = strain - 4 * q, j = 5 + ((decl + 1) & 3) - 4 * q;  // places in this lane's four
  unsigned e[4];
#pragma unroll
  for (int k = 0; k < 4; k++) e[k] = k == i || k == j ? 0x3F80u : 0u;
  return make_uint2(e[0] | e[1] << 16, e[2] | e[3] << 16);
}

// The activations of one unit in LDS, as fragments. Two k chunks lie side by side, so that a
// lane reads both with one 16-byte access (8-byte ones reach half the LDS's rate).
struct UnitLayer {
  uint4 f[4][KCH / 2][64];
  __device__ inline uint2& at(int sample, int kc, int lane) { return ((uint2*)&f[sample][kc >> 1][lane])[kc & 1]; }
  __device__ inline uint2 at(int sample, int kc, int lane) const {
    return ((const uint2*)&f[sample][kc >> 1][lane])[kc & 1];
  }
  __device__ inline void two(int sample, int kc2, int lane, uint2 b[2]) const {
    const uint4 v = f[sample][kc2][lane];
    b[0] = make_uint2(v.x, v.y);
    b[1] = make_uint2(v.z, v.w);
  }
};
struct UnitLds {
  UnitLayer h1, h2;
};

// Wave `w` of four takes neuron tiles 4w..4w+3. The cards' part of the first layer for the 16
// deals whose hands the lanes hold.
template <int UNROLL>
__device__ inline void layer1_cards(const bf16* W, const uint64_t h[4], int w, int lane, v4f base[4]) {
#pragma unroll
  for (int i = 0; i < 4; i++) base[i] = v4f{0.f, 0.f, 0.f, 0.f};
#pragma unroll UNROLL
  for (int kc = 0; kc < KC1 - 1; kc++) {
    const uint2 b = card_frag(h, kc, lane >> 4);
#pragma unroll
    for (int i = 0; i < 4; i++) base[i] = mfma16(frag(W, PK1, (4 * w + i) * KC1 + kc, lane), b, base[i]);
  }
}
// A wave's two tiles of a 256 x 256 product for the four samples of a unit, from weights in
// registers.
__device__ inline void load_held(const bf16* W, size_t matrix, int w, int lane, uint2 a[2][KCH]) {
#pragma unroll
  for (int i = 0; i < 2; i++)
#pragma unroll
    for (int kc = 0; kc < KCH; kc++) a[i][kc] = frag(W, matrix, (2 * w + i) * KCH + kc, lane);
}
__device__ inline void hidden_held(const uint2 a[2][KCH], const UnitLayer& y, int lane, v4f z[2][4]) {
#pragma unroll
  for (int i = 0; i < 2; i++)
#pragma unroll
    for (int s = 0; s < 4; s++) z[i][s] = v4f{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int kc = 0; kc < KCH; kc += 2) {
    uint2 b[4][2];
#pragma unroll
    for (int s = 0; s < 4; s++) y.two(s, kc / 2, lane, b[s]);
#pragma unroll
    for (int j = 0; j < 2; j++)
#pragma unroll
      for (int i = 0; i < 2; i++)
#pragma unroll
        for (int s = 0; s < 4; s++) z[i][s] = mfma16(a[i][kc + j], b[s][j], z[i][s]);
  }
}

// Logits (without bias) of one sample tile: D[class][deal]; w3: the output layer's fragments.
__device__ inline v4f layer3(const uint2* w3, int sample, int lane, const UnitLayer& y) {
  v4f z = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int kc = 0; kc < KCH; kc += 2) {
    uint2 b[2];
    y.two(sample, kc / 2, lane, b);
    z = mfma16(w3[kc * 64 + lane], b[0], z);
    z = mfma16(w3[(kc + 1) * 64 + lane], b[1], z);
  }
  return z;
}

// The most likely class of every deal of a tile: the first of the largest logits.
__device__ inline int argmax16(v4f z, const float* b3, int lane) {
  const int q = lane >> 4;
  float mx = -1e30f;
  int arg = 0;
#pragma unroll
  for (int r = 0; r < 4; r++) {
    const int j = 4 * q + r;
    const float v = z[r] + b3[j];
    if (j < OUT_USED && v > mx) {
      mx = v;
      arg = j;
    }
  }
#pragma unroll
  for (int m = 16; m <= 32; m <<= 1) {
    const float o = __shfl_xor(mx, m);
    const int oa = __shfl_xor(arg, m);
    if (o > mx || (o == mx && oa < arg)) {
      mx = o;
      arg = oa;
    }
  }
  return arg;
}

__device__ inline void load_hands(const uint64_t* hands, long long deal, bool in, uint64_t h[4]) {
#pragma unroll
  for (int i = 0; i < 4; i++) h[i] = in ? hands[4 * deal + i] : 0;
}

// Seeds of one sample tile (16 deals, one strain and declarer) per block: few deals, or any number
// while a stream is open. Latency counts, so a deal's 20 samples run on 20 CUs; and so do registers
// and LDS: this kernel has to fit beside a stream's (16 KB of LDS, so that the compiler does not
// pad the registers to the occupancy that the LDS would allow).
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(8, 8))) void predict_tile_kernel(
    const uint64_t* hands, long long n, const bf16* W, const float* p, uint8_t* seeds) {
  __shared__ uint2 h1[KCH][64], h2[KCH][64];
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63, q = lane >> 4;
  const long long deal = (long long)(blockIdx.x / 20) * 16 + (lane & 15);
  const int sample = blockIdx.x % 20;
  v4f z[4];
  {
    uint64_t h[4];
    load_hands(hands, deal, deal < n, h);
    layer1_cards<2>(W, h, w, lane, z);
  }
  const uint2 t = strain_frag(sample / 4, sample % 4, q);
#pragma unroll
  for (int i = 0; i < 4; i++) {
    const int mt = 4 * w + i;
    const float4 bias = *(const float4*)(p + OFF_B1 + 16 * mt + 4 * q);
    h1[mt][lane] = relu_frag(mfma16(frag(W, PK1, mt * KC1 + KC1 - 1, lane), t, z[i]), bias);
    z[i] = v4f{0.f, 0.f, 0.f, 0.f};
  }
  __syncthreads();
#pragma unroll 2
  for (int kc = 0; kc < KCH; kc++) {
    const uint2 b = h1[kc][lane];
#pragma unroll
    for (int i = 0; i < 4; i++) z[i] = mfma16(frag(W, PK2, (4 * w + i) * KCH + kc, lane), b, z[i]);
  }
#pragma unroll
  for (int i = 0; i < 4; i++) {
    const int mt = 4 * w + i;
    h2[mt][lane] = relu_frag(z[i], *(const float4*)(p + OFF_B2 + 16 * mt + 4 * q));
  }
  __syncthreads();
  if (w != 0) return;
  v4f y = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 4
  for (int kc = 0; kc < KCH; kc++) y = mfma16(frag(W, PK3, kc, lane), h2[kc][lane], y);
  const int arg = argmax16(y, p + OFF_B3, lane);
  if (q == 0 && deal < n) seeds[20 * deal + sample] = (uint8_t)arg;
}

// Seeds of many deals: one persistent block of eight waves per CU, each wave with its two tiles of
// the hidden weights in registers (64 VGPRs) for good, so that the loop reads only activations,
// from LDS. The three layers of successive units run in one phase between two barriers -- the
// first of unit t + 1, the second of unit t, the output of unit t - 1, each layer's activations in
// two LDS buffers -- so that one wave's conversions overlap another's matrix instructions. Bound by
// the matrix cores (16x16x16 tiles at half their peak rate, which keeps every sum in the order of
// the plain product). 100,000 deals: 14.6 ms with a kernel per layer and its activations in
// memory (11 GB of traffic), 0.39 ms here, launch and wait included.
__global__ __launch_bounds__(512, 1) void predict_kernel(const uint64_t* hands, long long n, const bf16* W,
                                                         const float* p, uint8_t* seeds) {
  __shared__ UnitLayer h1[2], h2[2];
  __shared__ uint2 w3[KCH * 64];
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63, q = lane >> 4;
  for (int i = threadIdx.x; i < KCH * 64; i += 512) w3[i] = ((const uint2*)(W + PK3))[i];
  uint2 a2[2][KCH], a1[2];
  float4 bias1[2], bias2[2];
  load_held(W, PK2, w, lane, a2);
#pragma unroll
  for (int i = 0; i < 2; i++) {
    const int mt = 2 * w + i;
    a1[i] = frag(W, PK1, mt * KC1 + KC1 - 1, lane);
    bias1[i] = *(const float4*)(p + OFF_B1 + 16 * mt + 4 * q);
    bias2[i] = *(const float4*)(p + OFF_B2 + 16 * mt + 4 * q);
  }
  const long long groups = (n + 15) / 16;
  const int mine = (int)((groups - blockIdx.x + gridDim.x - 1) / gridDim.x), units = 5 * mine;
  auto deal_of = [&](int unit) { return ((long long)blockIdx.x + (long long)(unit / 5) * gridDim.x) * 16 + (lane & 15); };
  uint64_t h[4];  // the hands of the next group to start
  load_hands(hands, deal_of(0), deal_of(0) < n, h);
  v4f base[2];
  // First layer of unit t into buffer t & 1.
  auto first = [&](int t) {
    if (t % 5 == 0) {
#pragma unroll
      for (int i = 0; i < 2; i++) base[i] = v4f{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int kc = 0; kc < KC1 - 1; kc++) {
        const uint2 b = card_frag(h, kc, q);
#pragma unroll
        for (int i = 0; i < 2; i++) base[i] = mfma16(frag(W, PK1, (2 * w + i) * KC1 + kc, lane), b, base[i]);
      }
      load_hands(hands, deal_of(t + 5), deal_of(t + 5) < n, h);  // arrives while five units are computed
    }
#pragma unroll
    for (int s = 0; s < 4; s++) {
      const uint2 b = strain_frag(t % 5, s, q);
#pragma unroll
      for (int i = 0; i < 2; i++) h1[t & 1].at(s, 2 * w + i, lane) = relu_frag(mfma16(a1[i], b, base[i]), bias1[i]);
    }
  };
  first(0);
  __syncthreads();
#pragma unroll 1
  for (int t = 0; t <= units; t++) {
    if (t > 0 && w < 4) {  // the output of unit t - 1, declarer w
      const int arg = argmax16(layer3(w3, w, lane, h2[(t - 1) & 1]), p + OFF_B3, lane);
      const long long deal = deal_of(t - 1);
      if (q == 0 && deal < n) seeds[20 * deal + 4 * ((t - 1) % 5) + w] = (uint8_t)arg;
    }
    if (t == units) break;
    if (t + 1 < units) first(t + 1);
    v4f z[2][4];
    hidden_held(a2, h1[t & 1], lane, z);
#pragma unroll
    for (int i = 0; i < 2; i++)
#pragma unroll
      for (int s = 0; s < 4; s++) h2[t & 1].at(s, 2 * w + i, lane) = relu_frag(z[i][s], bias2[i]);
    __syncthreads();
  }
}

// What a training step keeps of its samples for the weight gradients, as bf16 [neuron][row]: rows
// are samples, unit by unit (64 rows: 4 declarers x 16 deals), rows = 64 * units. And the cards of
// each 16 deals as a bit per deal and input, [16 deals][224].
struct TrainActs {
  bf16 *h1, *h2, *d2, *d1, *dz;
  unsigned short* x;
  long long rows;
};
// Stores neuron tile mt of a unit's activations: eight rows of one neuron per lane, gathered from
// the fragments the wave itself wrote (its LDS accesses take effect in order), 64 bytes per neuron
// and store instead of four stores of two bytes per lane.
__device__ inline void store_tile(const UnitLayer& y, int mt, int lane, bf16* t, long long rows, long long row0) {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  const int c = lane & 15, q = lane >> 4;  // neuron 16 * mt + c, rows 8q..8q+7 of a pair of samples
#pragma unroll
  for (int pair = 0; pair < 2; pair++) {
    // Row 8q + r: sample 2 * pair + (q >> 1), deal 8 * (q & 1) + r, held by lane 16 * (c / 4) + deal.
    const bf16* f = (const bf16*)&y.f[2 * pair + (q >> 1)][mt >> 1][16 * (c >> 2) + 8 * (q & 1)] + 4 * (mt & 1) + (c & 3);
    unsigned v[8];
#pragma unroll
    for (int r = 0; r < 8; r++) v[r] = f[8 * r];
    *(uint4*)(t + (size_t)(16 * mt + c) * rows + row0 + 32 * pair + 8 * q) =
        make_uint4(v[0] | v[1] << 16, v[2] | v[3] << 16, v[4] | v[5] << 16, v[6] | v[7] << 16);
  }
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
}

// The cards' inputs of 16 deals as bits (the four q agree): wave w writes suit w / 2, two owners.
__device__ inline void write_cards(const uint64_t h[4], int w, int lane, unsigned short* x) {
#pragma unroll 2
  for (int f = 0; f < 26; f++) {
    const int o = 2 * (w & 1) + (f & 1), rank = f >> 1;
    const uint64_t hh = w & 1 ? (f & 1 ? h[3] : h[2]) : (f & 1 ? h[1] : h[0]);
    const unsigned m = (unsigned)__ballot((hh >> (16 * (w >> 1) + rank)) & 1) & 0xFFFFu;
    if (lane == 0) x[4 * (13 * (w >> 1) + rank) + o] = (unsigned short)m;
  }
}
// Loss of a unit and the gradient of its logits zs, by one wave; lane = row of the unit: declarer
// lane / 16, deal lane % 16.
__device__ inline void unit_loss(const float* p, const uint8_t* tables, long long deal, bool in, int strain, long long n,
                                 int lane, const float (&zs)[64][17], bf16 (&dzs)[64][OUT], const TrainActs& t,
                                 long long row0, float* stats) {
  const int decl = lane >> 4;
  int y = -1;
  if (in) {
    const int tr = tables[20 * deal + 4 * strain + decl];  // 255: unknown
    y = tr == 255 ? -1 : (decl & 1) == 0 ? tr : 13 - tr;
  }
  float z[OUT];
  float mx = -1e30f;
  int arg = 0;
#pragma unroll
  for (int j = 0; j < OUT_USED; j++) {
    z[j] = zs[lane][j] + p[OFF_B3 + j];
    if (z[j] > mx) {
      mx = z[j];
      arg = j;
    }
  }
  float sum = 0.f, zy = 0.f;
#pragma unroll
  for (int j = 0; j < OUT_USED; j++) {
    sum += expf(z[j] - mx);
    if (j == y) zy = z[j];
  }
  float loss = 0.f, right = 0.f;
  if (y >= 0) {
    loss = logf(sum) - (zy - mx);
    right = arg == y ? 1.f : 0.f;
  }
  const float inv = y >= 0 ? 1.f / (float)(20 * n) : 0.f;
#pragma unroll
  for (int j = 0; j < OUT; j++) {
    const float pj = j < OUT_USED ? expf(z[j < OUT_USED ? j : 0] - mx) / sum : 0.f;
    const bf16 d = to_bf16((j == y ? pj - 1.f : pj) * inv);
    dzs[lane][j] = d;
    t.dz[(size_t)j * t.rows + row0 + lane] = d;
  }
  for (int m = 32; m; m >>= 1) {
    loss += __shfl_xor(loss, m);
    right += __shfl_xor(right, m);
  }
  if (lane == 0) {
    atomicAdd(&stats[0], loss);
    atomicAdd(&stats[1], right);
  }
}

// Forward, loss and the gradients of the activations, one unit per block. order: the deals of the
// batch (null: 0..n-1). The mean runs over 20 * n samples; unknown labels (255) add no loss and
// get a zero gradient. Softmax cross-entropy over the 14 used logits: dZ = (p - y) / M; the loss
// and the count of right argmax predictions are summed into stats[0], stats[1].
__global__ __launch_bounds__(512, 1) void train_unit_kernel(const uint64_t* hands, const uint8_t* tables,
                                                            const long long* order, long long n, const bf16* W,
                                                            const float* p, TrainActs t, float* stats) {
  __shared__ UnitLds u;
  __shared__ float zs[64][17];
  __shared__ bf16 dzs[64][OUT];
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63, q = lane >> 4, col = lane & 15;
  const long long g = blockIdx.x / 5, at = g * 16 + col;
  const int strain = blockIdx.x % 5;
  const bool in = at < n;
  const long long deal = in ? (order ? order[at] : at) : 0;
  const long long row0 = (long long)blockIdx.x * 64;
  uint2 a2[2][KCH], a3[2];
  float4 bias2[2];
  v4f zz[2][4];
  {
    // All of the first layer's weights are on their way before the hands are. (Read chunk by chunk,
    // each waited for memory: 29 us a step of 256 deals, 27 so.)
    uint2 a1[2][KC1];
#pragma unroll
    for (int kc = 0; kc < KC1; kc++)
#pragma unroll
      for (int i = 0; i < 2; i++) a1[i][kc] = frag(W, PK1, (2 * w + i) * KC1 + kc, lane);
    float4 bias1[2];
#pragma unroll
    for (int i = 0; i < 2; i++) {
      bias1[i] = *(const float4*)(p + OFF_B1 + 16 * (2 * w + i) + 4 * q);
      bias2[i] = *(const float4*)(p + OFF_B2 + 16 * (2 * w + i) + 4 * q);
    }
    uint64_t h[4];
    load_hands(hands, deal, in, h);
    load_held(W, PK2, w, lane, a2);  // arrive during the first layer
#pragma unroll
    for (int i = 0; i < 2; i++) a3[i] = frag(W, PK3T, 2 * w + i, lane);
    if (strain == 0) write_cards(h, w, lane, t.x + g * IN);
    v4f base[2];
#pragma unroll
    for (int i = 0; i < 2; i++) base[i] = v4f{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int kc = 0; kc < KC1 - 1; kc++) {
      const uint2 b = card_frag(h, kc, q);
#pragma unroll
      for (int i = 0; i < 2; i++) base[i] = mfma16(a1[i][kc], b, base[i]);
    }
#pragma unroll
    for (int i = 0; i < 2; i++) {
      const int mt = 2 * w + i;
#pragma unroll
      for (int s = 0; s < 4; s++) u.h1.at(s, mt, lane) = relu_frag(mfma16(a1[i][KC1 - 1], strain_frag(strain, s, q), base[i]), bias1[i]);
    }
  }
  __syncthreads();
  hidden_held(a2, u.h1, lane, zz);
  load_held(W, PK2T, w, lane, a2);  // arrive during the loss
#pragma unroll
  for (int i = 0; i < 2; i++) {
    const int mt = 2 * w + i;
#pragma unroll
    for (int s = 0; s < 4; s++) u.h2.at(s, mt, lane) = relu_frag(zz[i][s], bias2[i]);
  }
  __syncthreads();
  if (w < 4) {
    const v4f z = layer3((const uint2*)(W + PK3), w, lane, u.h2);
#pragma unroll
    for (int r = 0; r < 4; r++) zs[16 * w + col][4 * q + r] = z[r];
  }
  __syncthreads();
  if (w == 0) unit_loss(p, tables, deal, in, strain, n, lane, zs, dzs, t, row0, stats);
  __syncthreads();
  // Gradient of the second hidden layer, in place of its activations.
#pragma unroll
  for (int i = 0; i < 2; i++) {
    const int mt = 2 * w + i;
    store_tile(u.h2, mt, lane, t.h2, t.rows, row0);
#pragma unroll
    for (int s = 0; s < 4; s++) {
      const uint2 dz = *(const uint2*)&dzs[16 * s + col][4 * q];
      u.h2.at(s, mt, lane) = mask_frag(mfma16(a3[i], dz, v4f{0.f, 0.f, 0.f, 0.f}), u.h2.at(s, mt, lane));
    }
    store_tile(u.h2, mt, lane, t.d2, t.rows, row0);
  }
  __syncthreads();
  // Gradient of the first.
  hidden_held(a2, u.h2, lane, zz);
#pragma unroll
  for (int i = 0; i < 2; i++) {
    const int mt = 2 * w + i;
    store_tile(u.h1, mt, lane, t.h1, t.rows, row0);
#pragma unroll
    for (int s = 0; s < 4; s++) u.h1.at(s, mt, lane) = mask_frag(zz[i][s], u.h1.at(s, mt, lane));
    store_tile(u.h1, mt, lane, t.d1, t.rows, row0);
  }
}

// The same on a device on which a stream is open (ddx_resident.h), in the registers that it
// leaves: four waves, each doing the work of waves w and w + 4 above one after the other, the weights
// read as they are needed. Every sum is the same, in the same order. (Gradients of 333 deals take
// 166 us beside a stream so, 130 us with the kernel above and no stream.)
__device__ inline void hidden_streamed(const bf16* W, size_t matrix, int w, const UnitLayer& y, int lane, v4f z[2][4]) {
#pragma unroll
  for (int i = 0; i < 2; i++)
#pragma unroll
    for (int s = 0; s < 4; s++) z[i][s] = v4f{0.f, 0.f, 0.f, 0.f};
#pragma unroll 1
  for (int kc = 0; kc < KCH; kc++) {
    uint2 a[2];
#pragma unroll
    for (int i = 0; i < 2; i++) a[i] = frag(W, matrix, (2 * w + i) * KCH + kc, lane);
#pragma unroll
    for (int s = 0; s < 4; s++) {
      const uint2 b = y.at(s, kc, lane);
#pragma unroll
      for (int i = 0; i < 2; i++) z[i][s] = mfma16(a[i], b, z[i][s]);
    }
  }
}
__global__ __launch_bounds__(256) __attribute__((amdgpu_num_vgpr(ddx::kRoomVgprs / 2))) void train_unit_small_kernel(
    const uint64_t* hands, const uint8_t* tables, const long long* order, long long n, const bf16* W, const float* p,
    TrainActs t, float* stats) {
  __shared__ UnitLds u;
  __shared__ float zs[64][17];
  __shared__ bf16 dzs[64][OUT];
  const int w4 = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63, q = lane >> 4, col = lane & 15;
  const long long g = blockIdx.x / 5, at = g * 16 + col;
  const int strain = blockIdx.x % 5;
  const bool in = at < n;
  const long long deal = in ? (order ? order[at] : at) : 0;
  const long long row0 = (long long)blockIdx.x * 64;
  v4f zz[2][4];
  {
    uint64_t h[4];
    load_hands(hands, deal, in, h);
#pragma unroll 1
    for (int w = w4; w < 8; w += 4) {
      if (strain == 0) write_cards(h, w, lane, t.x + g * IN);
      v4f base[2] = {v4f{0.f, 0.f, 0.f, 0.f}, v4f{0.f, 0.f, 0.f, 0.f}};
#pragma unroll 1
      for (int kc = 0; kc < KC1 - 1; kc++) {
        const uint2 b = card_frag(h, kc, q);
#pragma unroll
        for (int i = 0; i < 2; i++) base[i] = mfma16(frag(W, PK1, (2 * w + i) * KC1 + kc, lane), b, base[i]);
      }
#pragma unroll
      for (int i = 0; i < 2; i++) {
        const int mt = 2 * w + i;
        const uint2 a = frag(W, PK1, mt * KC1 + KC1 - 1, lane);
        const float4 bias = *(const float4*)(p + OFF_B1 + 16 * mt + 4 * q);
#pragma unroll
        for (int s = 0; s < 4; s++) u.h1.at(s, mt, lane) = relu_frag(mfma16(a, strain_frag(strain, s, q), base[i]), bias);
      }
    }
  }
  __syncthreads();
#pragma unroll 1
  for (int w = w4; w < 8; w += 4) {
    hidden_streamed(W, PK2, w, u.h1, lane, zz);
#pragma unroll
    for (int i = 0; i < 2; i++) {
      const int mt = 2 * w + i;
      const float4 bias = *(const float4*)(p + OFF_B2 + 16 * mt + 4 * q);
#pragma unroll
      for (int s = 0; s < 4; s++) u.h2.at(s, mt, lane) = relu_frag(zz[i][s], bias);
    }
  }
  __syncthreads();
  {
    const v4f z = layer3((const uint2*)(W + PK3), w4, lane, u.h2);
#pragma unroll
    for (int r = 0; r < 4; r++) zs[16 * w4 + col][4 * q + r] = z[r];
  }
  __syncthreads();
  if (w4 == 0) unit_loss(p, tables, deal, in, strain, n, lane, zs, dzs, t, row0, stats);
  __syncthreads();
#pragma unroll 1
  for (int mt = 2 * w4; mt < 16; mt += (mt & 1) ? 7 : 1) {
    const uint2 a = frag(W, PK3T, mt, lane);
    store_tile(u.h2, mt, lane, t.h2, t.rows, row0);
#pragma unroll
    for (int s = 0; s < 4; s++) {
      const uint2 dz = *(const uint2*)&dzs[16 * s + col][4 * q];
      u.h2.at(s, mt, lane) = mask_frag(mfma16(a, dz, v4f{0.f, 0.f, 0.f, 0.f}), u.h2.at(s, mt, lane));
    }
    store_tile(u.h2, mt, lane, t.d2, t.rows, row0);
  }
  __syncthreads();
#pragma unroll 1
  for (int w = w4; w < 8; w += 4) {
    hidden_streamed(W, PK2T, w, u.h2, lane, zz);
#pragma unroll
    for (int i = 0; i < 2; i++) {
      const int mt = 2 * w + i;
      store_tile(u.h1, mt, lane, t.h1, t.rows, row0);
#pragma unroll
      for (int s = 0; s < 4; s++) u.h1.at(s, mt, lane) = mask_frag(zz[i][s], u.h1.at(s, mt, lane));
      store_tile(u.h1, mt, lane, t.d1, t.rows, row0);
    }
  }
}

// Weight gradients: products over the samples, D[out][in] = sum over rows of d[out][row] y[in][row],
// 32 rows per v_mfma_f32_16x16x32_bf16 (lane l: row l%16 of the operand, k = 8q..8q+7). One wave
// takes a 64 x 64 block of one matrix (36 blocks in all: 16 of W1t, 16 of W2t, 4 of W3t) over its
// share of the units (blockIdx.y of gridDim.y) and writes it to its own partial gradient vector;
// the next kernel sums the shares. Bias gradients are the products with a vector of ones: for b1
// that is unused input 217, set to one here; for b2 and b3 an extra column of the first block.
typedef __bf16 v8b __attribute__((ext_vector_type(8)));
__device__ inline v4f mfma32(uint4 a, uint4 b, v4f c) {
  union {
    uint4 u;
    v8b b;
  } x, y;
  x.u = a;
  y.u = b;
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(x.b, y.b, c, 0, 0, 0);
}
__device__ inline unsigned two_bits(unsigned m) {  // bits 0 and 1 as two bf16 ones
  return (m & 1) * 0x3F80u | ((m >> 1) & 1) * 0x3F800000u;
}

// R: tiles of 16 outputs that a wave takes: 4, the whole block, or 1, with four times the waves, in
// the registers that an open stream leaves.
template <int R>
__device__ inline void wgrad(const TrainActs& t, int units, float* parts) {
  const int task = blockIdx.x / (4 / R), i0 = R * (blockIdx.x % (4 / R)), lane = threadIdx.x, q = lane >> 4, col = lane & 15;
  float* out = parts + (size_t)blockIdx.y * NPARAM;
  const int u0 = (int)((long long)units * blockIdx.y / gridDim.y), u1 = (int)((long long)units * (blockIdx.y + 1) / gridDim.y);
  const int matrix = task < 16 ? 0 : task < 32 ? 1 : 2;           // W1t, W2t, W3t
  const int ob = matrix == 2 ? 0 : (task & 15) >> 2, ib = task & 3;  // 64-blocks of outputs, inputs
  const bf16* A = matrix == 0 ? t.d1 : matrix == 1 ? t.d2 : t.dz;
  const bf16* B = matrix == 1 ? t.h1 : t.h2;
  const int mts = matrix == 2 ? 1 : 4, nts = matrix == 0 && ib == 3 ? 2 : 4;
  v4f acc[R][4], ones_acc[R];
#pragma unroll
  for (int i = 0; i < R; i++) {
    ones_acc[i] = v4f{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int j = 0; j < 4; j++) acc[i][j] = v4f{0.f, 0.f, 0.f, 0.f};
  }
  const uint4 ones = make_uint4(0x3F803F80u, 0x3F803F80u, 0x3F803F80u, 0x3F803F80u);
  const bool bias = matrix != 0 && ib == 0;
  uint4 x[4];  // W1t: the cards of the current 16 deals
  int group = -1;
  for (int un = u0; un < u1; un++) {
    if (matrix == 0 && un / 5 != group) {
      group = un / 5;
#pragma unroll
      for (int j = 0; j < 4; j++) {
        const int f = 64 * ib + 16 * j + col;
        const unsigned m = f < 208 ? (unsigned)t.x[(size_t)group * IN + f] >> (8 * (q & 1)) : 0u;
        x[j] = make_uint4(two_bits(m), two_bits(m >> 2), two_bits(m >> 4), two_bits(m >> 6));
      }
    }
#pragma unroll
    for (int half = 0; half < 2; half++) {  // declarers 2 * half, 2 * half + 1
      const size_t row = (size_t)un * 64 + 32 * half + 8 * q;
      uint4 a[R], b[4];
#pragma unroll
      for (int i = 0; i < R; i++)
        if (i0 + i < mts) a[i] = *(const uint4*)(A + (size_t)(64 * ob + 16 * (i0 + i) + col) * t.rows + row);
#pragma unroll
      for (int j = 0; j < 4; j++) {
        if (j >= nts) continue;
        if (matrix != 0) {
          b[j] = *(const uint4*)(B + (size_t)(64 * ib + 16 * j + col) * t.rows + row);
        } else {
          b[j] = x[j];
          if (ib == 3 && j == 1) {  // inputs 208..223: strain, leader, the ones
            const int leader = (2 * half + (q >> 1) + 1) & 3;
            const bool on = col == un % 5 || col == 5 + leader || col == 9;
            b[j] = on ? ones : make_uint4(0, 0, 0, 0);
          }
        }
      }
#pragma unroll
      for (int i = 0; i < R; i++) {
        if (i0 + i >= mts) continue;
#pragma unroll
        for (int j = 0; j < 4; j++)
          if (j < nts) acc[i][j] = mfma32(a[i], b[j], acc[i][j]);
        if (bias) ones_acc[i] = mfma32(a[i], ones, ones_acc[i]);
      }
    }
  }
  const size_t off = matrix == 0 ? OFF_W1 : matrix == 1 ? OFF_W2 : OFF_W3;
  const int width = matrix == 0 ? IN : H;
#pragma unroll
  for (int i = 0; i < R; i++) {
    if (i0 + i >= mts) continue;
#pragma unroll
    for (int r = 0; r < 4; r++) {
      const int o = 64 * ob + 16 * (i0 + i) + 4 * q + r;
#pragma unroll
      for (int j = 0; j < 4; j++)
        if (j < nts) out[off + (size_t)o * width + 64 * ib + 16 * j + col] = acc[i][j][r];
      if (bias && col == 0) out[(matrix == 1 ? OFF_B2 : OFF_B3) + o] = ones_acc[i][r];
    }
  }
}
__global__ __launch_bounds__(64) void wgrad_kernel(TrainActs t, int units, float* parts) { wgrad<4>(t, units, parts); }
__global__ __launch_bounds__(64) void wgrad_small_kernel(TrainActs t, int units, float* parts) { wgrad<1>(t, units, parts); }

// Writes parameter i's bf16 value to the packed matrices it belongs to.
__device__ inline void pack_param(long long i, float v, bf16* w) {
  const bf16 b = to_bf16(v);
  if (i < (long long)OFF_B1) {
    w[PK1 + packed((int)(i / IN), (int)(i % IN), KC1)] = b;
  } else if (i >= (long long)OFF_W2 && i < (long long)OFF_B2) {
    const int o = (int)((i - OFF_W2) / H), k = (int)((i - OFF_W2) % H);
    w[PK2 + packed(o, k, KCH)] = b;
    w[PK2T + packed(k, o, KCH)] = b;
  } else if (i >= (long long)OFF_W3 && i < (long long)OFF_B3) {
    const int o = (int)((i - OFF_W3) / H), k = (int)((i - OFF_W3) % H);
    w[PK3 + packed(o, k, KCH)] = b;
    w[PK3T + packed(k, o, 1)] = b;
  }
}
__global__ void pack_kernel(const float* p, bf16* w) {
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < (long long)NPARAM) pack_param(i, p[i], w);
}

// Sums the shares of the weight gradients into g, and for a training step (m != null) applies
// Adam and refreshes the packed weights.
struct Adam {
  float *p, *m, *v;
  bf16* w;
  float lr, b1, b2, c1, c2, eps;
};
__global__ __launch_bounds__(256) void reduce_kernel(const float* parts, int shares, float* g, Adam ad) {
  // 64 parameters per block, every fourth share per group of 64 threads.
  __shared__ float sums[4][64];
  const int lane = threadIdx.x & 63, quarter = threadIdx.x >> 6;
  const long long i = (long long)blockIdx.x * 64 + lane;
  const bool in = i < (long long)NPARAM;
  // b1's gradient is W1t's input 217; the padding's gradients are zero.
  const bool pad = (i < (long long)OFF_B1 && i % IN >= IN_USED) ||
                   (i >= (long long)OFF_W3 && i < (long long)OFF_B3 && (i - (long long)OFF_W3) / H >= OUT_USED) ||
                   i >= (long long)OFF_B3 + OUT_USED;
  const long long at = i >= (long long)OFF_B1 && i < (long long)OFF_W2 ? (i - (long long)OFF_B1) * IN + IN_USED : i;
  float s = 0.f;
  if (in && !pad)
#pragma unroll 8
    for (int k = quarter; k < shares; k += 4) s += parts[(size_t)k * NPARAM + at];
  sums[quarter][lane] = s;
  __syncthreads();
  if (quarter != 0 || !in) return;
  s = (sums[0][lane] + sums[1][lane]) + (sums[2][lane] + sums[3][lane]);
  g[i] = s;
  if (!ad.m) return;
  const float mi = ad.b1 * ad.m[i] + (1.f - ad.b1) * s, vi = ad.b2 * ad.v[i] + (1.f - ad.b2) * s * s;
  ad.m[i] = mi;
  ad.v[i] = vi;
  const float pi = ad.p[i] - ad.lr * (mi / ad.c1) / (sqrtf(vi / ad.c2) + ad.eps);
  ad.p[i] = pi;
  pack_param(i, pi, ad.w);
}

__global__ void fill_f32_kernel(float* p, long long n, float v) {
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = v;
}

inline unsigned blocks(long long n, int t = 256) { return (unsigned)((n + t - 1) / t); }

}  // namespace

struct ddx_mlp {
  int device = 0;
  float* p = nullptr;  // fp32 master parameters
  float* g = nullptr;  // gradients
  float* m = nullptr;  // Adam moments
  float* v = nullptr;
  bf16* w = nullptr;  // packed bf16 copy of p (weights used by the matrix products)
  long long steps = 0;
  // Training: activations for `cap` units, `shares` partial gradients, per-step statistics.
  long long cap = 0, stats_cap = 0, order_cap = 0;
  int shares = 0;
  bf16* acts = nullptr;
  unsigned short* x = nullptr;
  float *parts = nullptr, *stats = nullptr;
  long long* d_order = nullptr;
  uint64_t* d_hands = nullptr;
  uint8_t* d_tables = nullptr;
  long long host_cap = 0;
  uint8_t* d_seeds = nullptr;  // predictions for ddx_mlp_predict_host
  long long seeds_cap = 0;
  uint64_t* pin_hands = nullptr;  // mapped host memory for predictions of a few deals
  uint8_t* pin_seeds = nullptr;
  int cus = 0;
  hipStream_t s = nullptr;
  hipEvent_t used = nullptr;  // the last prediction on a caller's stream
  std::vector<void*> outgrown;  // buffers to free when no stream is open
};

constexpr long long kPinDeals = 64;  // deals that ddx_mlp_predict_host passes through mapped memory
constexpr int kMaxShares = 32;

static long long units_of(long long deals) { return (deals + 15) / 16 * 5; }

// Gives up a buffer that is to be replaced by a larger one. hipFree waits for the whole device, so
// beside an open stream, whose kernel does not end, the buffer is kept for a later time.
template <class T>
static void give_up(ddx_mlp* h, T*& p) {
  std::lock_guard<std::mutex> lock(ddx::resident().mu);  // no stream opens meanwhile
  bool keep = ddx::resident().streams(h->device) != 0;
  if (keep && p) {
    try {
      h->outgrown.push_back(p);
    } catch (const std::bad_alloc&) {
      keep = false;
    }
  }
  if (!keep) {
    if (p) (void)hipFree(p);
    for (void* q : h->outgrown) (void)hipFree(q);
    h->outgrown.clear();
  }
  p = nullptr;
}
// The size for a buffer that holds `cap` and has to hold n: few growths, and what is outgrown beside a
// stream together no more than the buffer.
static long long grown(long long cap, long long n) { return n < 2 * cap ? 2 * cap : n; }

// Buffers of a training step of `deals` deals (rounded up to 16).
static int train_reserve(ddx_mlp* h, long long deals, long long steps) {
  const long long units = units_of(deals);
  if (units > h->cap) {
    give_up(h, h->acts);
    give_up(h, h->x);
    h->cap = 0;
    HIPCHECK(hipMalloc(&h->acts, (size_t)units * 64 * (4 * H + OUT) * 2));
    HIPCHECK(hipMalloc(&h->x, (size_t)units / 5 * IN * 2));
    h->cap = units;
  }
  if (!h->parts) HIPCHECK(hipMalloc(&h->parts, (size_t)kMaxShares * NPARAM * 4));
  if (steps > h->stats_cap) {
    give_up(h, h->stats);
    steps = grown(h->stats_cap, steps);
    h->stats_cap = 0;
    HIPCHECK(hipMalloc(&h->stats, (size_t)steps * 8));
    h->stats_cap = steps;
  }
  return DDX_OK;
}

static int mlp_stage_host(ddx_mlp* h, const uint64_t* hands, const uint8_t* tables, long long n) {
  if (n > h->host_cap) {
    give_up(h, h->d_hands);
    give_up(h, h->d_tables);
    const long long cap = grown(h->host_cap, n);
    h->host_cap = 0;
    HIPCHECK(hipMalloc(&h->d_hands, cap * 32));
    HIPCHECK(hipMalloc(&h->d_tables, cap * 20));
    h->host_cap = cap;
  }
  HIPCHECK(hipMemcpyAsync(h->d_hands, hands, n * 32, hipMemcpyHostToDevice, h->s));
  if (tables) HIPCHECK(hipMemcpyAsync(h->d_tables, tables, n * 20, hipMemcpyHostToDevice, h->s));
  return DDX_OK;
}

// Whether large kernels may be launched on the net's device (ddx_resident.h); held while they are.
struct LargeKernels {
  std::unique_lock<std::mutex> lock;
  bool allowed = false;
  LargeKernels(const ddx_mlp* h, bool wanted) : lock(ddx::resident().mu, std::defer_lock) {
    if (!wanted) return;
    lock.lock();
    allowed = ddx::resident().streams(h->device) == 0;
  }
};

// Gradients of one batch of n deals of the staged ones (order: which, null = the first n) into
// h->g, its loss and accuracy sums into stats; with lr != 0 the Adam step on them.
static void train_step(ddx_mlp* h, const long long* order, long long n, float* stats, bool adam, float lr) {
  const long long units = units_of(n), rows = units * 64;
  TrainActs t;
  t.h1 = h->acts;
  t.h2 = t.h1 + (size_t)H * rows;
  t.d2 = t.h2 + (size_t)H * rows;
  t.d1 = t.d2 + (size_t)H * rows;
  t.dz = t.d1 + (size_t)H * rows;
  t.x = h->x;
  t.rows = rows;
  const LargeKernels large(h, true);
  if (large.allowed)
    hipLaunchKernelGGL(train_unit_kernel, dim3((unsigned)units), dim3(512), 0, h->s, h->d_hands, h->d_tables, order, n,
                       h->w, h->p, t, stats);
  else
    hipLaunchKernelGGL(train_unit_small_kernel, dim3((unsigned)units), dim3(256), 0, h->s, h->d_hands, h->d_tables, order,
                       n, h->w, h->p, t, stats);
  // A wave reads one share after the other with little else to do: many short shares, but two units
  // or more in each for the 16 KB of partial results it writes.
  const int shares = (int)(units / 2 > kMaxShares ? kMaxShares : units / 2);
  if (large.allowed) hipLaunchKernelGGL(wgrad_kernel, dim3(36, shares), dim3(64), 0, h->s, t, (int)units, h->parts);
  else hipLaunchKernelGGL(wgrad_small_kernel, dim3(144, shares), dim3(64), 0, h->s, t, (int)units, h->parts);
  Adam ad{h->p, nullptr, h->v, h->w, lr, 0.9f, 0.999f, 1.f, 1.f, 1e-8f};
  if (adam) {
    h->steps++;
    ad.m = h->m;
    ad.c1 = 1.f - powf(ad.b1, (float)h->steps);
    ad.c2 = 1.f - powf(ad.b2, (float)h->steps);
  }
  hipLaunchKernelGGL(reduce_kernel, dim3(blocks(NPARAM, 64)), dim3(256), 0, h->s, h->parts, shares, h->g, ad);
}

static void clear_stats(ddx_mlp* h, long long steps) {
  hipLaunchKernelGGL(fill_f32_kernel, dim3(blocks(2 * steps)), dim3(256), 0, h->s, h->stats, 2 * steps, 0.f);
}

static void sync_bf16(ddx_mlp* h) {
  hipLaunchKernelGGL(pack_kernel, dim3(blocks(NPARAM)), dim3(256), 0, h->s, h->p, h->w);
}

// Seeds of n deals on stream s. Few deals are spread over a block per sample tile; from 512 deals
// (640 blocks) on, the persistent kernel is faster although its blocks have less than a group of
// 16 deals per CU then. Beside a stream, and in a capture, whose replays may be beside one, any
// number of deals goes tile by tile: 100,000 deals in 2.1 ms beside a stream, 0.39 ms otherwise.
static void launch_predict(const ddx_mlp* h, hipStream_t s, const uint64_t* d_hands, long long n, uint8_t* d_seeds,
                           bool captured) {
  const long long groups = (n + 15) / 16;
  const LargeKernels large(h, groups >= 32 && !captured);
  if (large.allowed) {
    hipLaunchKernelGGL(predict_kernel, dim3((unsigned)(groups < h->cus ? groups : h->cus)), dim3(512), 0, s, d_hands, n,
                       h->w, h->p, d_seeds);
  } else {
    hipLaunchKernelGGL(predict_tile_kernel, dim3((unsigned)(20 * groups)), dim3(256), 0, s, d_hands, n, h->w, h->p, d_seeds);
  }
}

constexpr long long kNoAllocDeals = 256;  // the most that ddx_mlp_predict_noalloc takes

extern "C" int ddx_mlp_create(int device, uint64_t seed, ddx_mlp** out) {
  if (!out) return DDX_E_ARG;
  int ndev = 0;
  if (hipGetDeviceCount(&ndev) != hipSuccess || ndev <= device) {
    ddx_set_error("ddx_mlp_create: no HIP device %d", device);
    return DDX_E_NODEV;
  }
  HIPCHECK(hipSetDevice(device));
  ddx_mlp* h = new (std::nothrow) ddx_mlp;
  if (!h) return DDX_E_NOMEM;
  h->device = device;
  HIPCHECK(hipStreamCreateWithFlags(&h->s, hipStreamNonBlocking));
  HIPCHECK(hipEventCreateWithFlags(&h->used, hipEventDisableTiming));
  HIPCHECK(hipMalloc(&h->p, NPARAM * 4));
  HIPCHECK(hipMalloc(&h->g, NPARAM * 4));
  HIPCHECK(hipMalloc(&h->m, NPARAM * 4));
  HIPCHECK(hipMalloc(&h->v, NPARAM * 4));
  HIPCHECK(hipMalloc(&h->w, NPACK * 2));
  HIPCHECK(hipDeviceGetAttribute(&h->cus, hipDeviceAttributeMultiprocessorCount, device));
  // He initialisation of the used weights, zero biases and padding.
  std::vector<float> p(NPARAM, 0.f);
  std::mt19937_64 rng(seed);
  ddx::init_matrix(p.data() + OFF_W1, H, IN, H, IN_USED, IN_USED, rng);
  ddx::init_matrix(p.data() + OFF_W2, H, H, H, H, H, rng);
  ddx::init_matrix(p.data() + OFF_W3, OUT, H, OUT_USED, H, H, rng);
  HIPCHECK(hipMemcpyAsync(h->p, p.data(), NPARAM * 4, hipMemcpyHostToDevice, h->s));
  HIPCHECK(hipMemsetAsync(h->m, 0, NPARAM * 4, h->s));
  HIPCHECK(hipMemsetAsync(h->v, 0, NPARAM * 4, h->s));
  sync_bf16(h);
  HIPCHECK(hipStreamSynchronize(h->s));
  *out = h;
  return DDX_OK;
}

extern "C" void ddx_mlp_destroy(ddx_mlp* h) {
  if (!h) return;
  (void)hipSetDevice(h->device);
  if (h->s) (void)hipStreamSynchronize(h->s);
  if (h->pin_hands) (void)hipHostFree(h->pin_hands);
  if (h->pin_seeds) (void)hipHostFree(h->pin_seeds);
  void* ptrs[] = {h->p,     h->g,     h->m,       h->v,       h->w,        h->acts,   h->x,
                  h->parts, h->stats, h->d_order, h->d_hands, h->d_tables, h->d_seeds};
  for (void* q : ptrs)
    if (q) (void)hipFree(q);
  for (void* q : h->outgrown) (void)hipFree(q);
  if (h->s) (void)hipStreamDestroy(h->s);
  if (h->used) (void)hipEventDestroy(h->used);
  delete h;
}

extern "C" int64_t ddx_mlp_param_count(void) { return (int64_t)NPARAM; }

extern "C" int ddx_mlp_params(ddx_mlp* h, float* buf, int get) {
  if (!h || !buf) return DDX_E_ARG;
  HIPCHECK(hipSetDevice(h->device));
  // On the handle's stream, behind the predictions that still read the parameters (ddx_mlp_predict).
  if (get) {
    HIPCHECK(hipMemcpyAsync(buf, h->p, NPARAM * 4, hipMemcpyDeviceToHost, h->s));
  } else {
    HIPCHECK(hipMemcpyAsync(h->p, buf, NPARAM * 4, hipMemcpyHostToDevice, h->s));
    sync_bf16(h);
    HIPCHECK(hipGetLastError());
  }
  HIPCHECK(hipStreamSynchronize(h->s));
  return DDX_OK;
}

extern "C" int ddx_mlp_grads(ddx_mlp* h, const uint64_t* hands, const uint8_t* tables, int64_t n,
                             float* grads, float* loss_acc) {
  if (!h || !hands || !tables || n <= 0) return DDX_E_ARG;
  HIPCHECK(hipSetDevice(h->device));
  int rc;
  if ((rc = train_reserve(h, n, 1)) != DDX_OK || (rc = mlp_stage_host(h, hands, tables, n)) != DDX_OK) return rc;
  clear_stats(h, 1);
  train_step(h, nullptr, n, h->stats, false, 0.f);
  HIPCHECK(hipGetLastError());
  HIPCHECK(hipStreamSynchronize(h->s));
  if (grads) HIPCHECK(hipMemcpy(grads, h->g, NPARAM * 4, hipMemcpyDeviceToHost));
  if (loss_acc) {
    float st[2];
    HIPCHECK(hipMemcpy(st, h->stats, 8, hipMemcpyDeviceToHost));
    loss_acc[0] = st[0] / (float)(n * 20);
    loss_acc[1] = st[1] / (float)(n * 20);
  }
  return DDX_OK;
}

extern "C" int ddx_mlp_train(ddx_mlp* h, const uint64_t* hands, const uint8_t* tables, int64_t n,
                             int epochs, int batch_deals, float lr, uint64_t shuffle_seed,
                             float* loss_acc) {
  if (!h || !hands || !tables || n <= 0 || epochs < 1 || batch_deals < 1) {
    ddx_set_error("ddx_mlp_train: bad arguments");
    return DDX_E_ARG;
  }
  HIPCHECK(hipSetDevice(h->device));
  int rc;
  const long long steps = n / batch_deals;  // per epoch; the rest of the last batch is left out
  if ((rc = train_reserve(h, batch_deals, steps > 0 ? steps : 1)) != DDX_OK) return rc;
  // The whole set goes to the device once; a batch is a range of the epoch's order, so a step is
  // three kernels and nothing else, and the host waits at the end only.
  if ((rc = mlp_stage_host(h, hands, tables, n)) != DDX_OK) return rc;
  if (n > h->order_cap) {
    give_up(h, h->d_order);
    const long long cap = grown(h->order_cap, n);
    h->order_cap = 0;
    HIPCHECK(hipMalloc(&h->d_order, cap * 8));
    h->order_cap = cap;
  }
  std::vector<long long> order(n);
  for (long long i = 0; i < n; i++) order[i] = i;
  std::mt19937_64 rng(shuffle_seed);
  for (int e = 0; e < epochs; e++) {
    std::shuffle(order.begin(), order.end(), rng);
    HIPCHECK(hipMemcpyAsync(h->d_order, order.data(), n * 8, hipMemcpyHostToDevice, h->s));
    if (steps) clear_stats(h, steps);
    for (long long b = 0; b < steps; b++)
      train_step(h, h->d_order + b * batch_deals, batch_deals, h->stats + 2 * b, true, lr);
    HIPCHECK(hipGetLastError());
    HIPCHECK(hipStreamSynchronize(h->s));  // before the order changes on the host
  }
  if (loss_acc && steps > 0) {
    std::vector<float> st(2 * steps);
    HIPCHECK(hipMemcpy(st.data(), h->stats, steps * 8, hipMemcpyDeviceToHost));
    double loss_sum = 0, acc_sum = 0;
    const double samples = 20.0 * batch_deals * steps;
    for (long long b = 0; b < steps; b++) {
      loss_sum += st[2 * b];
      acc_sum += st[2 * b + 1];
    }
    loss_acc[0] = (float)(loss_sum / samples);
    loss_acc[1] = (float)(acc_sum / samples);
  }
  return DDX_OK;
}

extern "C" int ddx_mlp_predict(ddx_mlp* h, const uint64_t* d_hands, int64_t n, uint8_t* d_seeds,
                               void* stream) {
  if (!h || !d_hands || !d_seeds || n < 0) return DDX_E_ARG;
  HIPCHECK(hipSetDevice(h->device));
  hipStream_t s = stream ? (hipStream_t)stream : h->s;
  hipStreamCaptureStatus capture = hipStreamCaptureStatusNone;
  if (stream) HIPCHECK(hipStreamIsCapturing(s, &capture));
  const bool captured = capture != hipStreamCaptureStatusNone;
  if (n) launch_predict(h, s, d_hands, n, d_seeds, captured);
  HIPCHECK(hipGetLastError());
  if (!stream) {
    HIPCHECK(hipStreamSynchronize(h->s));
    return DDX_OK;
  }
  // Later work of the handle (training, new parameters) waits until these weights were read. A
  // capture leaves no work behind now, and the handle's stream must not be drawn into it.
  if (!captured) {
    HIPCHECK(hipEventRecord(h->used, s));
    HIPCHECK(hipStreamWaitEvent(h->s, h->used, 0));
  }
  return DDX_OK;
}

// ddx_mlp_predict for at most kNoAllocDeals deals, on the caller's stream (NULL: the null stream,
// and the call waits for the seeds). No prediction allocates or keeps activations in memory.
extern "C" int ddx_mlp_predict_noalloc(const ddx_mlp* h, const uint64_t* d_hands, int64_t n,
                                       uint8_t* d_seeds, void* stream) {
  if (!h || n < 0 || (n > 0 && (!d_hands || !d_seeds))) {
    ddx_set_error("ddx_mlp_predict_noalloc: bad arguments");
    return DDX_E_ARG;
  }
  if (n > kNoAllocDeals) {
    ddx_set_error("ddx_mlp_predict_noalloc: %lld deals exceed the %lld it takes", (long long)n, kNoAllocDeals);
    return DDX_E_ARG;
  }
  HIPCHECK(hipSetDevice(h->device));
  if (n == 0) return DDX_OK;
  launch_predict(h, (hipStream_t)stream, d_hands, n, d_seeds, false);
  HIPCHECK(hipGetLastError());
  if (!stream) HIPCHECK(hipStreamSynchronize(nullptr));
  return DDX_OK;
}

// Host in, host out. Everything runs on the handle's non-blocking stream and buffers are reused
// (no per-call allocation or free, which could wait for the whole device), so predictions can be
// made while a stream's persistent kernel runs (ddx_resident.h). A few deals pass through mapped
// host memory, which the kernel reads and writes itself: one launch and one wait instead of
// two copies more (one deal: 81 us with copies and five kernels).
extern "C" int ddx_mlp_predict_host(ddx_mlp* h, const uint64_t* hands, int64_t n, uint8_t* seeds) {
  if (!h || !hands || !seeds || n < 0) return DDX_E_ARG;
  HIPCHECK(hipSetDevice(h->device));
  int rc;
  if (n <= kPinDeals) {
    if (!h->pin_seeds) {
      if (!h->pin_hands) HIPCHECK(hipHostMalloc((void**)&h->pin_hands, kPinDeals * 32, hipHostMallocMapped));
      HIPCHECK(hipHostMalloc((void**)&h->pin_seeds, kPinDeals * 20, hipHostMallocMapped));
    }
    void *dh = nullptr, *ds = nullptr;
    HIPCHECK(hipHostGetDevicePointer(&dh, h->pin_hands, 0));
    HIPCHECK(hipHostGetDevicePointer(&ds, h->pin_seeds, 0));
    memcpy(h->pin_hands, hands, n * 32);
    if ((rc = ddx_mlp_predict(h, (const uint64_t*)dh, n, (uint8_t*)ds, nullptr)) != DDX_OK) return rc;
    memcpy(seeds, h->pin_seeds, n * 20);
    return DDX_OK;
  }
  if ((rc = mlp_stage_host(h, hands, nullptr, n)) != DDX_OK) return rc;
  if (n > h->seeds_cap) {
    give_up(h, h->d_seeds);
    const long long cap = grown(h->seeds_cap, n);
    h->seeds_cap = 0;
    HIPCHECK(hipMalloc(&h->d_seeds, cap * 20 + 16));
    h->seeds_cap = cap;
  }
  launch_predict(h, h->s, h->d_hands, n, h->d_seeds, false);
  HIPCHECK(hipGetLastError());
  HIPCHECK(hipMemcpyAsync(seeds, h->d_seeds, n * 20, hipMemcpyDeviceToHost, h->s));
  HIPCHECK(hipStreamSynchronize(h->s));
  return DDX_OK;
}

// File: "DDXMLP1\0", int64 count, then count fp32 parameters.
extern "C" int ddx_mlp_save(ddx_mlp* h, const char* path) {
  std::vector<float> p(NPARAM);
  int rc = ddx_mlp_params(h, p.data(), 1);
  if (rc != DDX_OK) return rc;
  FILE* f = fopen(path, "wb");
  if (!f) {
    ddx_set_error("cannot write %s", path);
    return DDX_E_IO;
  }
  const int64_t cnt = NPARAM;
  bool ok = fwrite("DDXMLP1", 1, 8, f) == 8 && fwrite(&cnt, 8, 1, f) == 1 &&
            fwrite(p.data(), 4, NPARAM, f) == NPARAM;
  fclose(f);
  return ok ? DDX_OK : DDX_E_IO;
}

extern "C" int ddx_mlp_load(ddx_mlp* h, const char* path) {
  FILE* f = fopen(path, "rb");
  if (!f) {
    ddx_set_error("cannot open %s", path);
    return DDX_E_IO;
  }
  char magic[8];
  int64_t cnt = 0;
  std::vector<float> p(NPARAM);
  bool ok = fread(magic, 1, 8, f) == 8 && !memcmp(magic, "DDXMLP1", 8) && fread(&cnt, 8, 1, f) == 1 &&
            cnt == (int64_t)NPARAM && fread(p.data(), 4, NPARAM, f) == NPARAM;
  fclose(f);
  if (!ok) {
    ddx_set_error("%s is not a ddx MLP file", path);
    return DDX_E_IO;
  }
  return ddx_mlp_params(h, p.data(), 0);
}
