// ncs_convnet.hip -- the learned warm start: a 4-layer 3x3 conv net
// (2 -> 32 -> 32 -> 32 -> 1, ReLU after layers 1-3, 'same' zero padding
// inside each 16x16 tile) on BF16 MFMA with FP32 accumulation.
//
// Input channels per tile (normalisation shared with ncs_amd/warmstart.py):
//   mu = mean(d), sigma = sqrt(max(mu, 1) + mean(gamma)),
//   x0 = (d - mu) / sigma,  x1 = gamma / sigma^2;
// the net predicts y and the warm start is u0 = d + sigma * y.
//
// Convolution as GEMM on v_mfma_f32_16x16x32_bf16: for one output pixel row
// y and a block of 16 output channels,
//   D[cout][x] += sum_taps  W_tap[cout][cin] * In[cin][y + dy][x + dx],
// A = weights (pre-packed per tap and block: lane (g, i) holds cout i,
// K chunk 8g..8g+7), B = activations (lane (g, x) holds K chunk g of pixel
// x), D: lane (g, x) holds couts 4g..4g+3 of pixel x.  In the forward pass a
// tile's activations stay in registers (16 rows x 4 VGPRs per lane, see
// fwd_channel); the dx = -1 / +1 taps are DPP row_shr:1 / row_shl:1 of a
// row, whose zero fill at the row end is exactly the zero padding of the
// tile edge.  LDS holds the forward weight packs and biases, staged once
// per workgroup, and per wave the input grid / layer 4's partial sums.
//
// Backward: the data gradient is the same convolution with flipped,
// transposed weight packs; the weight gradient is a GEMM over pixels whose
// operands come from transposing LDS reads, kept in registers over all of a
// workgroup's tiles and added to memory once.
#include <algorithm>

#include "ncs_common.h"

namespace ncs {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef float f4 __attribute__((ext_vector_type(4)));
typedef int i4 __attribute__((ext_vector_type(4)));

constexpr int kCh = 32;
// FP32 parameter vector: per layer weights [cout][cin][3][3] then bias
constexpr int OFF_W1 = 0, OFF_B1 = 576, OFF_W2 = 608, OFF_B2 = 9824, OFF_W3 = 9856,
              OFF_B3 = 19072, OFF_W4 = 19104, OFF_B4 = 19392, N_PARAMS = 19393;
static_assert(N_PARAMS == NCS_NET_PARAMS, "parameter count");
// MFMA operand packs (64 lanes x 8 BF16 = 1 KB each)
constexpr int PK_L1 = 0;    // 2: layer 1 A, K = (tap, cin) padded to 32
constexpr int PK_L2 = 2;    // 18: layer 2 A, block * 9 + tap, K order fwd_channel
constexpr int PK_L3 = 20;   // 18
constexpr int PK_L4T = 38;  // 3: layer 4 B per dy, column n = dx (n < 3), K order fwd_channel
constexpr int PK_B4 = 41;   // 2: layer-4 data gradient, K = tap padded to 32
constexpr int PK_B3 = 43;   // 18: layer-3 data gradient (flipped, transposed)
constexpr int PK_B2 = 61;   // 18: layer-2 data gradient
constexpr int N_PACKS = 79;

// Forward activations live in registers.  With the K index k = 8g + e of a
// 32-channel layer's operand mapped to channel fwd_channel(k) (e < 4: 4g + e,
// else 16 + 4g + e - 4), the D fragments of a row's two output blocks at lane
// (g, x) -- couts 4g..4g+3, then 16 + 4g..16 + 4g + 3, of pixel x -- are in
// that order exactly the 8-channel fragment lane (g, x) supplies to the next
// layer.  A tile's activations are 16 rows x 4 VGPRs per lane and never cross
// lanes; the packs of layers 2-4 carry the permutation in their K order.
__host__ __device__ constexpr int fwd_channel(int k) {
  return (k & 7) < 4 ? 4 * (k >> 3) + (k & 7) : 12 + 4 * (k >> 3) + (k & 7);
}

__device__ __forceinline__ float w_at(const float *P, int off, int cin_n, int co, int ci,
                                      int tap) {
  return P[off + (co * cin_n + ci) * 9 + tap];
}

// Builds the BF16 A-operand packs [first, end) from the FP32 parameters: the
// forward pass takes those before PK_B4, the backward pass the others.  Also
// clears `sums` (may be NULL), the backward pass's gradient: with a launch of
// its own for that, and all packs for each pass, the backward call took 24.7 us
// where it takes 23.3 (128 tiles), 51.0 where it takes 49.3 (1024).
__global__ void net_pack_kernel(const float *__restrict__ P, __bf16 *__restrict__ packs, int first,
                                int end, float *__restrict__ sums) {
  const int item = blockIdx.x * blockDim.x + threadIdx.x;
  if (sums != nullptr && item < N_PARAMS) sums[item] = 0.0f;
  const int idx = first * 512 + item;
  if (idx >= end * 512) return;
  const int pack = idx >> 9, lane = (idx >> 3) & 63, e = idx & 7;
  const int i = lane & 15, g = lane >> 4;
  const int k = 8 * g + e;
  float v = 0.0f;
  if (pack < PK_L2) {  // layer 1: k = tap * 2 + cin
    const int co = 16 * (pack - PK_L1) + i;
    if (k < 18) v = w_at(P, OFF_W1, 2, co, k & 1, k >> 1);
  } else if (pack < PK_L3) {
    const int q = pack - PK_L2, co = 16 * (q / 9) + i;
    v = w_at(P, OFF_W2, kCh, co, fwd_channel(k), q % 9);
  } else if (pack < PK_L4T) {
    const int q = pack - PK_L3, co = 16 * (q / 9) + i;
    v = w_at(P, OFF_W3, kCh, co, fwd_channel(k), q % 9);
  } else if (pack < PK_B4) {  // B operand: lane (g, n) holds K = cin 8g..8g+7 of column n
    const int dy = pack - PK_L4T;
    if (i < 3) v = w_at(P, OFF_W4, kCh, 0, fwd_channel(k), dy * 3 + i);
  } else if (pack < PK_B3) {  // d(layer-3 act) from d(out): cout' = L4 cin, k = tap
    const int co = 16 * (pack - PK_B4) + i;
    if (k < 9) v = w_at(P, OFF_W4, kCh, 0, co, 8 - k);
  } else if (pack < PK_B2) {
    const int q = pack - PK_B3, co = 16 * (q / 9) + i;  // co = L3 cin, k = L3 cout
    v = w_at(P, OFF_W3, kCh, k, co, 8 - q % 9);
  } else {
    const int q = pack - PK_B2, co = 16 * (q / 9) + i;
    v = w_at(P, OFF_W2, kCh, k, co, 8 - q % 9);
  }
  packs[idx] = (__bf16)v;
}

__device__ __forceinline__ f4 mfma_bf16(i4 a, i4 b, f4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a),
                                                 __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}

template <int CTRL>
__device__ __forceinline__ i4 dpp_i4(i4 v) {
  i4 r;
  r.x = __builtin_amdgcn_update_dpp(0, v.x, CTRL, 0xF, 0xF, true);
  r.y = __builtin_amdgcn_update_dpp(0, v.y, CTRL, 0xF, 0xF, true);
  r.z = __builtin_amdgcn_update_dpp(0, v.z, CTRL, 0xF, 0xF, true);
  r.w = __builtin_amdgcn_update_dpp(0, v.w, CTRL, 0xF, 0xF, true);
  return r;
}
// A zero the optimiser cannot see through.  A loop-invariant address offset
// by it keeps its loads inside the per-tile loop (the operand packs of all
// four layers would not fit in registers beside the working set), and the
// address keeps its address space.
__device__ __forceinline__ int opaque_zero() {
  int z = 0;
  asm volatile("" : "+s"(z));
  return z;
}

// Orders one wave's LDS accesses across its lanes.  The LDS performs a
// wave's instructions in issue order, so only the compiler has to be kept
// from moving accesses across this point (wavefront-scope fences emit no
// instructions).
__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Accumulator start of the 16-channel block b: the bias of the output
// channels lane (g, x) holds (16 b + 4 g + r, r = 0..3).
__device__ __forceinline__ f4 bias4(const float *bias, int b, int lane) {
  const int g = lane >> 4;
  return (f4){bias[16 * b + 4 * g], bias[16 * b + 4 * g + 1], bias[16 * b + 4 * g + 2],
              bias[16 * b + 4 * g + 3]};
}

constexpr int kRowShr1 = 0x111;  // lane x <- lane x-1 in its row (0 at x = 0)
constexpr int kRowShl1 = 0x101;  // lane x <- lane x+1 in its row (0 at x = 15)

// Two floats as packed BF16 (round to nearest even), low half first.
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float f2 __attribute__((ext_vector_type(2)));
typedef short s2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ int bf16_pair(float lo, float hi) {
  const f2 v = {lo, hi};
  return __builtin_bit_cast(int, __builtin_convertvector(v, bf16x2));
}

// ReLU of a packed BF16 pair, clamping the halves as signed 16-bit integers
// at 0: a BF16 with its sign bit set is a negative int16 and a positive one
// keeps its order, so this equals rounding after the ReLU (negative values,
// -0 included, become +0).
__device__ __forceinline__ int relu_pair(float lo, float hi) {
  const s2 z = {0, 0};
  const s2 h = __builtin_bit_cast(s2, bf16_pair(lo, hi));
  return __builtin_bit_cast(int, __builtin_elementwise_max(h, z));
}

// ReLU of one row's two block accumulators as a BF16 register row.
__device__ __forceinline__ i4 relu_row(f4 a0, f4 a1) {
  i4 r;
  r.x = relu_pair(a0.x, a0.y);
  r.y = relu_pair(a0.z, a0.w);
  r.z = relu_pair(a1.x, a1.y);
  r.w = relu_pair(a1.z, a1.w);
  return r;
}

// A data gradient's four channels of one pixel as BF16, zero where the
// activations `act` (BF16, the same channels) are not positive.
typedef int i2v __attribute__((ext_vector_type(2)));
typedef short s4v __attribute__((ext_vector_type(4)));
__device__ __forceinline__ i2v relu_masked(f4 v, i2v act) {
  const bf16x4 a = __builtin_bit_cast(bf16x4, act);
  return (i2v){bf16_pair((float)a.x > 0.0f ? v.x : 0.0f, (float)a.y > 0.0f ? v.y : 0.0f),
               bf16_pair((float)a.z > 0.0f ? v.z : 0.0f, (float)a.w > 0.0f ? v.w : 0.0f)};
}

// A register row written as row y of a [256][32] BF16 buffer in the
// standard channel order (the activations kept for the backward pass).  Lane
// (g, x) holds channels 4g.. and 16 + 4g.. of pixel x; exchanged with the
// lane group next to it (the row swap trades the second half of an even group
// for the first half of the odd one), every lane has eight channels in a row,
// 16 (g & 1) + 8 (g >> 1).., and a wave's store is one stretch of 1 KB
// (8000 tiles, 393 MB of activations: 108 -> 96 us; two stores of 8 bytes a lane
// before).
__device__ __forceinline__ void store_row_std(__bf16 *dst, int y, int lane, i4 v) {
  const int x = lane & 15, g = lane >> 4;
  const auto a = __builtin_amdgcn_permlane16_swap((unsigned int)v.x, (unsigned int)v.z, false,
                                                  false);
  const auto b = __builtin_amdgcn_permlane16_swap((unsigned int)v.y, (unsigned int)v.w, false,
                                                  false);
  __bf16 *const px = dst + (y * 16 + x) * kCh + 16 * (g & 1) + 8 * (g >> 1);
  *reinterpret_cast<i4 *>(px) = (i4){(int)a[0], (int)b[0], (int)a[1], (int)b[1]};
}

// Layer 1 (2 -> 32 channels), K = tap * 2 + cin padded to 32.  The inputs sit
// in LDS as an 18 x 18 grid of (x0, x1) BF16 pairs with a zero border, so
// lane (g, x) reads its K = 8g..8g+7 (taps 4g..4g+3) of row y as four pairs
// at fixed offsets; taps past 8 read the zero border column of the row.
// Rounded once when it is written, a pair is not converted again for each of
// the nine taps that read it.
__device__ __forceinline__ int in_pad_offset(int tap, int x) {
  return tap < 9 ? (tap / 3) * 18 + x + tap % 3 : 0;
}

template <class Keep>
__device__ __forceinline__ void layer_in2(const int *in_pad, const i4 *packs,
                                          const float *bias, int lane, i4 (&act)[16],
                                          Keep keep) {
  const i4 A0 = packs[lane], A1 = packs[64 + lane];
  const f4 c0 = bias4(bias, 0, lane), c1 = bias4(bias, 1, lane);
  const int x = lane & 15, g = lane >> 4;
  int off[4];
#pragma unroll
  for (int j = 0; j < 4; j++) off[j] = in_pad_offset(4 * g + j, x);
#pragma unroll
  for (int y = 0; y < 16; y++) {
    i4 B;
#pragma unroll
    for (int j = 0; j < 4; j++) B[j] = in_pad[y * 18 + off[j]];
    act[y] = relu_row(mfma_bf16(A0, B, c0), mfma_bf16(A1, B, c1));
    keep(y, act[y]);
  }
}

// A 32 -> 32 channel layer in place over the register rows, two output rows
// per step (four independent accumulation chains: two rows x two blocks).
// Input rows y - 1 .. y + 2 and their dx = -1 / +1 shifts (DPP row_shr:1 /
// row_shl:1, whose zero fill at the row end is the tile's zero padding) are
// held as values when rows y and y + 1 are overwritten; rows y + 1 and y + 2
// carry over to the next step, so each row is shifted once per layer.
template <class Keep>
__device__ __forceinline__ void layer32(i4 (&act)[16], const i4 *packs_in, const float *bias_in,
                                        int lane, Keep keep) {
  const int z0 = opaque_zero();
  const i4 *packs = packs_in + z0;
  const float *bias = bias_in + z0;
  i4 A[2][9];
  // in the order of their first use, so that the first products need not wait
  // for the last of them
  constexpr int order[9] = {3, 0, 4, 1, 5, 2, 6, 7, 8};
#pragma unroll
  for (int i = 0; i < 9; i++)
#pragma unroll
    for (int b = 0; b < 2; b++)
      A[b][order[i]] = packs[(b * 9 + order[i]) * 64 + lane];
  const f4 c0 = bias4(bias, 0, lane), c1 = bias4(bias, 1, lane);
  const i4 z = {0, 0, 0, 0};
  i4 C[4], L[4], R[4];  // rows y - 1 .. y + 2: centre, dx = -1, dx = +1
  C[0] = L[0] = R[0] = z;
  C[1] = act[0];
  L[1] = dpp_i4<kRowShr1>(C[1]);
  R[1] = dpp_i4<kRowShl1>(C[1]);
#pragma unroll
  for (int y = 0; y < 16; y += 2) {
    C[2] = act[y + 1];
    L[2] = dpp_i4<kRowShr1>(C[2]);
    R[2] = dpp_i4<kRowShl1>(C[2]);
    if (y + 2 < 16) {
      C[3] = act[y + 2];
      L[3] = dpp_i4<kRowShr1>(C[3]);
      R[3] = dpp_i4<kRowShl1>(C[3]);
    }
    f4 acc[2][2] = {{c0, c1}, {c0, c1}};
#pragma unroll
    for (int q = 0; q < 4; q++) {  // input row y - 1 + q
      if ((q == 0 && y == 0) || (q == 3 && y + 2 >= 16)) continue;  // zero rows
#pragma unroll
      for (int dx = 0; dx < 3; dx++) {
        const i4 in = dx == 0 ? L[q] : (dx == 1 ? C[q] : R[q]);
#pragma unroll
        for (int o = 0; o < 2; o++) {  // output row y + o: dy = q - o
          const int dy = q - o;
          if (dy < 0 || dy > 2) continue;
#pragma unroll
          for (int b = 0; b < 2; b++) acc[o][b] = mfma_bf16(A[b][dy * 3 + dx], in, acc[o][b]);
        }
      }
    }
    act[y] = relu_row(acc[0][0], acc[0][1]);
    keep(y, act[y]);
    act[y + 1] = relu_row(acc[1][0], acc[1][1]);
    keep(y + 1, act[y + 1]);
    C[0] = C[2];
    L[0] = L[2];
    R[0] = R[2];
    C[1] = C[3];
    L[1] = L[3];
    R[1] = R[3];
  }
}

// Layer 4 (32 -> 1 channel) with the register rows as the A operand: lane
// (g, x) holds A[x][8g..8g+7] (pixel x, K chunk g), and B_dy[k][n] =
// W4[fwd_channel(k)][dy][n] for n = dx < 3.  Three chained MFMA per row give
// D_y[x'][n] = sum_dy sum_ci a3[ci][y + dy - 1][x'] W4[ci][dy][n] (D lane
// (g, n) holds x' = 4g..4g+3); all 16 rows go to dbuf (three FP32 planes
// [16][16] in LDS, kOutPlane apart so that the planes' writes use different
// banks) and, after one barrier,
//   out[y][x] = b4 + D_y[x - 1][0] + D_y[x][1] + D_y[x + 1][2]
// (zero past the tile) for the pixels (4g + r, x) of lane (g, x), r = 0..3.
constexpr int kOutPlane = 256 + 16;
__device__ __forceinline__ f4 layer_out1(const i4 (&act)[16], const i4 *packs,
                                         float *dbuf, float b4, int lane) {
  const i4 B0 = packs[lane], B1 = packs[64 + lane], B2 = packs[128 + lane];
  const int n = lane & 15, g = lane >> 4;
  f4 d[16];
#pragma unroll
  for (int y = 0; y < 16; y++) {
    d[y] = (f4){0.f, 0.f, 0.f, 0.f};
    if (y > 0) d[y] = mfma_bf16(act[y - 1], B0, d[y]);
    d[y] = mfma_bf16(act[y], B1, d[y]);
    if (y < 15) d[y] = mfma_bf16(act[y + 1], B2, d[y]);
  }
  if (n < 3)
#pragma unroll
    for (int y = 0; y < 16; y++)
      *reinterpret_cast<f4 *>(dbuf + n * kOutPlane + y * 16 + 4 * g) = d[y];
  wave_sync();
  const int nl = n > 0 ? n - 1 : 0, nr = n < 15 ? n + 1 : 15;
  f4 out;
#pragma unroll
  for (int r = 0; r < 4; r++) {
    const float *D = dbuf + (4 * g + r) * 16;
    const float l = D[nl], c = D[kOutPlane + n], rr = D[2 * kOutPlane + nr];
    float v = b4 + c;
    v += n > 0 ? l : 0.0f;
    v += n < 15 ? rr : 0.0f;
    out[r] = v;
  }
  return out;
}

// Writes the zero border of the 18 x 18 input grid (68 cells); the tiles
// write the inside only.
__device__ __forceinline__ void in_pad_border(int *in_pad, int lane) {
  for (int c = lane; c < 68; c += 64) {
    int cell;
    if (c < 18) cell = c;                          // top row
    else if (c < 36) cell = 17 * 18 + (c - 18);    // bottom row
    else if (c < 52) cell = (c - 35) * 18;         // left column, rows 1..16
    else cell = (c - 51) * 18 + 17;                // right column, rows 1..16
    in_pad[cell] = 0;
  }
}

__device__ __forceinline__ void in_pad_put(int *in_pad, int row, int col, float x0, float x1) {
  in_pad[(row + 1) * 18 + col + 1] = bf16_pair(x0, x1);
}

// a and b summed over the wave (uniform), lanes 32, 16, 8, 4, 2 and 1 apart:
// row swaps and DPP, where __shfl_xor would take twelve LDS round trips.
template <int CTRL>
__device__ __forceinline__ float dpp_add(float v) {
  return v + __int_as_float(
                 __builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xF, 0xF, true));
}
__device__ __forceinline__ void wave_sum2(float &a, float &b) {
  const auto p = __builtin_amdgcn_permlane32_swap(__float_as_uint(a), __float_as_uint(b),
                                                  false, false);
  float s = __uint_as_float(p[0]) + __uint_as_float(p[1]);  // a below lane 32, b above
  const auto q = __builtin_amdgcn_permlane16_swap(__float_as_uint(s), __float_as_uint(s),
                                                  false, false);
  s = __uint_as_float(q[0]) + __uint_as_float(q[1]);
  s = dpp_add<0x128>(s);  // row_ror:8
  s = dpp_add<0x124>(s);  // row_ror:4 (equal 8 lanes apart by now)
  s = dpp_add<0x4E>(s);   // quad_perm [2, 3, 0, 1]
  s = dpp_add<0xB1>(s);   // quad_perm [1, 0, 3, 2]
  a = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(s), 0));
  b = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(s), 32));
}

// Normalises one tile held in the solver's lane layout (lane (g, x) has
// rows 4g + r, column x) into the padded input grid; returns sigma.
__device__ __forceinline__ void tile_inputs(const float *d_tile_lane, const float *gm_lane,
                                            int *in_pad, int lane, float &sigma) {
  float mu = d_tile_lane[0] + d_tile_lane[1] + (d_tile_lane[2] + d_tile_lane[3]);
  float gmean = gm_lane[0] + gm_lane[1] + (gm_lane[2] + gm_lane[3]);
  wave_sum2(mu, gmean);
  mu *= 1.0f / 256.0f;
  gmean *= 1.0f / 256.0f;
  sigma = sqrtf(fmaxf(mu, 1.0f) + gmean);
  const float inv = 1.0f / sigma;
  const int x = lane & 15, g = lane >> 4;
#pragma unroll
  for (int r = 0; r < 4; r++)
    in_pad_put(in_pad, 4 * g + r, x, (d_tile_lane[r] - mu) * inv, gm_lane[r] * inv * inv);
}

// A wave's LDS: the padded input grid (18 x 18 BF16 pairs), layer 4's partial
// sums and the tile's data.
constexpr int kNetGridInts = 18 * 18;
constexpr int kNetOutFloats = 3 * kOutPlane;
constexpr int kNetWaveFloats = kNetGridInts + kNetOutFloats + 256;
static_assert(kNetGridInts % 4 == 0 && kNetWaveFloats % 4 == 0, "16-byte rows of dbuf");

// The network body on one tile whose inputs are in the padded grid; returns
// the output y at pixels (4g + r, x) of lane (g, x).  pk / bl: the forward
// packs and biases staged in LDS.  acts (may be NULL): post-ReLU layer 1-3
// activations, BF16 [3][n][256][32] in the standard channel order, of tile t.
// One wave runs it; the grid and dbuf are the wave's own.  before_out() runs
// before layer 4: loads of the next tile are issued there, where the middle
// layers' weights have left their registers and three matrix products a row
// cover the loads' way.
template <class BeforeOut>
__device__ __forceinline__ f4 net_body(const int *grid, float *dbuf, const i4 *pk,
                                       const float *bl, int lane, __bf16 *acts, long long n,
                                       long long t, BeforeOut before_out) {
  auto keep = [&](int layer) {
    return [=](int y, i4 v) {
      if (acts != nullptr)
        store_row_std(acts + (((long long)layer * n + t) * 256) * kCh, y, lane, v);
    };
  };
  const int z = opaque_zero();
  i4 act[16];
  wave_sync();  // the input grid is complete
  layer_in2(grid, pk + (PK_L1 - PK_L1) * 64 + z, bl + z, lane, act, keep(0));
  layer32(act, pk + (PK_L2 - PK_L1) * 64, bl + 32, lane, keep(1));
  layer32(act, pk + (PK_L3 - PK_L1) * 64, bl + 64, lane, keep(2));
  before_out();
  return layer_out1(act, pk + (PK_L4T - PK_L1) * 64 + z, dbuf, bl[96 + z], lane);
}

// Forward workgroups: kNetWaves waves, each running its own tiles, share the
// forward packs (layers 1-4, 41 KB) and biases staged once in LDS.
constexpr int kNetWaves = 4;
constexpr int kFwdPacks = PK_B4 - PK_L1;
constexpr int kNetFwdLdsBytes = kFwdPacks * 1024 + 128 * 4 + kNetWaves * kNetWaveFloats * 4;

// Copies the forward packs and the biases [b1 | b2 | b3 | b4] into LDS, all
// of a thread's loads in flight together (one behind the other they delayed a
// workgroup's first tile by 1 us).
__device__ __forceinline__ void stage_forward(const i4 *__restrict__ packs,
                                              const float *__restrict__ P, i4 *pk, float *bl) {
  constexpr int kThreads = 64 * kNetWaves, kItems = kFwdPacks * 64;
  constexpr int kEach = (kItems + kThreads - 1) / kThreads;
  const int tid = threadIdx.x;
  i4 v[kEach];
#pragma unroll
  for (int k = 0; k < kEach; k++) v[k] = packs[PK_L1 * 64 + min(tid + k * kThreads, kItems - 1)];
  const int layer = tid >> 5;
  const int at = (layer == 0 ? OFF_B1 : layer == 1 ? OFF_B2 : OFF_B3) + (tid & 31);
  const float b = P[tid < 96 ? at : OFF_B4];
#pragma unroll
  for (int k = 0; k < kEach; k++)
    if (tid + k * kThreads < kItems) pk[tid + k * kThreads] = v[k];
  if (tid < 97) bl[tid] = b;
  __syncthreads();
}

// Training / tensor mode: x [n][2][256] normalised inputs -> y [n][256].
// One wave per tile, its activations in registers; KEEP: written to acts too.
// A tile's inputs are loaded where they are used.  Loaded under the layer 4
// before (as the kernel over frames does) they spilled 13 registers of a build
// for both kinds, which took longer than what it hid: 8000 tiles with
// activations 97 us, 85 now; without 53 and 48; 2048 without 18.6 and 15.8
// (17.4 before the loads were moved).
template <bool KEEP>
__global__ __launch_bounds__(64 * kNetWaves) __attribute__((amdgpu_waves_per_eu(2)))
void net_fwd_kernel(const float *__restrict__ xin, float *__restrict__ yout,
                    __bf16 *__restrict__ acts, const i4 *__restrict__ packs,
                    const float *__restrict__ P, long long n) {
  extern __shared__ __align__(16) unsigned char lds_raw[];
  i4 *pk = reinterpret_cast<i4 *>(lds_raw);
  float *bl = reinterpret_cast<float *>(pk + kFwdPacks * 64);
  // the wave index is uniform: read it into a scalar register so the tile
  // loop's index arithmetic and frame-table reads stay on the scalar unit
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  int *const grid = reinterpret_cast<int *>(bl + 128 + wave * kNetWaveFloats);
  float *const dbuf = reinterpret_cast<float *>(grid + kNetGridInts);
  const int col = lane & 15, grp = lane >> 4;
  stage_forward(packs, P, pk, bl);
  in_pad_border(grid, lane);
  for (long long t = (long long)blockIdx.x * kNetWaves + wave; t < n;
       t += (long long)gridDim.x * kNetWaves) {
    const float *const x = xin + t * 512;
    float x0[4], x1[4];
#pragma unroll
    for (int k = 0; k < 4; k++) {
      x0[k] = x[lane + 64 * k];
      x1[k] = x[lane + 64 * k + 256];
    }
#pragma unroll
    for (int k = 0; k < 4; k++) in_pad_put(grid, 4 * k + grp, col, x0[k], x1[k]);
    const f4 y = net_body(grid, dbuf, pk, bl, lane, KEEP ? acts : nullptr, n, t, [] {});
#pragma unroll
    for (int r = 0; r < 4; r++) yout[t * 256 + (4 * grp + r) * 16 + col] = y[r];
    wave_sync();
  }
}

// Inference mode over frames: gather each window exactly like the solver,
// normalise, run the net and write u0 = d + sigma * y as [tiles][256].
__global__ __launch_bounds__(64 * kNetWaves) __attribute__((amdgpu_waves_per_eu(2)))
void net_warm_kernel(WithFrames<NetWarmArgs> W) {
  const long long total = W.args.total;
  const i4 *__restrict__ packs = reinterpret_cast<const i4 *>(W.args.packs);
  const float *__restrict__ P = W.args.params;
  extern __shared__ __align__(16) unsigned char lds_raw[];
  i4 *pk = reinterpret_cast<i4 *>(lds_raw);
  float *bl = reinterpret_cast<float *>(pk + kFwdPacks * 64);
  // the wave index is uniform: read it into a scalar register so the tile
  // loop's index arithmetic and frame-table reads stay on the scalar unit
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const FrameConst *fc = frame_table<NetWarmArgs>(W.args.frames);
  int *const grid = reinterpret_cast<int *>(bl + 128 + wave * kNetWaveFloats);
  float *const dbuf = reinterpret_cast<float *>(grid + kNetGridInts);
  float *const dkeep = dbuf + kNetOutFloats;
  const int col = lane & 15, grp = lane >> 4;

  // Tile t's window, edge-clamped in the reference geometry and zero-padded
  // in blocks, and the place of its start.  Both read the clamped pixel (32-bit
  // offsets from uniform pointers: the host keeps every frame below 2^31
  // elements), so that the eight loads go out together.
  auto load = [&](long long t, float (&d)[4], float (&gm)[4]) -> float * {
    int ln = lane;  // formed here: held across the layers it would be spilled
    asm volatile("" : "+v"(ln));
    const int col = ln & 15, grp = ln >> 4;
    int lo = 0, hi = W.args.n_frames - 1;
    while (lo < hi) {
      int mid = (lo + hi + 1) >> 1;
      if (fc[mid].first <= t) lo = mid; else hi = mid - 1;
    }
    const FrameConst &F = fc[lo];
    const int local = (int)(t - F.first);  // a frame has fewer than 2^31 windows
    const int a = (int)div_by((unsigned int)local, (unsigned int)F.ty, F.ty_magic);
    const int b = local - a * F.ty;
    const bool ref = F.geom == NCS_GEOM_REFERENCE;
    const int bx = ref ? min(-1 + 14 * a, F.H - 15) : 16 * a;
    const int by = ref ? min(-1 + 14 * b, F.W - 15) : 16 * b;
    const unsigned int gc = (unsigned int)min(max(by + col, 0), F.W - 1);
#pragma unroll
    for (int r = 0; r < 4; r++) {
      const unsigned int gr = (unsigned int)min(max(bx + 4 * grp + r, 0), F.H - 1);
      d[r] = F.data[gr * (unsigned int)F.ds + gc];
      gm[r] = F.gamma[gr * (unsigned int)F.gs + gc];
    }
    if (!ref) {
#pragma unroll
      for (int r = 0; r < 4; r++) {
        const bool ok = bx + 4 * grp + r < F.H && by + col < F.W;
        d[r] = ok ? d[r] : 0.0f;
        gm[r] = ok ? gm[r] : 0.0f;
      }
    }
    // starts are indexed in the caller's frame order
    return W.args.u0 + (F.slot + local) * 256;
  };

  const long long stride = (long long)gridDim.x * kNetWaves;
  long long t = (long long)blockIdx.x * kNetWaves + wave;
  float d[4], gm[4];
  float *u0 = nullptr;
  if (t < total) u0 = load(t, d, gm);
  stage_forward(packs, P, pk, bl);
  in_pad_border(grid, lane);
  // The two waves of a SIMD start together and run the same tile in the same
  // time: both would convert, shift and wait in step, with the matrix cores
  // idle.  Each is favoured on every other tile, which keeps them apart (two
  // 2048^2 frames, net and solve: 424 -> 418 us; always the same one: 427).  Up
  // to one and a half tiles a wave the other one would end alone: 2116 tiles on
  // 2048 waves 23.7 us so and 21.7 without, 3025 23.9 and 22.1; 3249 26.0 and
  // 28.0.
  const bool apart = 2 * total > 3 * stride;
  bool favoured = 2 * blockIdx.x >= gridDim.x;
  for (; t < total; t += stride) {
    if (apart) {
      if (favoured) __builtin_amdgcn_s_setprio(1);
      else __builtin_amdgcn_s_setprio(0);
      favoured = !favoured;
    }
    float sigma;
    tile_inputs(d, gm, grid, lane, sigma);
#pragma unroll
    for (int r = 0; r < 4; r++) dkeep[r * 64 + lane] = d[r];
    float *const w = u0;
    const f4 y = net_body(grid, dbuf, pk, bl, lane, nullptr, 0, 0, [&] {
      if (t + stride < total) u0 = load(t + stride, d, gm);
    });
#pragma unroll
    for (int r = 0; r < 4; r++)
      w[(4 * grp + r) * 16 + col] = dkeep[r * 64 + lane] + sigma * y[r];
    wave_sync();
  }
}

// ---------------------------------------------------------------------------
// backward
// ---------------------------------------------------------------------------

// The backward pass of one tile is 2 x 72 MFMA per wave and layer for four
// waves (a team): the weight gradient is a GEMM over the tile's 256 pixels,
// the data gradient the forward convolution with flipped, transposed weights.
// What bounds it is the feed of the matrix cores, so the layout is chosen for
// that:
//  * activations and data gradients sit in LDS as 18 x 18 pixels of 32 BF16
//    channels with a zero border, so a tap is a fixed address offset and no
//    read needs a bounds check;
//  * the weight gradient wants 8 pixels of one channel per lane where memory
//    has channels innermost: the transposing LDS read (ds_read_b64_tr_b16:
//    lane 16 g + i of a group gets elements 0..3 of column i from the 4 x 16
//    block the group addresses) takes them straight from the same buffer the
//    convolution reads.  A K chunk of 32 is rows r and r + 8, so the fragment
//    of an input row serves all three dy taps;
//  * each wave keeps its quarter of every layer's weight gradient (one
//    16 x 16 block of all nine taps) in registers over all its tiles; the
//    19,393 sums go to memory once per workgroup, through LDS, so that the
//    atomics are contiguous.
// One workgroup of two teams per CU (142 KB of LDS) walks its tiles, with the
// next activations loaded into registers while the present ones are used.
// Per two tiles a CU takes 17.5k cycles, 10.5k of them matrix work (an
// in-kernel clock: 5.4k per middle layer, 152 MFMA per wave on two waves per
// SIMD).  With the parameter packing and the clearing of the sums before it,
// one call on 1024 tiles went from 1264 us to 51 us and on 8000 from 7306 us
// to 197 us against the kernel before it (one wave per tile, 16-bit LDS
// gathers for the weight gradient, every tile's sums added in memory).  A
// tile's inputs and dL/dout are asked for a phase before they are stored:
// loaded where they are used, each cost the way to memory once per tile (8000
// tiles: 192.6 us, 183.9 now).
constexpr int kBwdTeams = 2;
constexpr int kPixBytes = 2 * kCh;                 // one pixel's channels
constexpr int kRowBytes = 18 * kPixBytes;          // one padded row
constexpr int kActBytes = 18 * kRowBytes;          // one padded tile
constexpr int kPlaneBytes = 18 * 32;               // [18 rows][16 pixels] BF16, rows padded
constexpr int kDyPlanes = 9;                       // (split of 3) x (dx of 3)
constexpr int kXPlanes = 6;                        // (channel of 2) x (dx of 3)
constexpr int kTeamBytes = 3 * kActBytes + (kDyPlanes + kXPlanes) * kPlaneBytes;
constexpr int kBwdLdsBytes = kBwdTeams * kTeamBytes;
static_assert(kBwdLdsBytes >= (N_PARAMS + kBwdTeams * (27 * kCh + 4)) * 4,
              "the sums are staged in the same LDS");
static_assert(OFF_B4 - OFF_W4 < kBwdTeams * 256, "one thread per layer-4 parameter");
static_assert(kTeamBytes % 16 == 0 && kBwdLdsBytes <= 160 * 1024, "LDS of one CU");

typedef __attribute__((address_space(3))) unsigned char LdsByte;
typedef __attribute__((address_space(3))) s4v LdsS4;

// Byte of a pixel's 16-channel block in its row: padded column c, block b.
// The two blocks of columns 8..15 are swapped, so that the two lane groups of
// a transposed read that are eight columns apart use different banks (a row
// of 64-byte pixels comes back to the same bank every four).
__device__ __forceinline__ int pix_block(int c, int b) {
  return c * kPixBytes + 32 * (b ^ ((c >> 3) & 1));
}

// 8 pixels of one channel (an operand's K chunk): lane (g, i) gets channel i
// of the 16-channel block a and b point into, pixels 0..3 and 4..7.
__device__ __forceinline__ i4 tr_frag(const LdsByte *pa, const LdsByte *pb) {
  const s4v a = __builtin_amdgcn_ds_read_tr16_b64_v4i16((LdsS4 *)pa);
  const s4v b = __builtin_amdgcn_ds_read_tr16_b64_v4i16((LdsS4 *)pb);
  const i2v ai = __builtin_bit_cast(i2v, a), bi = __builtin_bit_cast(i2v, b);
  return (i4){ai.x, ai.y, bi.x, bi.y};
}

__device__ __forceinline__ i4 lds_i4(const LdsByte *p) {
  return *reinterpret_cast<const __attribute__((address_space(3))) i4 *>(p);
}

// Weight gradient of a 32 -> 32 layer, this wave's 16 x 16 block of the nine
// taps: w[tap][co][ci] += sum_p dz[p][co] act[p + tap][ci].  dz and act are
// the padded tiles, oz[j] and oa[dx][j] the lane's offsets of a transposed
// read of its block in padded row 0 (j: pixels 0..3 or 4..7 of the chunk, dx:
// the tap's column); chunk r of dz is its rows r and r + 8, and the act
// fragment of rows r', r' + 8 meets the chunks r' - dy.
__device__ __forceinline__ void grad_w32(const LdsByte *dz, const int (&oz)[2],
                                         const LdsByte *act, const int (&oa)[3][2], f4 (&w)[9],
                                         f4 &bias, bool with_bias) {
  const int one2 = 0x3f803f80;  // BF16 1.0, twice
  const i4 ones = {one2, one2, one2, one2};
  i4 prev = {0, 0, 0, 0}, cur = prev, next = prev;  // dz chunks r' - 1, r', r' + 1
#pragma unroll
  for (int rp = -1; rp <= 8; rp++) {
    prev = cur;
    cur = next;
    if (rp + 1 <= 7) {
      next = tr_frag(dz + oz[0] + (rp + 2) * kRowBytes, dz + oz[1] + (rp + 2) * kRowBytes);
      if (with_bias) bias = mfma_bf16(next, ones, bias);
    }
#pragma unroll
    for (int dx = 0; dx < 3; dx++) {
      const i4 a = tr_frag(act + oa[dx][0] + (rp + 1) * kRowBytes,
                           act + oa[dx][1] + (rp + 1) * kRowBytes);
      if (rp + 1 <= 7) w[0 + dx] = mfma_bf16(next, a, w[0 + dx]);             // dy = -1
      if (rp >= 0 && rp <= 7) w[3 + dx] = mfma_bf16(cur, a, w[3 + dx]);       // dy = 0
      if (rp >= 1) w[6 + dx] = mfma_bf16(prev, a, w[6 + dx]);                 // dy = +1
    }
  }
}

// Data gradient of a 32-channel layer for this wave's output block and eight
// rows, masked by the ReLU of the activations there, as BF16 in registers:
// the convolution of dz with the flipped, transposed weights (packs: the
// lane's entries of the nine taps, read from L2 at each use: kept in
// registers over the tiles they spilled), each accumulator from zero.  z
// points at the lane's pixel of padded row 8 h, act at the lane's four channels
// of row 8 h's pixels (padded).
__device__ __forceinline__ void grad_data32(const LdsByte *z, const LdsByte *act,
                                            const i4 *__restrict__ packs, i2v (&out)[8]) {
  i4 A[9];
#pragma unroll
  for (int t = 0; t < 9; t++) A[t] = packs[t * 64];
  i4 C[4], L[4], R[4];
#pragma unroll
  for (int q = 0; q < 2; q++) {
    C[q] = lds_i4(z + q * kRowBytes);
    L[q] = dpp_i4<kRowShr1>(C[q]);
    R[q] = dpp_i4<kRowShl1>(C[q]);
  }
#pragma unroll
  for (int y = 0; y < 8; y += 2) {
#pragma unroll
    for (int q = 2; q < 4; q++) {
      C[q] = lds_i4(z + (y + q) * kRowBytes);
      L[q] = dpp_i4<kRowShr1>(C[q]);
      R[q] = dpp_i4<kRowShl1>(C[q]);
    }
    f4 acc[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
#pragma unroll
    for (int q = 0; q < 4; q++)
#pragma unroll
      for (int dx = 0; dx < 3; dx++) {
        const i4 in = dx == 0 ? L[q] : (dx == 1 ? C[q] : R[q]);
#pragma unroll
        for (int o = 0; o < 2; o++) {
          const int dy = q - o;
          if (dy < 0 || dy > 2) continue;
          acc[o] = mfma_bf16(A[dy * 3 + dx], in, acc[o]);
        }
      }
#pragma unroll
    for (int o = 0; o < 2; o++)
      out[y + o] = relu_masked(
          acc[o], *reinterpret_cast<const __attribute__((address_space(3))) i2v *>(
                      act + (y + o) * kRowBytes));
#pragma unroll
    for (int q = 0; q < 2; q++) {
      C[q] = C[q + 2];
      L[q] = L[q + 2];
      R[q] = R[q + 2];
    }
  }
}

// The pixel's value in the three dx planes of one quantity: plane dx holds
// v[row][x + dx - 1] at (row, x), zero where that is outside the tile (those
// entries, like the padding rows, are never written).
__device__ __forceinline__ void put_planes(LdsByte *planes, int row, int col, short v) {
#pragma unroll
  for (int dx = 0; dx < 3; dx++) {
    const int x = col + 1 - dx;
    if (x >= 0 && x < 16)
      *reinterpret_cast<__attribute__((address_space(3))) short *>(
          planes + dx * kPlaneBytes + (row + 1) * 32 + 2 * x) = v;
  }
}

// Layer 4's weight gradient (input channel ci, tap tp) over a workgroup's tiles
// first + k step + (0 .. kBwdTeams - 1) in plain FP32, in-tile taps only.  It
// takes the place of the splits' matrix products where those do not hold: a
// sum that is not finite (dL/dout past BF16's largest value splits into an
// infinity, and a remainder's or a border's zero times an infinite activation
// is NaN), or one so small that dL/dout's remainders may have been below
// BF16's smallest value, 2^-133.  Rare, and slow: one thread per sum.
constexpr float kW4Small = 0x1p-96f;
__device__ float w4_fp32(const __bf16 *a3, const float *gout, int ci, int tp, long long first,
                         long long step, long long n) {
  const int dy = tp / 3 - 1, dx = tp % 3 - 1;
  float sum = 0.0f;
#pragma unroll 1
  for (long long t0 = first; t0 < n; t0 += step)
#pragma unroll 1
    for (long long t = t0; t < n && t < t0 + kBwdTeams; t++) {
      float s = 0.0f;
#pragma unroll 1
      for (int p = 0; p < 256; p++) {
        const int y = (p >> 4) + dy, x = (p & 15) + dx;
        if (y >= 0 && y < 16 && x >= 0 && x < 16)
          s += gout[t * 256 + p] * (float)a3[(t * 256 + y * 16 + x) * kCh + ci];
      }
      sum += s;
    }
  return sum;
}

__global__ __launch_bounds__(kBwdTeams * 256) __attribute__((amdgpu_waves_per_eu(2, 2)))
void net_bwd_kernel(const float *__restrict__ xin, const __bf16 *__restrict__ acts,
                    const float *__restrict__ gout, float *__restrict__ gP,
                    const i4 *__restrict__ packs, long long n) {
  __shared__ __align__(16) unsigned char lds_all[kBwdLdsBytes];
  const int team = __builtin_amdgcn_readfirstlane(threadIdx.x >> 8);
  const int wave = __builtin_amdgcn_readfirstlane((threadIdx.x >> 6) & 3);
  const int tid = threadIdx.x & 255, lane = threadIdx.x & 63;
  const int i = lane & 15, g = lane >> 4;
  const int hi = wave >> 1, lo = wave & 1;

  LdsByte *const base = (LdsByte *)lds_all + team * kTeamBytes;
  LdsByte *const buf0 = base, *const buf1 = base + kActBytes, *const buf2 = base + 2 * kActBytes;
  LdsByte *const dyp = base + 3 * kActBytes, *const xp = dyp + kDyPlanes * kPlaneBytes;
  // lane offsets: of a transposed read of this wave's blocks (dz: hi, act:
  // lo) in padded row 0 of the lane's chunk, of the lane's pixel as the
  // convolution reads it, of its four output channels
  int o_hi[2], o_lo[3][2];
#pragma unroll
  for (int j = 0; j < 2; j++) {
    const int row = 8 * (g >> 1) * kRowBytes + 8 * (i & 3), c = 8 * (g & 1) + 4 * j + (i >> 2);
    o_hi[j] = row + pix_block(c + 1, hi);
#pragma unroll
    for (int dx = 0; dx < 3; dx++) o_lo[dx][j] = row + pix_block(c + dx, lo);
  }
  const int conv0 = 8 * hi * kRowBytes + pix_block(i + 1, g >> 1) + 16 * (g & 1);
  const int own0 = (8 * hi + 1) * kRowBytes + pix_block(i + 1, lo) + 8 * g;
  // planes: chunk r of a plane is rows r and r + 8, eight pixels per lane
  const int pl0 = (8 * (g >> 1) + 1) * 32 + 16 * (g & 1);
  // layer 4: A row m = split * 9 + tap is the split's plane moved by -tap
  const int m4 = 16 * hi + i < 27 ? 16 * hi + i : 0;
  const int t4 = m4 % 9;
  const int dy_off = (3 * (m4 / 9) + 2 - t4 % 3) * kPlaneBytes + pl0 + (1 - t4 / 3) * 32;
  // layer 1: B column n = tap * 2 + ci, then a column of ones for the bias
  const int n1 = 16 * lo + i;
  const int t1 = n1 < 18 ? n1 >> 1 : 0;
  const int x_off = (3 * (n1 & 1) + t1 % 3) * kPlaneBytes + pl0 + (t1 / 3 - 1) * 32;

  const i4 A4 = packs[(PK_B4 + lo) * 64 + lane];
  f4 w3[9], w2[9], w1 = {0.f, 0.f, 0.f, 0.f}, w4 = w1, b3 = w1, b2 = w1;
#pragma unroll
  for (int t = 0; t < 9; t++) w3[t] = w2[t] = w1;
  float db4 = 0.0f;

  // one activation tile: four 16-byte pieces per thread, in registers on the
  // way from memory to a buffer
  typedef i4 Stage[4];
  Stage st;
  auto fetch_to = [&](Stage &st, int layer, long long t) {
    const i4 *src = reinterpret_cast<const i4 *>(acts + (((long long)layer * n + t) * 256) * kCh);
#pragma unroll
    for (int k = 0; k < 4; k++) st[k] = src[k * 256 + tid];
  };
  auto put_from = [&](const Stage &st, LdsByte *dst) {
#pragma unroll
    for (int k = 0; k < 4; k++) {
      const int px = 64 * k + (tid >> 2), part = tid & 3;
      *reinterpret_cast<__attribute__((address_space(3))) i4 *>(
          dst + ((px >> 4) + 1) * kRowBytes + pix_block((px & 15) + 1, part >> 1) +
          16 * (part & 1)) = st[k];
    }
  };
  auto fetch = [&](int layer, long long t) { fetch_to(st, layer, t); };
  auto put = [&](LdsByte *dst) { put_from(st, dst); };
  auto put_own = [&](LdsByte *dst, const i2v (&v)[8]) {
#pragma unroll
    for (int y = 0; y < 8; y++)
      *reinterpret_cast<__attribute__((address_space(3))) i2v *>(dst + own0 + y * kRowBytes) = v[y];
  };
  // dL/dout of the tile as three BF16 splits, whose sum is the FP32 value
  // (but for values past BF16's largest and remainders below its smallest,
  // see w4_fp32)
  auto put_dy = [&](float v) {
    db4 += v;
    const int row = tid >> 4, col = tid & 15;
    const __bf16 s0 = (__bf16)v;
    const bool fin = fabsf((float)s0) <= 3.4e38f;
    const float r1 = fin ? v - (float)s0 : 0.0f;
    const __bf16 s1 = (__bf16)r1;
    const __bf16 s2 = (__bf16)(r1 - (float)s1);
    put_planes(dyp, row, col, __builtin_bit_cast(short, s0));
    put_planes(dyp + 3 * kPlaneBytes, row, col, __builtin_bit_cast(short, s1));
    put_planes(dyp + 6 * kPlaneBytes, row, col, __builtin_bit_cast(short, s2));
  };

  const long long step = (long long)gridDim.x * kBwdTeams;
  long long t = (long long)blockIdx.x * kBwdTeams + team;
  // both teams run the iterations of the first (it has at least as many)
  const long long first = (long long)blockIdx.x * kBwdTeams;
  const int iters = first < n ? (int)((n - first + step - 1) / step) : 0;
  float x0 = 0.0f, x1 = 0.0f;  // the tile's inputs, loaded one layer ahead
  auto fetch_x = [&](long long t) {
    x0 = xin[t * 512 + tid];
    x1 = xin[t * 512 + 256 + tid];
  };
  {
    Stage s2, s1;
    float dy = 0.0f;
    if (t < n) {
      fetch_to(s2, 2, t);
      fetch_to(s1, 1, t);
      dy = gout[t * 256 + tid];
      fetch(0, t);
      fetch_x(t);
    }
    // the borders' zeros, while the first tile is on its way
    for (int k = threadIdx.x; k < kBwdLdsBytes / 16; k += blockDim.x)
      reinterpret_cast<i4 *>(lds_all)[k] = (i4){0, 0, 0, 0};
    __syncthreads();
    if (t < n) {
      put_from(s2, buf0);
      put_from(s1, buf1);
      put_dy(dy);
    }
  }
  for (int it = 0; it < iters; it++, t += step) {
    const bool on = t < n, more = t + step < n;  // uniform over the team
    i2v own[8];
    __syncthreads();  // a3 in buf0, a2 in buf1, dy planes; a1 on its way
    if (on) {
      // layer 4: dW4[tap][ci] = sum_q dy[q - tap] a3[q] per split of dy
#pragma unroll
      for (int r = 0; r < 8; r++)
        w4 = mfma_bf16(lds_i4(dyp + dy_off + r * 32),
                       tr_frag(buf0 + o_lo[1][0] + (r + 1) * kRowBytes,
                               buf0 + o_lo[1][1] + (r + 1) * kRowBytes), w4);
      // dz3 = conv(dy, flipped W4) masked by a3 > 0, K = tap padded to 32
      const int m0 = g == 0 ? -1 : 0, m1 = g == 1 ? 0xffff : 0;
      int v[3][3];  // BF16 dy of rows y - 1 .. y + 1 at x - 1 .. x + 1
      auto dy_row = [&](int yy, int (&o)[3]) {  // yy: padded row; dx by DPP
        o[1] = *reinterpret_cast<const __attribute__((address_space(3))) unsigned short *>(
            dyp + kPlaneBytes + yy * 32 + 2 * i);
        o[0] = __builtin_amdgcn_update_dpp(0, o[1], kRowShr1, 0xF, 0xF, true);
        o[2] = __builtin_amdgcn_update_dpp(0, o[1], kRowShl1, 0xF, 0xF, true);
      };
      dy_row(8 * hi, v[0]);
      dy_row(8 * hi + 1, v[1]);
#pragma unroll
      for (int y = 0; y < 8; y++) {
        dy_row(8 * hi + y + 2, v[2]);
        const i4 B = {(m0 & (v[0][0] | v[0][1] << 16)) | (m1 & v[2][2]),
                      m0 & (v[0][2] | v[1][0] << 16), m0 & (v[1][1] | v[1][2] << 16),
                      m0 & (v[2][0] | v[2][1] << 16)};
        const f4 z = {0.f, 0.f, 0.f, 0.f};
        own[y] = relu_masked(
            mfma_bf16(A4, B, z), *reinterpret_cast<const __attribute__((address_space(3))) i2v *>(
                                     buf0 + own0 + y * kRowBytes));
#pragma unroll
        for (int dx = 0; dx < 3; dx++) {
          v[0][dx] = v[1][dx];
          v[1][dx] = v[2][dx];
        }
      }
    }
    __syncthreads();  // every read of a3 is done
    if (on) {
      put_own(buf0, own);
      put(buf2);
      put_planes(xp, tid >> 4, tid & 15, __builtin_bit_cast(short, (__bf16)x0));
      put_planes(xp + 3 * kPlaneBytes, tid >> 4, tid & 15, __builtin_bit_cast(short, (__bf16)x1));
    }
    if (more) fetch(2, t + step);
    __syncthreads();  // dz3 in buf0, a2 in buf1, a1 in buf2, x planes
    if (on) {
      grad_w32(buf0, o_hi, buf1, o_lo, w3, b3, lo == 0);
      grad_data32(buf0 + conv0, buf1 + own0, packs + (PK_B3 + lo * 9) * 64 + lane + opaque_zero(), own);
    }
    __syncthreads();
    if (on) put_own(buf1, own);
    float dy = 0.0f;
    if (more) {
      put(buf0);
      fetch(1, t + step);
      dy = gout[(t + step) * 256 + tid];
    }
    __syncthreads();  // dz2 in buf1, a1 in buf2
    if (on) {
      grad_w32(buf1, o_hi, buf2, o_lo, w2, b2, lo == 0);
      grad_data32(buf1 + conv0, buf2 + own0, packs + (PK_B2 + lo * 9) * 64 + lane + opaque_zero(), own);
    }
    __syncthreads();
    if (on) put_own(buf2, own);
    if (more) {
      put(buf1);
      put_dy(dy);
      fetch(0, t + step);
      fetch_x(t + step);
    }
    __syncthreads();  // dz1 in buf2
    if (on) {
      const int one2 = 0x3f803f80;
      const i4 ones = {one2, one2, one2, one2};
#pragma unroll
      for (int r0 = 0; r0 < 8; r0 += 4) {
        i4 za[4], xb[4];
#pragma unroll
        for (int r = 0; r < 4; r++) {
          za[r] = tr_frag(buf2 + o_hi[0] + (r0 + r + 1) * kRowBytes,
                          buf2 + o_hi[1] + (r0 + r + 1) * kRowBytes);
          xb[r] = lds_i4(xp + x_off + (r0 + r) * 32);
        }
#pragma unroll
        for (int r = 0; r < 4; r++) w1 = mfma_bf16(za[r], n1 == 18 ? ones : xb[r], w1);
      }
    }
  }

  // The workgroup's sums, in the order of the parameters in LDS: the first
  // team stores, the second adds (LDS float atomics took 50 us here), then
  // one contiguous pass of atomics to memory.  Layer 4's three splits and
  // the waves' parts of its bias are added up on the way out.
  __syncthreads();
  for (int off = 32; off >= 1; off >>= 1) db4 += __shfl_xor(db4, off);
  float *const sum = reinterpret_cast<float *>(lds_all);
  float *const sum4 = sum + N_PARAMS;               // [team][27][32]
  float *const sumb = sum4 + kBwdTeams * 27 * kCh;  // [team][wave]
  for (int q = 0; q < kBwdTeams; q++) {
    if (team == q) {
      auto add = [&](int k, float v) { sum[k] = q == 0 ? v : sum[k] + v; };
#pragma unroll
      for (int r = 0; r < 4; r++) {
        const int co = 16 * hi + 4 * g + r;
        const int k = (co * kCh + 16 * lo + i) * 9;
#pragma unroll
        for (int tp = 0; tp < 9; tp++) {
          add(OFF_W3 + k + tp, w3[tp][r]);
          add(OFF_W2 + k + tp, w2[tp][r]);
        }
        if (lo == 0 && i == 0) {
          add(OFF_B3 + co, b3[r]);
          add(OFF_B2 + co, b2[r]);
        }
        if (n1 < 18) add(OFF_W1 + (co * 2 + (n1 & 1)) * 9 + (n1 >> 1), w1[r]);
        if (n1 == 18) add(OFF_B1 + co, w1[r]);
        const int m = 16 * hi + 4 * g + r;
        if (m < 27) sum4[(q * 27 + m) * kCh + 16 * lo + i] = w4[r];
      }
      if (lane == 0) sumb[q * 4 + wave] = db4;
    }
    __syncthreads();
  }
  for (int k = threadIdx.x; k < OFF_W4; k += blockDim.x) atomicAdd(&gP[k], sum[k]);
  if (threadIdx.x < OFF_B4 - OFF_W4) {
    const int ci = threadIdx.x / 9, tp = threadIdx.x - 9 * ci;
    float v = 0.0f;
#pragma unroll
    for (int m = 0; m < kBwdTeams * 3; m++) v += sum4[(m * 9 + tp) * kCh + ci];
    if (!(fabsf(v) < INFINITY) || (v != 0.0f && fabsf(v) < kW4Small))
      v = w4_fp32(acts + 2 * n * 256 * kCh, gout, ci, tp, first, step, n);
    atomicAdd(&gP[OFF_W4 + threadIdx.x], v);
  }
  if (threadIdx.x == OFF_B4 - OFF_W4) {
    float v = 0.0f;
#pragma unroll
    for (int k = 0; k < kBwdTeams * 4; k++) v += sumb[k];
    atomicAdd(&gP[OFF_B4], v);
  }
}

// ---------------------------------------------------------------------------
// launches
// ---------------------------------------------------------------------------

// Packs what a pass needs of the parameters (NULL: nothing), and clears the
// N_PARAMS sums when given.
static hipError_t pack(const float *P, void *packs, int first, int end, float *sums,
                       hipStream_t s) {
  if (P == nullptr) end = first;
  const int items = std::max((end - first) * 512, sums != nullptr ? N_PARAMS : 0);
  if (items == 0) return hipSuccess;
  hipLaunchKernelGGL(net_pack_kernel, dim3((items + 255) / 256), dim3(256), 0, s, P,
                     reinterpret_cast<__bf16 *>(packs), first, end, sums);
  return hipGetLastError();
}
hipError_t net_pack(const float *P, void *packs, hipStream_t s) {
  return pack(P, packs, 0, N_PACKS, nullptr, s);
}
hipError_t net_pack_forward(const float *P, void *packs, hipStream_t s) {
  return pack(P, packs, 0, PK_B4, nullptr, s);
}
hipError_t net_pack_backward(const float *P, void *packs, float *gP, hipStream_t s) {
  const uintptr_t p = reinterpret_cast<uintptr_t>(P), g = reinterpret_cast<uintptr_t>(gP);
  constexpr uintptr_t bytes = N_PARAMS * sizeof(float);
  if (P == nullptr || p >= g + bytes || g >= p + bytes) return pack(P, packs, PK_B4, N_PACKS, gP, s);
  // the gradient takes the parameters' place: read them all first
  const hipError_t e = pack(P, packs, PK_B4, N_PACKS, nullptr, s);
  return e == hipSuccess ? pack(nullptr, packs, PK_B4, N_PACKS, gP, s) : e;
}

size_t net_packs_bytes() { return (size_t)N_PACKS * 512 * 2; }

// Forward workgroups (kNetWaves waves, one tile per wave at a time) that fill
// the device: the occupancy limit of the forward kernels times the CUs, at
// most one tile per wave.
int net_forward_grid(long long n, int cus) {
  int blocks = 0;
  if (hipOccupancyMaxActiveBlocksPerMultiprocessor(
          &blocks, reinterpret_cast<const void *>(net_warm_kernel), 64 * kNetWaves,
          kNetFwdLdsBytes) != hipSuccess ||
      blocks < 1)
    blocks = 1;
  const long long need = (n + kNetWaves - 1) / kNetWaves;
  return (int)std::max<long long>(1, std::min<long long>(need, (long long)blocks * cus));
}

hipError_t net_forward(const float *x, float *y, void *acts, const void *packs, const float *P,
                       long long n, int grid, hipStream_t s) {
  if (n <= 0) return hipSuccess;
  hipLaunchKernelGGL(acts != nullptr ? net_fwd_kernel<true> : net_fwd_kernel<false>, dim3(grid),
                     dim3(64 * kNetWaves), kNetFwdLdsBytes, s, x, y,
                     reinterpret_cast<__bf16 *>(acts), reinterpret_cast<const i4 *>(packs), P, n);
  return hipGetLastError();
}

// gP: cleared by net_pack_backward.
hipError_t net_backward(const float *x, const void *acts, const float *gout, float *gP,
                        const void *packs, long long n, int cus, hipStream_t s) {
  if (n <= 0) return hipSuccess;
  const long long pairs = (n + kBwdTeams - 1) / kBwdTeams;
  const int grid = (int)std::max<long long>(1, std::min<long long>(pairs, cus));
  hipLaunchKernelGGL(net_bwd_kernel, dim3(grid), dim3(kBwdTeams * 256), 0, s, x,
                     reinterpret_cast<const __bf16 *>(acts), gout, gP,
                     reinterpret_cast<const i4 *>(packs), n);
  return hipGetLastError();
}

// The starts of every tile of a.n_frames frames: at a.frames (device), or
// without that at most kInlineFrames at inline_frames (host).
hipError_t net_warm(const NetWarmArgs &a, const FrameDev *inline_frames, int grid, hipStream_t s) {
  if (a.total <= 0) return hipSuccess;
  WithFrames<NetWarmArgs> W;
  W.args = a;
  if (a.frames == nullptr) set_inline(W, inline_frames, a.n_frames);
  hipLaunchKernelGGL(net_warm_kernel, dim3(grid), dim3(64 * kNetWaves), kNetFwdLdsBytes, s, W);
  return hipGetLastError();
}

}  // namespace ncs
