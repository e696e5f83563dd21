// Learned coarse-velocity closure: BF16 MFMA convolution network, forward,
// backward and Adam, for gfx950.  Interface and arithmetic: include/vpfc.h.
//
// Data layouts
//   rows of f, x, y, target, dy: [rows][256] FP32
//   stored activations a1..a3 and the pre-activation gradient dz2:
//     [rows][256][64] BF16, position-major (channels contiguous), the order of
//     the LDS tile
//   LDS "position-major" tile of one row: [260][kP] BF16, row p+2 holds the
//     64 channels at position p (rows 0, 1, 258, 259 are the zero padding),
//     kP = 80 keeps every 8-channel group 16-byte aligned and the MFMA
//     operand reads (16 positions x 16 bytes per lane group) free of LDS
//     bank conflicts: with a 144-byte pitch (kP = 72) they measured 2-way
//     conflicted on gfx950, with 160 bytes conflict-free
//
// MFMA v_mfma_f32_16x16x32_bf16 (D = A B + C, A 16x32, B 32x16): lane l
// supplies A[l%16][8(l/16)+j] and B[8(l/16)+j][l%16] for j < 8 and holds
// D[4(l/16)+j][l%16] for j < 4.

#include <hip/hip_runtime.h>

#include <cmath>
#include <cstring>
#include <string>
#include <vector>

#include "vpfc.h"
#include "vpfp.h"

namespace {

thread_local std::string g_err;

int fail(int code, const std::string& msg) {
  g_err = msg;
  return code;
}

#define FC_HIP(x)                                                                                   \
  do {                                                                                              \
    hipError_t e_ = (x);                                                                            \
    if (e_ != hipSuccess) return fail(VPFP_EHIP, std::string(#x) + ": " + hipGetErrorString(e_)); \
  } while (0)

typedef __bf16 bf16;
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef float floatx4 __attribute__((ext_vector_type(4)));

constexpr int kNV = VPFC_NV, kCH = VPFC_CHANNELS, kKS = VPFC_KERNEL, kK = kCH * kKS;
constexpr int kP = 80;          // position-major pitch (BF16)
constexpr int kRowsP = kNV + 4;
constexpr int oW1 = 0, oB1 = oW1 + kCH * kKS, oW2 = oB1 + kCH, oB2 = oW2 + kCH * kK, oW3 = oB2 + kCH,
              oB3 = oW3 + kCH * kK, oW4 = oB3 + kCH, oB4 = oW4 + kK, kParams = oB4 + 1;
static_assert(kParams == VPFC_NPARAMS, "parameter layout");
constexpr int kPart = (kParams + 3) & ~3;  // pitch of the partial gradients: 16-byte rows
constexpr int kPartWG = 256;    // workgroups of the gradient kernels (rows strided over them)

__device__ __forceinline__ float bfr(float x) { return (float)(bf16)x; }

__device__ __forceinline__ floatx4 mfma(const bf16x8& a, const bf16x8& b, const floatx4& c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

// ----------------------------------------------------------------------------
// 64 -> 64 convolution of one row on MFMA
//   out[co][p] = sum_{k, ci} W[co][k*64 + ci] in[ci][p + k - 2]
// in: position-major LDS tile; A: this wave's fragments of W [64][320] BF16
// (load_a).  Wave w computes
// co in [16w, 16w + 16) for all 256 positions and hands acc[nt][j] =
// out[16w + 4(l/16) + j][16 nt + l%16] to `epi`.
// ----------------------------------------------------------------------------
// A fragments of this wave's 16 output channels for the 10 K-chunks
__device__ __forceinline__ void load_a(const bf16* W, bf16x8 (&A)[10]) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const bf16* wr = W + (16 * wave + (lane & 15)) * kK + 8 * (lane >> 4);
#pragma unroll
  for (int c = 0; c < 10; ++c) A[c] = *reinterpret_cast<const bf16x8*>(wr + 32 * c);
}

template <class Epi>
__device__ __forceinline__ void mconv(const bf16* in, const bf16x8 (&A)[10], Epi epi) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int m = lane & 15, g = lane >> 4;
  floatx4 acc[16];
#pragma unroll
  for (int nt = 0; nt < 16; ++nt) acc[nt] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int c = 0; c < 10; ++c) {
    const int tap = c >> 1;
    const int ci0 = (c & 1) * 32 + 8 * g;
#pragma unroll
    for (int nt = 0; nt < 16; ++nt) {
      const bf16x8 b = *reinterpret_cast<const bf16x8*>(in + (16 * nt + m + tap) * kP + ci0);
      acc[nt] = mfma(A[c], b, acc[nt]);
    }
  }
  epi(acc, 16 * wave + 4 * g, m);
}

// zero the padding rows of a position-major tile
__device__ __forceinline__ void zero_pad_p(bf16* P) {
  for (int i = threadIdx.x; i < 4 * kP; i += blockDim.x) {
    const int r = i / kP, row = r < 2 ? r : kNV + r;
    P[row * kP + i % kP] = (bf16)0.f;
  }
}

// ----------------------------------------------------------------------------
// forward: one workgroup (256 threads, thread = position) per row, rows strided
//
// All four layers run on MFMA over one position-major LDS tile P:
//  * layer 1 (1 -> 64, K = 5): row p+2 of P keeps, in its pad columns 64..71,
//    the stencil record x[p-2..p+2] (BF16, zero outside the row, three zero
//    slots); wave w multiplies it by W1[16w + i][k] (A fragment with K < 5);
//  * layers 2 and 3 (64 -> 64): mconv, then in place over P once every wave
//    holds its sums (the records in columns 64..71 are not touched);
//  * layer 4 (64 -> 1, K = 320): W4 in every row of the A operand, so each
//    lane's sums are y at its own position; wave w takes positions
//    64w..64w+63 and hands y to the position's thread through LDS.
// The activations get tanh, rounded to BF16, as they leave the accumulators.
// ----------------------------------------------------------------------------
struct FwdArgs {
  const float* f;       // [rows][256]
  int rows;
  float in_scale, out_scale;
  const float* bg;      // [256] background profile, or null: the network then sees
                        // (f - bg) / s with s the row's rms of f - bg, and its output and
                        // target are in units of s
  const float* cons;    // [256 * 4 + 9] conservation projection (v, w, bg, unused, G^-1)
                        // applied to the correction, or null
  const float* p;       // FP32 parameters (W1, b1, b2, b3, W4, b4 are read here)
  const bf16* w2;       // [64][320] BF16 copies
  const bf16* w3;
  float* f_out;         // f + out_scale * y (may alias f) or null
  float* y_out;         // y or null
  // training (null otherwise)
  bf16* xin;            // [rows][256] L1 input
  bf16* a1;
  bf16* a2;
  bf16* a3;
  const float* target;  // [rows][256]
  float gscale;         // dy = gscale * (y - target)
  float* dy;            // [rows][256]
  float* loss_rows;     // [rows]: sum_v (y - target)^2
};

// the position-major tile (with the layer-1 stencil records in its pad
// columns) + reduction slots + BF16 W4 + layer-1 A rows + the layer-4
// outputs: 44352 bytes, so three workgroups share a CU's 160 KiB
constexpr int kFwdLds = kRowsP * kP * 2 + 64 + kK * 2 + kCH * 16 + kNV * 4;

// sum over the 256 threads of a workgroup (all threads get it); red: 4 floats
__device__ __forceinline__ float block_sum(float v, float* red) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  __syncthreads();
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
  __syncthreads();
  return (red[0] + red[1]) + (red[2] + red[3]);
}

// tanh for activations that are rounded to BF16 next, as x P(x^2) / Q(x^2)
// with P, Q of degree 4 in x^2 (coefficients fitted for the least maximum
// relative error on |x| <= 9 by vlapy_amd/csrc/tanh_fit.py) and x clamped to
// +-9 (tanh(9) = 1 - 3e-8).  FP32 evaluation: relative error <= 4e-7, so GPU
// and oracle activations seldom round to different BF16 values (a one-ulp
// flip moves the outputs it feeds by ~1e-3 of max |y|).  One reciprocal and
// no branch: 13 VALU instructions, against 14 with two transcendentals for
// sign(x) (1 - e^{-2|x|}) / (1 + e^{-2|x|}) with a Taylor series near 0.
__device__ __forceinline__ float tanh_act(float x) {
  const float c = __builtin_amdgcn_fmed3f(x, -9.f, 9.f);
  const float y = c * c;
  const float p =
      fmaf(fmaf(fmaf(fmaf(1.335543409e-08f, y, 2.060965016e-05f), y, 3.495623358e-03f), y, 1.338105500e-01f), y, 1.f);
  const float q =
      fmaf(fmaf(fmaf(fmaf(7.776877737e-07f, y, 3.285691782e-04f), y, 2.587711625e-02f), y, 4.671437144e-01f), y, 1.f);
  return (c * p) * __builtin_amdgcn_rcpf(q);
}

// tanh(acc + b) of accumulator tile nt (channels co0..co0+3 of lane (m, g),
// position 16 nt + m) into P at pr = P + (m + 2) kP + co0
template <int NT>
__device__ __forceinline__ void act_tile(const floatx4& acc, const float (&b)[4], bf16* pr) {
  bf16x4 o;
#pragma unroll
  for (int j = 0; j < 4; ++j) o[j] = (bf16)tanh_act(acc[j] + b[j]);
  *reinterpret_cast<bf16x4*>(pr + 16 * NT * kP) = o;
}

// act_tile over the 16 tiles of a 64 -> 64 layer
template <int NT = 0>
__device__ __forceinline__ void act_tiles(const floatx4* acc, const float (&b)[4], bf16* pr) {
  if constexpr (NT < 16) {
    act_tile<NT>(acc[NT], b, pr);
    act_tiles<NT + 1>(acc, b, pr);
  }
}

// the 256 positions of the LDS tile to a stored row of activations, 16 bytes
// per thread and pass (written by the lanes that form them instead, each
// channel's 2 bytes on its own, the forward pass of 4096 training rows took
// 194 us, with this 178)
__device__ __forceinline__ void store_tile(const bf16* P, bf16* dst) {
#pragma unroll
  for (int u = 0; u < 8; ++u) {
    const int i = threadIdx.x + 256 * u;
    *reinterpret_cast<bf16x8*>(dst + 8 * i) = *reinterpret_cast<const bf16x8*>(P + ((i >> 3) + 2) * kP + 8 * (i & 7));
  }
}

// three waves per SIMD (<= 168 registers) to match the three workgroups the
// LDS allows; left to itself the compiler takes 260 registers (one wave per
// SIMD), which measured 2.4x slower at 262144 rows.  TRAIN, the variant that
// stores what the backward pass needs, is a kernel of its own: in one kernel
// its addresses spilled 140 bytes and applying cost 4 % more
template <bool TRAIN>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(3))) void k_fwd(FwdArgs a) {
  extern __shared__ __align__(16) unsigned char lds[];
  bf16* P = reinterpret_cast<bf16*>(lds);
  float* red = reinterpret_cast<float*>(P + kRowsP * kP);
  bf16* w4b = reinterpret_cast<bf16*>(red + 16);  // BF16 W4, K order k*64 + ci
  bf16* w1b = w4b + kK;                            // [64][8]: W1[co][k], k < 5, then zeros
  float* ys = reinterpret_cast<float*>(w1b + 8 * kCH);  // layer-4 output by position
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6, m = lane & 15, g = lane >> 4;
  bf16x8 z8;
#pragma unroll
  for (int j = 0; j < 8; ++j) z8[j] = (bf16)0.f;
  zero_pad_p(P);
  *reinterpret_cast<bf16x8*>(P + (t + 2) * kP + kCH) = z8;  // stencil records start at zero
  for (int i = t; i < kK; i += 256) w4b[i] = (bf16)a.p[oW4 + i];
  for (int i = t; i < 8 * kCH; i += 256) w1b[i] = (bf16)((i & 7) < kKS ? a.p[oW1 + (i >> 3) * kKS + (i & 7)] : 0.f);
  const int co0 = 16 * wave + 4 * g;
  bf16* const pr = P + (m + 2) * kP + co0;  // this lane's activation slots (tile 0)
  __syncthreads();  // records zeroed before any thread writes into them
  for (int row = blockIdx.x; row < a.rows; row += gridDim.x) {
    const size_t ro = (size_t)row * kNV;
    const float fv = a.f[ro + t];
    // row scale: rms of the deviation from the background (1 without one)
    float d = fv, srow = 1.f;
    if (a.bg) {
      d = fv - a.bg[t];
      srow = sqrtf(block_sum(d * d, red) * (1.f / kNV) + 1e-30f);
    }
    const bf16 xb = (bf16)((a.in_scale / srow) * d);
    if constexpr (TRAIN) a.xin[ro + t] = xb;
    // x[t] is entry k of the record of position t + 2 - k
#pragma unroll
    for (int k = 0; k < kKS; ++k) {
      const int p = t + 2 - k;
      if (p >= 0 && p < kNV) P[(p + 2) * kP + kCH + k] = xb;
    }
    __syncthreads();
    // layer 1: 1 -> 64, tanh (writes columns 0..63 only, while the records are read)
    {
      // A[i][k] = W1[16 wave + i][k] for k < 5, zero beyond (lanes g > 0 read
      // the zero padding row of P)
      const bf16x8 A1 = *reinterpret_cast<const bf16x8*>(g == 0 ? w1b + 8 * (16 * wave + m) : P);
      const float b[4] = {a.p[oB1 + co0], a.p[oB1 + co0 + 1], a.p[oB1 + co0 + 2], a.p[oB1 + co0 + 3]};
      const bf16* rec = P + (m + 2) * kP + kCH;
      floatx4 acc[16];
#pragma unroll
      for (int nt = 0; nt < 16; ++nt)
        acc[nt] = mfma(A1, *reinterpret_cast<const bf16x8*>(rec + 16 * nt * kP), floatx4{0.f, 0.f, 0.f, 0.f});
      act_tiles(acc, b, pr);
    }
    __syncthreads();
    if constexpr (TRAIN) store_tile(P, a.a1 + (size_t)row * kCH * kNV);
    // layers 2 and 3: 64 -> 64, tanh, in place: every wave has its sums in
    // registers before any wave overwrites the tile.  The weight fragments are
    // reloaded per row (L2-resident): keeping both layers' in registers
    // measured slower (register pressure)
    {
      bf16x8 A[10];
      load_a(a.w2, A);
      mconv(P, A, [&](floatx4* acc, int c0, int) {
        const float b[4] = {a.p[oB2 + c0], a.p[oB2 + c0 + 1], a.p[oB2 + c0 + 2], a.p[oB2 + c0 + 3]};
        __syncthreads();
        act_tiles(acc, b, pr);
      });
    }
    __syncthreads();
    if constexpr (TRAIN) store_tile(P, a.a2 + (size_t)row * kCH * kNV);
    {
      bf16x8 A[10];
      load_a(a.w3, A);
      mconv(P, A, [&](floatx4* acc, int c0, int) {
        const float b[4] = {a.p[oB3 + c0], a.p[oB3 + c0 + 1], a.p[oB3 + c0 + 2], a.p[oB3 + c0 + 3]};
        __syncthreads();
        act_tiles(acc, b, pr);
      });
    }
    __syncthreads();
    if constexpr (TRAIN) store_tile(P, a.a3 + (size_t)row * kCH * kNV);
    // layer 4: 64 -> 1, linear; every row of A is W4, so lane (m, g) sums
    // y at position 16 nt + m in all four accumulator slots
    {
      floatx4 acc[4];
#pragma unroll
      for (int q = 0; q < 4; ++q) acc[q] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int c = 0; c < 10; ++c) {
        const int tap = c >> 1, ci0 = (c & 1) * 32 + 8 * g;
        const bf16x8 a4 = *reinterpret_cast<const bf16x8*>(w4b + 32 * c + 8 * g);
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const bf16x8 b = *reinterpret_cast<const bf16x8*>(P + (16 * (4 * wave + q) + m + tap) * kP + ci0);
          acc[q] = mfma(a4, b, acc[q]);
        }
      }
      if (g == 0) {
#pragma unroll
        for (int q = 0; q < 4; ++q) ys[16 * (4 * wave + q) + m] = acc[q][0];
      }
    }
    __syncthreads();
    float y = a.p[oB4] + ys[t];
    if (a.cons) {
      // remove bg (c0 + c1 v + c2 v^2): trapz moments 1, v, v^2 of y vanish
      const float vv = a.cons[t], w = a.cons[kNV + t], b = a.cons[2 * kNV + t];
      const float m0 = block_sum(w * y, red);
      const float m1 = block_sum(w * vv * y, red);
      const float m2 = block_sum(w * vv * vv * y, red);
      const float* gi = a.cons + 4 * kNV;
      const float c0 = gi[0] * m0 + gi[1] * m1 + gi[2] * m2;
      const float c1 = gi[3] * m0 + gi[4] * m1 + gi[5] * m2;
      const float c2 = gi[6] * m0 + gi[7] * m1 + gi[8] * m2;
      y -= b * (c0 + vv * (c1 + vv * c2));
    }
    if (a.y_out) a.y_out[ro + t] = y;
    if (a.f_out) a.f_out[ro + t] = fv + (a.out_scale * srow) * y;
    if constexpr (TRAIN) {
      const float e = y - a.target[ro + t] / srow;
      a.dy[ro + t] = a.gscale * e;
      const float s = block_sum(e * e, red);
      if (t == 0) a.loss_rows[row] = s;
    }
    __syncthreads();
  }
}
// ----------------------------------------------------------------------------
// backward: two kernels, rows strided over the workgroups (512 threads)
//
// k_bwd_out: output layer and layer 3.  dz3 is formed from dy and a3 straight
// into the LDS tile; from there the input gradient
//   dz2[p][ci] = bf16( (sum_{k', co} Wt[ci][k'*64 + co] dz3[p + k' - 2][co]) (1 - a2[p][ci]^2) )
// with Wt[ci][k'*64 + co] = W3[co][(4 - k')*64 + ci] (flipped, transposed), and
// the weight gradient
//   part[oW3 + co*320 + k*64 + ci] = sum_{rows, p} dz3[p][co] a2[p + k - 2][ci];
// the output layer's, part[oW4 + k*64 + ci] = sum dy[p - k + 2] a3[p][ci], is
// taken by the matrix units before dz3 replaces a3 in the tile (record tile R:
// row p holds dy[p - k + 2], k < 5).
// k_bwd_in: layer 2 the same way from dz2 and a1; its dz1 stays in LDS for
// the first layer's gradient.
//
// Both products of a layer read the same two position-major tiles: the input
// gradient takes the channels of a position as K (16-byte reads), the weight
// gradient the positions (transposing reads), so a tap is a shift of the row
// and needs no realignment.  Wave w takes output channels 16 (w & 3).. over
// half w >> 2 of the positions for the input gradient, and input channels
// 16 (w & 3).. by half w >> 2 of the output channels for the weight gradient.
// The next row's tiles are loaded into registers while this row is worked on.
// Apart (output layer, weight gradient and input gradient of each layer, first
// layer: six kernels that passed dz1..dz3 through memory and read every
// operand once per product) they took 917 us at 4096 rows; these two take 153
// and 114, for 0.67 GB (140 us at the rate of a copy) and 172 GFLOP (140 us).
// The matrix units are busy 0.2-0.3 of the time and LDS 0.3-0.5: what is left
// is the phases between barriers, one workgroup per CU.
// ----------------------------------------------------------------------------
constexpr int kBT = 512;
constexpr int kTile = kRowsP * kP;  // BF16 values of a tile
constexpr int kBwdOutLds = 2 * kTile * 2 + (kRowsP + 4 + kKS * kCH) * 4 + kNV * 16 * 2;
constexpr int kBwdInLds = 2 * kTile * 2 + kNV * 16 * 2;

typedef __attribute__((address_space(3))) bf16x4 lds_bf16x4;

// MFMA operand with K = 32 rows from `row` of a tile and the 16 columns from
// `col`: ds_read_b64_tr_b16 hands lane i of a group of 16 column i of the 4 x 16
// block whose row r the lanes 4r..4r+3 address.  Group g takes rows 4g.. and
// 16 + 4g.. for its 8 values of K (any order of the positions serves, both
// operands have the same): the 8 rows that half a wave reads then lie in
// different banks, rows 8g.. and 8g + 4.. meet two by two
__device__ __forceinline__ bf16x8 read_rows(const bf16* tile, int pitch, int row, int col) {
  const int l = threadIdx.x & 63;
  const bf16* p = tile + (row + (l >> 2)) * pitch + col + 4 * (l & 3);
  const bf16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((lds_bf16x4*)(__attribute__((address_space(3))) void*)p);
  const bf16x4 hi =
      __builtin_amdgcn_ds_read_tr16_b64_v4bf16((lds_bf16x4*)(__attribute__((address_space(3))) void*)(p + 16 * pitch));
  return __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
}

// fragments of weights [64][320] for output channels 16 mt .. 16 mt + 15
__device__ __forceinline__ void load_a_tile(const bf16* W, int mt, bf16x8 (&A)[10]) {
  const int lane = threadIdx.x & 63;
  const bf16* wr = W + (16 * mt + (lane & 15)) * kK + 8 * (lane >> 4);
#pragma unroll
  for (int c = 0; c < 10; ++c) A[c] = *reinterpret_cast<const bf16x8*>(wr + 32 * c);
}

// a stored row [256][64] <-> registers, 16 bytes per thread and pass
__device__ __forceinline__ void load_row(const bf16* src, bf16x8 (&v)[4]) {
#pragma unroll
  for (int u = 0; u < 4; ++u) v[u] = *reinterpret_cast<const bf16x8*>(src + 8 * (threadIdx.x + kBT * u));
}
__device__ __forceinline__ bf16* tile_at(bf16* P, int u) {
  const int i = threadIdx.x + kBT * u;
  return P + ((i >> 3) + 2) * kP + 8 * (i & 7);
}

// input gradient of a layer, this wave's channels and positions: dz P
// (A: the flipped weights), a X; out[nt] = bf16(acc (1 - a^2)) of channels
// 16 mt + 4g.. at position 16 (8 h + nt) + m
__device__ __forceinline__ void layer_data(const bf16* P, const bf16* X, const bf16x8 (&A)[10], int mt, int h,
                                           bf16x4 (&out)[8]) {
  const int lane = threadIdx.x & 63, m = lane & 15, g = lane >> 4;
  floatx4 acc[8];
#pragma unroll
  for (int nt = 0; nt < 8; ++nt) acc[nt] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int c = 0; c < 10; ++c) {
    const bf16* in = P + (128 * h + m + (c >> 1)) * kP + (c & 1) * 32 + 8 * g;
#pragma unroll
    for (int nt = 0; nt < 8; ++nt) acc[nt] = mfma(A[c], *reinterpret_cast<const bf16x8*>(in + 16 * nt * kP), acc[nt]);
  }
#pragma unroll
  for (int nt = 0; nt < 8; ++nt) {
    const bf16x4 a = *reinterpret_cast<const bf16x4*>(X + (128 * h + 16 * nt + m + 2) * kP + 16 * mt + 4 * g);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const float av = (float)a[j];
      out[nt][j] = (bf16)(acc[nt][j] * (1.f - av * av));
    }
  }
}

// weight gradient of a layer, this wave's share: acc[i][k] += dz a^T for output
// channels 16 (2 h + i).. and input channels 16 ct.., tap k; accb[i] the sums
// of dz (kept by the waves of ct = 0)
__device__ __forceinline__ void layer_weights(const bf16* P, const bf16* X, int ct, int h, floatx4 (&acc)[2][kKS],
                                              floatx4 (&accb)[2]) {
  bf16x8 ones;
#pragma unroll
  for (int j = 0; j < 8; ++j) ones[j] = (bf16)1.f;
#pragma unroll 2
  for (int c = 0; c < 8; ++c) {
    const int p0 = 32 * c;
    bf16x8 A[2];
#pragma unroll
    for (int i = 0; i < 2; ++i) A[i] = read_rows(P, kP, p0 + 2, 16 * (2 * h + i));
#pragma unroll
    for (int k = 0; k < kKS; ++k) {
      const bf16x8 B = read_rows(X, kP, p0 + k, 16 * ct);
#pragma unroll
      for (int i = 0; i < 2; ++i) acc[i][k] = mfma(A[i], B, acc[i][k]);
    }
    if (ct == 0) {
#pragma unroll
      for (int i = 0; i < 2; ++i) accb[i] = mfma(A[i], ones, accb[i]);
    }
  }
}

__device__ __forceinline__ void write_weights(float* out, int oW, int oB, int ct, int h, const floatx4 (&acc)[2][kKS],
                                              const floatx4 (&accb)[2]) {
  const int lane = threadIdx.x & 63, m = lane & 15, g = lane >> 4;
#pragma unroll
  for (int i = 0; i < 2; ++i) {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int co = 16 * (2 * h + i) + 4 * g + j;
#pragma unroll
      for (int k = 0; k < kKS; ++k) out[oW + co * kK + k * kCH + 16 * ct + m] = acc[i][k][j];
      if (ct == 0 && m == 0) out[oB + co] = accb[i][j];
    }
  }
}

__global__ __launch_bounds__(kBT) void k_bwd_out(const float* dy, const bf16* a3, const bf16* a2, const float* p,
                                                 const bf16* w3t, bf16* dz2, int rows, float* part) {
  extern __shared__ __align__(16) unsigned char lds[];
  bf16* P = reinterpret_cast<bf16*>(lds);  // dz3
  bf16* X = P + kTile;                     // a2
  float* ds = reinterpret_cast<float*>(X + kTile);  // bf(dy) at p + 2
  float* w4 = ds + kRowsP + 4;                      // bf(W4) [k][ci]
  bf16* R = reinterpret_cast<bf16*>(w4 + kK);       // [256][16]: bf(dy[p - k + 2]), k < 5
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6, m = lane & 15, g = lane >> 4;
  const int ct = wave & 3, h = wave >> 2;
  zero_pad_p(P);
  zero_pad_p(X);
  if (t < 4) ds[t < 2 ? t : kNV + t] = 0.f;
  for (int i = t; i < kK; i += kBT) w4[i] = bfr(p[oW4 + i]);
  for (int i = t; i < kNV * 16; i += kBT) R[i] = (bf16)0.f;
  bf16x8 A[10];
  load_a_tile(w3t, ct, A);
  floatx4 acc[2][kKS], accb[2];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    accb[i] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int k = 0; k < kKS; ++k) acc[i][k] = floatx4{0.f, 0.f, 0.f, 0.f};
  }
  floatx4 acc4 = floatx4{0.f, 0.f, 0.f, 0.f};  // output layer: channels 16 ct.., half h of the positions
  float gb = 0.f;
  bf16x8 n3[4], n2[4];
  float nd = 0.f;
  auto fetch = [&](int row) {
    const size_t ra = (size_t)row * kCH * kNV;
    load_row(a3 + ra, n3);
    load_row(a2 + ra, n2);
    if (t < kNV) nd = dy[(size_t)row * kNV + t];
  };
  fetch(blockIdx.x);
  __syncthreads();  // R cleared before any thread writes a record
  for (int row = blockIdx.x; row < rows; row += gridDim.x) {
    bf16x8 v3[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      v3[u] = n3[u];
      *reinterpret_cast<bf16x8*>(tile_at(P, u)) = n3[u];
      *reinterpret_cast<bf16x8*>(tile_at(X, u)) = n2[u];
    }
    if (t < kNV) {
      ds[t + 2] = bfr(nd);
#pragma unroll
      for (int k = 0; k < kKS; ++k) {
        const int q = t - 2 + k;
        if (q >= 0 && q < kNV) R[q * 16 + k] = (bf16)nd;
      }
      gb += nd;
    }
    if (row + gridDim.x < rows) fetch(row + gridDim.x);
    __syncthreads();
#pragma unroll
    for (int c = 0; c < 4; ++c)
      acc4 = mfma(read_rows(P, kP, 128 * h + 32 * c + 2, 16 * ct), read_rows(R, 16, 128 * h + 32 * c, 0), acc4);
    // four channels at a time: with the weights of all eight the kernel spills
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      floatx4 wk[kKS];
#pragma unroll
      for (int k = 0; k < kKS; ++k) wk[k] = *reinterpret_cast<const floatx4*>(w4 + k * kCH + 8 * (t & 7) + 4 * q);
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int pos = (t + kBT * u) >> 3;
        float d[kKS];
#pragma unroll
        for (int k = 0; k < kKS; ++k) d[k] = ds[pos - k + 4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          float s = 0.f;
#pragma unroll
          for (int k = 0; k < kKS; ++k) s = fmaf(wk[k][j], d[k], s);
          const float av = (float)v3[u][4 * q + j];
          v3[u][4 * q + j] = (bf16)(s * (1.f - av * av));
        }
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    __syncthreads();  // a3 read before dz3 takes its place
#pragma unroll
    for (int u = 0; u < 4; ++u) *reinterpret_cast<bf16x8*>(tile_at(P, u)) = v3[u];
    __syncthreads();
    bf16x4 out[8];
    layer_data(P, X, A, ct, h, out);
    bf16* dst = dz2 + (size_t)row * kCH * kNV + (128 * h + m) * kCH + 16 * ct + 4 * g;
#pragma unroll
    for (int nt = 0; nt < 8; ++nt) *reinterpret_cast<bf16x4*>(dst + 16 * nt * kCH) = out[nt];
    layer_weights(P, X, ct, h, acc, accb);
    __syncthreads();  // tiles read before the next row overwrites them
  }
  float* out = part + (size_t)blockIdx.x * kPart;
  write_weights(out, oW3, oB3, ct, h, acc, accb);
  // output layer: the two halves of the positions
  float* red = reinterpret_cast<float*>(lds);
  float* redb = red + 4 * 64 * 4;
  float s = gb;
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o, 64);
  if (lane == 0) redb[wave] = s;
  if (h == 1) {
#pragma unroll
    for (int j = 0; j < 4; ++j) red[(ct * 64 + lane) * 4 + j] = acc4[j];
  }
  __syncthreads();
  if (h == 0 && m < kKS) {
#pragma unroll
    for (int j = 0; j < 4; ++j) out[oW4 + m * kCH + 16 * ct + 4 * g + j] = acc4[j] + red[(ct * 64 + lane) * 4 + j];
  }
  if (t == 0) out[oB4] = (redb[0] + redb[1]) + (redb[2] + redb[3]);
}

// first layer (1 -> 64), from dz1 in P: part[oW1 + c*5 + k] = sum dz1[p][c]
// x[p + k - 2], part[oB1 + c] = sum dz1[p][c], as one product with the record
// tile R [256][16] whose row p holds x[p-2..p+2], 1 and zeros
__global__ __launch_bounds__(kBT) void k_bwd_in(const bf16* dz2, const bf16* a1, const bf16* xin, const bf16* w2t,
                                                int rows, float* part) {
  extern __shared__ __align__(16) unsigned char lds[];
  bf16* P = reinterpret_cast<bf16*>(lds);  // dz2, then dz1
  bf16* X = P + kTile;                     // a1
  bf16* R = X + kTile;
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6, m = lane & 15, g = lane >> 4;
  const int ct = wave & 3, h = wave >> 2;
  zero_pad_p(P);
  zero_pad_p(X);
  for (int i = t; i < kNV * 16; i += kBT) R[i] = (bf16)((i & 15) == kKS ? 1.f : 0.f);
  bf16x8 A[10];
  load_a_tile(w2t, ct, A);
  floatx4 acc[2][kKS], accb[2], acc1 = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    accb[i] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int k = 0; k < kKS; ++k) acc[i][k] = floatx4{0.f, 0.f, 0.f, 0.f};
  }
  bf16x8 nz[4], na[4];
  bf16 nxv = (bf16)0.f;
  auto fetch = [&](int row) {
    const size_t ra = (size_t)row * kCH * kNV;
    load_row(dz2 + ra, nz);
    load_row(a1 + ra, na);
    if (t < kNV) nxv = xin[(size_t)row * kNV + t];
  };
  fetch(blockIdx.x);
  __syncthreads();  // R cleared before any thread writes a record
  for (int row = blockIdx.x; row < rows; row += gridDim.x) {
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      *reinterpret_cast<bf16x8*>(tile_at(P, u)) = nz[u];
      *reinterpret_cast<bf16x8*>(tile_at(X, u)) = na[u];
    }
    if (t < kNV) {
#pragma unroll
      for (int k = 0; k < kKS; ++k) {
        const int q = t + 2 - k;
        if (q >= 0 && q < kNV) R[q * 16 + k] = nxv;
      }
    }
    if (row + gridDim.x < rows) fetch(row + gridDim.x);
    __syncthreads();
    bf16x4 out[8];
    layer_data(P, X, A, ct, h, out);
    layer_weights(P, X, ct, h, acc, accb);
    __syncthreads();  // dz2 read before dz1 takes its place
#pragma unroll
    for (int nt = 0; nt < 8; ++nt)
      *reinterpret_cast<bf16x4*>(P + (128 * h + 16 * nt + m + 2) * kP + 16 * ct + 4 * g) = out[nt];
    __syncthreads();
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      const int p0 = 128 * h + 32 * c;
      acc1 = mfma(read_rows(P, kP, p0 + 2, 16 * ct), read_rows(R, 16, p0, 0), acc1);
    }
    __syncthreads();
  }
  float* out = part + (size_t)blockIdx.x * kPart;
  write_weights(out, oW2, oB2, ct, h, acc, accb);
  // the two halves of the positions
  float* red = reinterpret_cast<float*>(lds);
  if (h == 1) {
#pragma unroll
    for (int j = 0; j < 4; ++j) red[(ct * 64 + lane) * 4 + j] = acc1[j];
  }
  __syncthreads();
  if (h == 0) {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const float s = acc1[j] + red[(ct * 64 + lane) * 4 + j];
      const int c = 16 * ct + 4 * g + j;
      if (m < kKS) out[oW1 + c * kKS + m] = s;
      if (m == kKS) out[oB1 + c] = s;
    }
  }
}

// grad[i] = sum over workgroups of part[wg][i], 256 parameters per workgroup
// and a sixteenth of the partials per wave, 16 loads in flight; the workgroup
// past the parameters forms loss = sum of loss_rows * lscale.  (256 partials:
// one thread per parameter with one load at a time 99 us, with 16 loads in
// flight 33 us, with 16-byte ones here 10.)
constexpr int kReduceWG = (kPart + 255) / 256;

__global__ __launch_bounds__(1024) void k_reduce(const float* part, int nwg, float* grad, const float* loss_rows,
                                                 int rows, float lscale, float* loss) {
  __shared__ floatx4 red[16][64];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  if (blockIdx.x == kReduceWG) {
    float s = 0.f;
    for (int r = threadIdx.x; r < rows; r += 1024) s += loss_rows[r];
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o, 64);
    float* rs = reinterpret_cast<float*>(red);
    if (lane == 0) rs[wave] = s;
    __syncthreads();
    if (threadIdx.x == 0) {
#pragma unroll
      for (int o = 8; o > 0; o >>= 1)
        for (int w = 0; w < o; ++w) rs[w] += rs[w + o];
      *loss = rs[0] * lscale;
    }
    return;
  }
  const int i = 256 * blockIdx.x + 4 * lane;
  floatx4 acc[4];
#pragma unroll
  for (int u = 0; u < 4; ++u) acc[u] = floatx4{0.f, 0.f, 0.f, 0.f};
  if (i < kPart) {
    for (int w = wave; w < nwg; w += 256) {
      floatx4 v[16];
#pragma unroll
      for (int u = 0; u < 16; ++u) {
        const int q = w + 16 * u;
        v[u] = *reinterpret_cast<const floatx4*>(part + (size_t)(q < nwg ? q : w) * kPart + i);
      }
#pragma unroll
      for (int u = 0; u < 16; ++u)
        if (w + 16 * u < nwg) acc[u & 3] += v[u];
    }
  }
  red[wave][lane] = (acc[0] + acc[1]) + (acc[2] + acc[3]);
  __syncthreads();
  if (wave >= 4) return;
  // parameter 256 blockIdx + threadIdx of the 16 waves' sums
  const float* rs = reinterpret_cast<const float*>(red) + threadIdx.x;
  float s = 0.f;
#pragma unroll
  for (int w = 0; w < 16; ++w) s += rs[256 * w];
  const int j = 256 * blockIdx.x + threadIdx.x;
  if (j < kParams) grad[j] = s;
}

// BF16 copies of W2, W3 ([co][k*64+ci]) and their flipped transposes
// ([ci][k'*64+co] = W[co][(4-k')*64+ci])
__device__ __forceinline__ void write_copies(int i, float v, bf16* w2, bf16* w3, bf16* w2t, bf16* w3t) {
  if (i >= oW2 && i < oB2) {
    const int j = i - oW2, co = j / kK, kk = j % kK, k = kk / kCH, ci = kk % kCH;
    w2[j] = (bf16)v;
    w2t[ci * kK + (4 - k) * kCH + co] = (bf16)v;
  } else if (i >= oW3 && i < oB3) {
    const int j = i - oW3, co = j / kK, kk = j % kK, k = kk / kCH, ci = kk % kCH;
    w3[j] = (bf16)v;
    w3t[ci * kK + (4 - k) * kCH + co] = (bf16)v;
  }
}

__global__ __launch_bounds__(256) void k_refresh(const float* p, bf16* w2, bf16* w3, bf16* w2t, bf16* w3t) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i < kParams) write_copies(i, p[i], w2, w3, w2t, w3t);
}

__global__ __launch_bounds__(256) void k_adam(float* p, float* mo, float* ve, const float* grad, float lr, float b1,
                                              float b2, float eps, float c1, float c2, bf16* w2, bf16* w3, bf16* w2t,
                                              bf16* w3t) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i >= kParams) return;
  const float gi = grad[i];
  const float m = b1 * mo[i] + (1.f - b1) * gi;
  const float v = b2 * ve[i] + (1.f - b2) * gi * gi;
  mo[i] = m;
  ve[i] = v;
  const float np = p[i] - lr * (m / c1) / (sqrtf(v / c2) + eps);
  p[i] = np;
  write_copies(i, np, w2, w3, w2t, w3t);
}

}  // namespace

struct vpfc_net_s {
  int max_rows = 0;
  float in_scale = 1.f, out_scale = 1.f;
  float* bg = nullptr;       // [256] background profile (device)
  bool has_bg = false;
  float* cons = nullptr;     // [256 * 4 + 9] conservation projection (device)
  bool has_cons = false;
  int adam_t = 0;
  float* p = nullptr;
  float* mo = nullptr;
  float* ve = nullptr;
  float* grad = nullptr;
  float* part = nullptr;
  bf16 *w2 = nullptr, *w3 = nullptr, *w2t = nullptr, *w3t = nullptr;
  bf16 *xin = nullptr, *a1 = nullptr, *a2 = nullptr, *a3 = nullptr, *dz2 = nullptr;
  float* dy = nullptr;
  float* loss_rows = nullptr;
  float* loss = nullptr;
  std::vector<void*> allocs;
  ~vpfc_net_s() {
    for (void* q : allocs) (void)hipFree(q);
  }
};

namespace {

template <class P>
int nalloc(vpfc_net_s* n, P** out, size_t bytes) {
  void* q = nullptr;
  hipError_t e = hipMalloc(&q, bytes > 0 ? bytes : 16);
  if (e != hipSuccess) return fail(VPFP_EHIP, std::string("hipMalloc: ") + hipGetErrorString(e));
  n->allocs.push_back(q);
  *out = reinterpret_cast<P*>(q);
  return VPFP_OK;
}

int launched() {
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return fail(VPFP_EHIP, std::string("kernel launch: ") + hipGetErrorString(e));
  return VPFP_OK;
}

int set_lds_all() {
  static bool done = false;
  if (done) return VPFP_OK;
  FC_HIP(hipFuncSetAttribute((const void*)k_fwd<false>, hipFuncAttributeMaxDynamicSharedMemorySize, kFwdLds));
  FC_HIP(hipFuncSetAttribute((const void*)k_fwd<true>, hipFuncAttributeMaxDynamicSharedMemorySize, kFwdLds));
  FC_HIP(hipFuncSetAttribute((const void*)k_bwd_out, hipFuncAttributeMaxDynamicSharedMemorySize, kBwdOutLds));
  FC_HIP(hipFuncSetAttribute((const void*)k_bwd_in, hipFuncAttributeMaxDynamicSharedMemorySize, kBwdInLds));
  done = true;
  return VPFP_OK;
}

hipStream_t S(void* s) { return reinterpret_cast<hipStream_t>(s); }

// rows are strided over the workgroups: 3072 = 4 x the 3 x 256 that are
// resident at once (measured 5 % faster than 4096, which leaves a partial wave)
int fwd_grid(int rows) { return rows < 3072 ? rows : 3072; }

int check_net(vpfc_net_t n) { return n ? VPFP_OK : fail(VPFP_EBADARG, "null network"); }

FwdArgs fwd_args(vpfc_net_t n, const float* x, int rows) {
  FwdArgs a;
  std::memset(&a, 0, sizeof(a));
  a.f = x;
  a.rows = rows;
  a.in_scale = n->in_scale;
  a.out_scale = n->out_scale;
  a.p = n->p;
  a.w2 = n->w2;
  a.w3 = n->w3;
  a.bg = n->has_bg ? n->bg : nullptr;
  a.cons = n->has_cons ? n->cons : nullptr;
  return a;
}

int run_fwd(const FwdArgs& a, hipStream_t s) {
  if (a.rows == 0) return VPFP_OK;
  if (int rc = set_lds_all()) return rc;
  if (a.dy)
    hipLaunchKernelGGL(k_fwd<true>, dim3(fwd_grid(a.rows)), dim3(256), kFwdLds, s, a);
  else
    hipLaunchKernelGGL(k_fwd<false>, dim3(fwd_grid(a.rows)), dim3(256), kFwdLds, s, a);
  return launched();
}

int gradients(vpfc_net_t n, const float* x, const float* target, int rows, float* grad, float* loss,
              hipStream_t s) {
  FwdArgs a = fwd_args(n, x, rows);
  a.cons = nullptr;  // the backward kernels differentiate the unprojected output
  a.xin = n->xin;
  a.a1 = n->a1;
  a.a2 = n->a2;
  a.a3 = n->a3;
  a.target = target;
  const float count = (float)rows * (float)kNV;
  a.gscale = 2.f / count;
  a.dy = n->dy;
  a.loss_rows = n->loss_rows;
  if (int rc = run_fwd(a, s)) return rc;
  const int G = rows < kPartWG ? rows : kPartWG;
  hipLaunchKernelGGL(k_bwd_out, dim3(G), dim3(kBT), kBwdOutLds, s, n->dy, n->a3, n->a2, n->p, n->w3t, n->dz2, rows,
                     n->part);
  if (int rc = launched()) return rc;
  hipLaunchKernelGGL(k_bwd_in, dim3(G), dim3(kBT), kBwdInLds, s, n->dz2, n->a1, n->xin, n->w2t, rows, n->part);
  if (int rc = launched()) return rc;
  hipLaunchKernelGGL(k_reduce, dim3(kReduceWG + (loss ? 1 : 0)), dim3(1024), 0, s, n->part, G, grad, n->loss_rows, rows,
                     1.f / count, loss);
  return launched();
}

}  // namespace

extern "C" {

const char* vpfc_last_error(void) { return g_err.c_str(); }

int vpfc_create(int max_rows, vpfc_net_t* out) {
  if (!out) return fail(VPFP_EBADARG, "null argument");
  *out = nullptr;
  if (max_rows < 1 || max_rows > (1 << 20)) return fail(VPFP_EBADARG, "max_rows must be in [1, 2^20]");
  auto* n = new vpfc_net_s();
  n->max_rows = max_rows;
  const size_t R = (size_t)max_rows, act = R * kCH * kNV * sizeof(bf16);
  int rc = VPFP_OK;
  if (!rc) rc = nalloc(n, &n->p, sizeof(float) * kParams);
  if (!rc) rc = nalloc(n, &n->mo, sizeof(float) * kParams);
  if (!rc) rc = nalloc(n, &n->ve, sizeof(float) * kParams);
  if (!rc) rc = nalloc(n, &n->grad, sizeof(float) * kParams);
  if (!rc) rc = nalloc(n, &n->part, sizeof(float) * kPart * kPartWG);
  if (!rc) rc = nalloc(n, &n->w2, sizeof(bf16) * kCH * kK);
  if (!rc) rc = nalloc(n, &n->w3, sizeof(bf16) * kCH * kK);
  if (!rc) rc = nalloc(n, &n->w2t, sizeof(bf16) * kCH * kK);
  if (!rc) rc = nalloc(n, &n->w3t, sizeof(bf16) * kCH * kK);
  if (!rc) rc = nalloc(n, &n->xin, R * kNV * sizeof(bf16));
  if (!rc) rc = nalloc(n, &n->a1, act);
  if (!rc) rc = nalloc(n, &n->a2, act);
  if (!rc) rc = nalloc(n, &n->a3, act);
  if (!rc) rc = nalloc(n, &n->dz2, act);
  if (!rc) rc = nalloc(n, &n->dy, R * kNV * sizeof(float));
  if (!rc) rc = nalloc(n, &n->loss_rows, R * sizeof(float));
  if (!rc) rc = nalloc(n, &n->loss, sizeof(float));
  if (!rc) rc = nalloc(n, &n->bg, sizeof(float) * kNV);
  if (!rc) rc = nalloc(n, &n->cons, sizeof(float) * (4 * kNV + 9));
  if (!rc) {
    std::vector<float> z(kParams, 0.f);
    hipError_t e = hipMemcpy(n->p, z.data(), sizeof(float) * kParams, hipMemcpyHostToDevice);
    if (e == hipSuccess) e = hipMemcpy(n->mo, z.data(), sizeof(float) * kParams, hipMemcpyHostToDevice);
    if (e == hipSuccess) e = hipMemcpy(n->ve, z.data(), sizeof(float) * kParams, hipMemcpyHostToDevice);
    if (e != hipSuccess) rc = fail(VPFP_EHIP, std::string("hipMemcpy: ") + hipGetErrorString(e));
  }
  if (!rc) {
    hipLaunchKernelGGL(k_refresh, dim3((kParams + 255) / 256), dim3(256), 0, 0, n->p, n->w2, n->w3, n->w2t, n->w3t);
    rc = launched();
    if (!rc) {
      hipError_t e = hipDeviceSynchronize();
      if (e != hipSuccess) rc = fail(VPFP_EHIP, std::string("hipDeviceSynchronize: ") + hipGetErrorString(e));
    }
  }
  if (rc) {
    delete n;
    return rc;
  }
  *out = n;
  return VPFP_OK;
}

int vpfc_destroy(vpfc_net_t n) {
  if (!n) return VPFP_OK;
  (void)hipDeviceSynchronize();
  delete n;
  return VPFP_OK;
}

int vpfc_set_params(vpfc_net_t n, const float* host) {
  if (int rc = check_net(n)) return rc;
  if (!host) return fail(VPFP_EBADARG, "null parameters");
  std::vector<float> z(kParams, 0.f);
  FC_HIP(hipDeviceSynchronize());
  FC_HIP(hipMemcpy(n->p, host, sizeof(float) * kParams, hipMemcpyHostToDevice));
  FC_HIP(hipMemcpy(n->mo, z.data(), sizeof(float) * kParams, hipMemcpyHostToDevice));
  FC_HIP(hipMemcpy(n->ve, z.data(), sizeof(float) * kParams, hipMemcpyHostToDevice));
  n->adam_t = 0;
  hipLaunchKernelGGL(k_refresh, dim3((kParams + 255) / 256), dim3(256), 0, 0, n->p, n->w2, n->w3, n->w2t, n->w3t);
  if (int rc = launched()) return rc;
  FC_HIP(hipDeviceSynchronize());
  return VPFP_OK;
}

int vpfc_get_params(vpfc_net_t n, float* host) {
  if (int rc = check_net(n)) return rc;
  if (!host) return fail(VPFP_EBADARG, "null parameters");
  FC_HIP(hipDeviceSynchronize());
  FC_HIP(hipMemcpy(host, n->p, sizeof(float) * kParams, hipMemcpyDeviceToHost));
  return VPFP_OK;
}

int vpfc_set_scales(vpfc_net_t n, float in_scale, float out_scale) {
  if (int rc = check_net(n)) return rc;
  if (!std::isfinite(in_scale) || !std::isfinite(out_scale)) return fail(VPFP_EBADARG, "non-finite scale");
  n->in_scale = in_scale;
  n->out_scale = out_scale;
  return VPFP_OK;
}

int vpfc_set_background(vpfc_net_t n, const float* host_bg) {
  if (int rc = check_net(n)) return rc;
  FC_HIP(hipDeviceSynchronize());
  if (host_bg) FC_HIP(hipMemcpy(n->bg, host_bg, sizeof(float) * kNV, hipMemcpyHostToDevice));
  n->has_bg = host_bg != nullptr;
  return VPFP_OK;
}

int vpfc_set_conservation(vpfc_net_t n, const double* v, const double* bg) {
  if (int rc = check_net(n)) return rc;
  FC_HIP(hipDeviceSynchronize());
  if (!v || !bg) {
    n->has_cons = false;
    return VPFP_OK;
  }
  // G[l][k] = sum_v w v^(l+k) bg(v) with trapz weights (1, ends 1/2)
  double G[3][3] = {{0, 0, 0}, {0, 0, 0}, {0, 0, 0}};
  std::vector<float> h(4 * kNV + 9, 0.f);
  for (int j = 0; j < kNV; ++j) {
    const double w = (j == 0 || j == kNV - 1) ? 0.5 : 1.0;
    double pw[5] = {1, v[j], v[j] * v[j], v[j] * v[j] * v[j], v[j] * v[j] * v[j] * v[j]};
    for (int l = 0; l < 3; ++l)
      for (int k = 0; k < 3; ++k) G[l][k] += w * pw[l + k] * bg[j];
    h[j] = (float)v[j];
    h[kNV + j] = (float)w;
    h[2 * kNV + j] = (float)bg[j];
  }
  // inverse of the symmetric 3x3 by cofactors
  const double c00 = G[1][1] * G[2][2] - G[1][2] * G[2][1], c01 = G[1][2] * G[2][0] - G[1][0] * G[2][2],
               c02 = G[1][0] * G[2][1] - G[1][1] * G[2][0];
  const double det = G[0][0] * c00 + G[0][1] * c01 + G[0][2] * c02;
  if (!(std::fabs(det) > 0.0)) return fail(VPFP_EBADARG, "singular moment matrix of the background");
  const double inv[9] = {c00 / det,
                         (G[0][2] * G[2][1] - G[0][1] * G[2][2]) / det,
                         (G[0][1] * G[1][2] - G[0][2] * G[1][1]) / det,
                         c01 / det,
                         (G[0][0] * G[2][2] - G[0][2] * G[2][0]) / det,
                         (G[0][2] * G[1][0] - G[0][0] * G[1][2]) / det,
                         c02 / det,
                         (G[0][1] * G[2][0] - G[0][0] * G[2][1]) / det,
                         (G[0][0] * G[1][1] - G[0][1] * G[1][0]) / det};
  for (int i = 0; i < 9; ++i) h[4 * kNV + i] = (float)inv[i];
  FC_HIP(hipMemcpy(n->cons, h.data(), sizeof(float) * h.size(), hipMemcpyHostToDevice));
  n->has_cons = true;
  return VPFP_OK;
}

int vpfc_forward(vpfc_net_t n, const float* x, int rows, float* y, void* stream) {
  if (int rc = check_net(n)) return rc;
  if (rows < 0) return fail(VPFP_EBADARG, "negative row count");
  if (rows && (!x || !y)) return fail(VPFP_EBADARG, "null array");
  FwdArgs a = fwd_args(n, x, rows);
  a.y_out = y;
  return run_fwd(a, S(stream));
}

int vpfc_apply(vpfc_net_t n, float* f, int rows, void* stream) {
  if (int rc = check_net(n)) return rc;
  if (rows < 0) return fail(VPFP_EBADARG, "negative row count");
  if (rows && !f) return fail(VPFP_EBADARG, "null array");
  FwdArgs a = fwd_args(n, f, rows);
  a.f_out = f;
  return run_fwd(a, S(stream));
}

int vpfc_gradients(vpfc_net_t n, const float* x, const float* target, int rows, float* grad, float* loss,
                   void* stream) {
  if (int rc = check_net(n)) return rc;
  if (rows < 1 || rows > n->max_rows) return fail(VPFP_EBADARG, "rows must be in [1, max_rows]");
  if (!x || !target || !grad) return fail(VPFP_EBADARG, "null array");
  return gradients(n, x, target, rows, grad, loss, S(stream));
}

int vpfc_train_step(vpfc_net_t n, const float* x, const float* target, int rows, float lr, float beta1,
                    float beta2, float eps, float* loss, void* stream) {
  if (int rc = check_net(n)) return rc;
  if (rows < 1 || rows > n->max_rows) return fail(VPFP_EBADARG, "rows must be in [1, max_rows]");
  if (!x || !target) return fail(VPFP_EBADARG, "null array");
  if (!(beta1 >= 0.f && beta1 < 1.f && beta2 >= 0.f && beta2 < 1.f && eps > 0.f))
    return fail(VPFP_EBADARG, "Adam needs 0 <= beta < 1 and eps > 0");
  const hipStream_t s = S(stream);
  if (int rc = gradients(n, x, target, rows, n->grad, loss ? loss : n->loss, s)) return rc;
  n->adam_t += 1;
  const float c1 = 1.f - std::pow(beta1, (float)n->adam_t), c2 = 1.f - std::pow(beta2, (float)n->adam_t);
  hipLaunchKernelGGL(k_adam, dim3((kParams + 255) / 256), dim3(256), 0, s, n->p, n->mo, n->ve, n->grad, lr, beta1,
                     beta2, eps, c1, c2, n->w2, n->w3, n->w2t, n->w3t);
  return launched();
}

}  // extern "C"
