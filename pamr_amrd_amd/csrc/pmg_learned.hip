// pmg_learned.hip -- the learned smoother / warm-start network on gfx950.
//
// Network: 3 layers of 3x3x3 convolutions, 1 -> H -> H -> 1 channels
// (H = 16), GELU (tanh form) after layers 1 and 2, zero padding.  It maps a
// normalised residual r/s to a normalised error estimate; the solver applies
// u += s * h^2 * N(r/s) and keeps the step only when the FP64 residual says
// it contracts (pmg_solver's learned mode).
//
// Kernels are implicit GEMMs on the MFMA units in BF16 with FP32 accumulation,
// the same ones for inference and training (their epilogues differ): tiles of
// (x, y) columns marching z with the input planes in LDS.  The hidden layer
// has 16 channels and tap pairs along K, layer 1 the taps of its one input
// channel along K, layer 3 the taps of its one output channel as columns.
// The master weights are padded to 16 x 16 channels per tap (the padding
// stays exactly zero under training).  Activations are channel-last BF16
// [point][16]; pre-activations FP32.
//
// Training kernels: backward-data is the same convolution with flipped taps
// and transposed weights, fused with the GELU derivative; backward-weight is
// a GEMM over points (K = points) per tap with per-block partials folded
// deterministically; Adam on FP32 master weights.
#include <cmath>
#include <cstring>
#include <vector>

#include "pmg_common.h"
#include "../../include/pamr_mg_gpu.h"

using namespace pmg;

namespace {

typedef short bf16x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float floatx4 __attribute__((ext_vector_type(4)));

constexpr int NC = 16;      // channels (padded)
constexpr int NTAP = 27;

// master layout per layer: W[tap][ci][co] (27*256 floats) then bias[co]
// (16 floats), i.e. 28 rows of 256 with the bias in row 27, entries 0..15
constexpr int LAYER_FLOATS = (NTAP + 1) * 256;

__host__ __device__ inline uint16_t f2bf(float f) {
  uint32_t u;
  __builtin_memcpy(&u, &f, 4);
  if ((u & 0x7f800000u) == 0x7f800000u) return (uint16_t)(u >> 16);  // inf / nan
  u += 0x7fffu + ((u >> 16) & 1u);  // round to nearest even
  return (uint16_t)(u >> 16);
}

struct Geom {
  int nx, ny, nz, nb;  // box shape and number of boxes (batch)
};

// ---------------------------------------------------------------------------
// MFMA lane layout self-test: D = A * B for 16x16 bf16 operands.  Lane l
// holds A[l%16][4*(l/16)+j], B[4*(l/16)+j][l%16] and D[4*(l/16)+i][l%16].
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(64) void k_mfma_probe(const uint16_t *A, const uint16_t *B, float *D) {
  const int l = threadIdx.x, m = l & 15, g = l >> 4;
  bf16x4 a, b;
  for (int j = 0; j < 4; j++) {
    a[j] = (short)A[m * 16 + 4 * g + j];
    b[j] = (short)B[(4 * g + j) * 16 + m];
  }
  floatx4 acc = {0.f, 0.f, 0.f, 0.f};
  acc = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, b, acc, 0, 0, 0);
  for (int i = 0; i < 4; i++) D[(4 * g + i) * 16 + m] = acc[i];
}

// The K = 32 form (v_mfma_f32_16x16x32_bf16): lane l holds A[l%16][8*(l/16)+j]
// and B[8*(l/16)+j][l%16], j = 0..7; D as above.
__global__ __launch_bounds__(64) void k_mfma32_probe(const uint16_t *A, const uint16_t *B, float *D) {
  const int l = threadIdx.x, m = l & 15, g = l >> 4;
  uint16_t a[8], b[8];
  for (int j = 0; j < 8; j++) {
    a[j] = A[m * 32 + 8 * g + j];
    b[j] = B[(8 * g + j) * 16 + m];
  }
  bf16x8 av, bv;
  __builtin_memcpy(&av, a, 16);
  __builtin_memcpy(&bv, b, 16);
  floatx4 acc = {0.f, 0.f, 0.f, 0.f};
  acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(av, bv, acc, 0, 0, 0);
  for (int i = 0; i < 4; i++) D[(4 * g + i) * 16 + m] = acc[i];
}

// two floats to two BF16 in one word, rounded to nearest even (one instruction)
__device__ inline unsigned pk_bf16(float lo, float hi) {
  typedef float f2 __attribute__((ext_vector_type(2)));
  typedef __bf16 b2 __attribute__((ext_vector_type(2)));
  const b2 r = __builtin_convertvector(f2{lo, hi}, b2);
  unsigned w;
  __builtin_memcpy(&w, &r, 4);
  return w;
}

// GELU (tanh form) through the logistic function: 0.5 x (1 + tanh u) = x s(u)
// with s = 1 / (1 + e^(-2u)), u = k (x + 0.044715 x^3), the constants folded
// into the power of two.  Its derivative is s + 2 x s (1 - s) u'.  Against 64
// bits the value is within 4 units in the last place for |x| <= 2, 9 for |x| <= 4
// and 33 down to -6, where it is 1e-10 (the exponent's rounding grows with |x|; the
// form with tanhf cancels there, 10^4 units at -4), the derivative within 2e-6:
// all far below the BF16 they are rounded to.  The epilogue's vector instructions, not the matrix units or LDS,
// bounded the hidden layer: with the IEEE division, tanhf and a software
// rounding to BF16 it took 0.27 of its 0.61 ms at 257^3.
__device__ inline float logistic2(float x) {
  const float c1 = -2.0f * 0.7978845608028654f * 1.4426950408889634f, c2 = c1 * 0.044715f;
  return __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(x * fmaf(c2, x * x, c1)));
}
__device__ inline float gelu_f(float x) { return x * logistic2(x); }
__device__ inline float gelu_grad_f(float x) {
  const float k2 = 2.0f * 0.7978845608028654f, k6 = k2 * 3.0f * 0.044715f;
  const float s = logistic2(x);
  return s + x * s * (1.0f - s) * fmaf(k6, x * x, k2);
}

// What a convolution tile does with its sums (they start from the bias).  The products are taken with
// the weights as the A operand, so lane (m, grp) holds channels 4grp .. +3 of
// point m of a 16-point segment starting at element `row`: its activations
// are one 8-byte store and its pre-activations one 16-byte store, channel-last
// and contiguous over the wave, with no exchange between lanes.
//   EPI 0: v -> Z (FP32), A = bf16(gelu(v))        (training)
//   EPI 2: A = bf16(v * gelu'(aux)), no bias       (backward data)
//   EPI 3: A = bf16(gelu(v))                       (inference)
template <int EPI>
__device__ __forceinline__ void conv_epilogue(floatx4 v, floatx4 aux, float *__restrict__ Z, uint16_t *__restrict__ A,
                                              size_t row, int npts) {
  const int lane = threadIdx.x & 63, m = lane & 15, grp = lane >> 4;
  if (m >= npts) return;
  const int p = m * NC + 4 * grp;
  float o[4];
#pragma unroll
  for (int i = 0; i < 4; i++) o[i] = EPI == 2 ? v[i] * gelu_grad_f(aux[i]) : gelu_f(v[i]);
  if constexpr (EPI == 0) *(floatx4 *)(Z + row * NC + p) = v;
  *(uint2 *)(A + row * NC + p) = make_uint2(pk_bf16(o[0], o[1]), pk_bf16(o[2], o[3]));
}
template <int EPI>
__device__ __forceinline__ floatx4 conv_aux(const float *__restrict__ aux, size_t row, int npts) {
  const int lane = threadIdx.x & 63, m = lane & 15, grp = lane >> 4;
  if constexpr (EPI == 2) return *(const floatx4 *)(aux + row * NC + (m < npts ? m * NC + 4 * grp : 0));
  else return floatx4{0.f, 0.f, 0.f, 0.f};
}

// The 16 -> 16 convolutions with the input staged in LDS: a block owns a
// CTX x CTY tile of (x, y) columns and marches ZC planes in z, keeping a ring
// of 4 input planes (tile plus a 1-point halo, 16 BF16 channels = 32 B per
// point, zero outside the box) in LDS.  Wave w computes rows 2w, 2w+1 of the
// tile, two 16-point segments each.  The 27 taps go in pairs through the K =
// 32 MFMA (14 per segment and plane, the last pair padded with zeros): lanes
// 0-31 read 16 channel bytes of the pair's first tap, lanes 32-63 of its
// second, as one 16-byte LDS read each; the 14 weight fragments stay in
// registers.  One barrier per plane: plane z+2 is stored into the slot plane
// z-2 left at the start of step z, plane z+3 is fetched into registers, and
// step z reads z-1..z+1.  The fetches are unconditional (positions outside
// the box read element 0 and are stored as zero), so they stay in flight
// across the step.
constexpr int CTX = 32, CTY = 8, CLX = CTX + 2, CLY = CTY + 2;
constexpr int CCHUNK = CLY * CLX * 2;                  // 16-byte chunks per staged plane
constexpr int CLOAD = (CCHUNK + 255) / 256;            // per thread
constexpr int NPAIR = (NTAP + 1) / 2;                  // tap pairs of the K = 32 form

// the wave's index in its block, in a scalar register: rows and row addresses
// are then scalar arithmetic
__device__ __forceinline__ int wave_ix() { return __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6); }

struct ConvTile {
  int x0, y0, z0, z1, b;
};
__device__ __forceinline__ ConvTile conv_tile(const Geom &g, int tx_, int ty_, int zc_) {
  const int ntx = (g.nx + tx_ - 1) / tx_, nty = (g.ny + ty_ - 1) / ty_, nzc = (g.nz + zc_ - 1) / zc_;
  int t = xcd_tile(blockIdx.x, gridDim.x);  // neighbouring tiles share an L2
  ConvTile c;
  c.x0 = (t % ntx) * tx_;
  t /= ntx;
  c.y0 = (t % nty) * ty_;
  t /= nty;
  c.z0 = (t % nzc) * zc_;
  c.b = t / nzc;
  c.z1 = min(g.nz, c.z0 + zc_);
  return c;
}
inline unsigned conv_blocks(const Geom &g, int tx_, int ty_, int zc_) {
  return (unsigned)((size_t)((g.nx + tx_ - 1) / tx_) * ((g.ny + ty_ - 1) / ty_) * ((g.nz + zc_ - 1) / zc_) * g.nb);
}

template <int EPI>
__global__ __launch_bounds__(256) void k_conv16_tile(const uint16_t *__restrict__ X,
                                                     const uint16_t *__restrict__ Wp,
                                                     const float *__restrict__ bias, const float *__restrict__ aux,
                                                     float *__restrict__ Zout, uint16_t *__restrict__ Aout, Geom g,
                                                     int zc) {
  __shared__ uint4 sX[4][CLY][CLX][2];
  __shared__ uint4 sZero;  // the operand of the tap past the 27th
  if (threadIdx.x == 0) sZero = make_uint4(0u, 0u, 0u, 0u);
  const ConvTile T = conv_tile(g, CTX, CTY, zc);
  const int x0 = T.x0, y0 = T.y0, z0 = T.z0, z1 = T.z1;
  const size_t box = (size_t)g.nx * g.ny * g.nz;
  const uint16_t *Xb = X + (size_t)T.b * box * NC;
  const int lane = threadIdx.x & 63, w = wave_ix(), m = lane & 15, grp = lane >> 4;
  uint4 reg[CLOAD];
  // element offset of this thread's chunks within a plane (64 bits: a plane of 16
  // channels may hold more than 2^31 elements), 0 for those outside the box
  size_t off[CLOAD];
  unsigned in = 0;
#pragma unroll
  for (int q = 0; q < CLOAD; q++) {
    const int idx = (int)threadIdx.x + q * 256;
    const int ly = idx / (CLX * 2), rem = idx % (CLX * 2), lx = rem >> 1, h = rem & 1;
    const int gx = x0 - 1 + lx, gy = y0 - 1 + ly;
    const bool ok = idx < CCHUNK && gx >= 0 && gx < g.nx && gy >= 0 && gy < g.ny;
    off[q] = ok ? ((size_t)gy * g.nx + gx) * NC + 8 * h : 0;
    in |= (unsigned)ok << q;
  }
  const size_t plane = (size_t)g.nx * g.ny * NC;
  auto fetch = [&](int k) {
    const uint16_t *Xk = Xb + (k >= 0 && k < g.nz ? (size_t)k * plane : 0);
#pragma unroll
    for (int q = 0; q < CLOAD; q++) reg[q] = *(const uint4 *)(Xk + off[q]);
  };
  auto store = [&](int k) {
    uint4 *S = &sX[k & 3][0][0][0];
    const bool kin = k >= 0 && k < g.nz;
#pragma unroll
    for (int q = 0; q < CLOAD; q++) {
      const int idx = (int)threadIdx.x + q * 256;
      if (idx < CCHUNK) S[idx] = kin && ((in >> q) & 1) ? reg[q] : make_uint4(0u, 0u, 0u, 0u);
    }
  };
  // the 14 weight fragments stay in registers for the whole march
  bf16x8 wk[NPAIR];
#pragma unroll
  for (int pr = 0; pr < NPAIR; pr++) wk[pr] = *(const bf16x8 *)(Wp + ((size_t)pr * 64 + lane) * 8);
  const int half = grp & 1, second = grp >> 1;  // channel half; first or second tap of the pair
  const floatx4 bm = EPI == 2 ? floatx4{0.f, 0.f, 0.f, 0.f} : *(const floatx4 *)(bias + 4 * grp);
  fetch(z0 - 1);
  store(z0 - 1);
  fetch(z0);
  store(z0);
  fetch(z0 + 1);
  store(z0 + 1);
  fetch(z0 + 2);
  __syncthreads();
  for (int z = z0; z < z1; z++) {
    store(z + 2);  // the slot of plane z-2, free since the barrier ending step z-1
    fetch(z + 3);
    floatx4 acc[4], ax[4];
    size_t row[4];
    int npts[4];  // points of the segment inside the box, 0 when there are none
#pragma unroll
    for (int q = 0; q < 4; q++) {
      const int y = y0 + 2 * w + (q >> 1), xs = x0 + 16 * (q & 1);
      npts[q] = y < g.ny && xs < g.nx ? min(16, g.nx - xs) : 0;
      row[q] = npts[q] ? (size_t)T.b * box + ((size_t)z * g.ny + y) * g.nx + xs : 0;
      acc[q] = bm;
      ax[q] = conv_aux<EPI>(aux, row[q], npts[q]);
    }
#pragma unroll
    for (int pr = 0; pr < NPAIR; pr++) {
      const int tap = 2 * pr + second;
      const bool live = tap < NTAP;
      const int tp = live ? tap : 0;
      const int dx = tp % 3 - 1, dy = (tp / 3) % 3 - 1, dz = tp / 9 - 1;
      const int slot = (z + dz) & 3;
#pragma unroll
      for (int q = 0; q < 4; q++) {
        const int r = 2 * w + (q >> 1), sg = q & 1;
        const uint4 *S = &sX[slot][r + 1 + dy][16 * sg + m + 1 + dx][half];
        const bf16x8 a = *(const bf16x8 *)(live ? S : &sZero);
        acc[q] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wk[pr], a, acc[q], 0, 0, 0);
      }
    }
#pragma unroll
    for (int q = 0; q < 4; q++)
      if (npts[q]) conv_epilogue<EPI>(acc[q], ax[q], Zout, Aout, row[q], npts[q]);  // uniform per wave
    __syncthreads();
  }
}

// Convolutions of one input channel (layer 1, and the backward data of layer
// 3) on the same tiles: the plane tile of bf16(scale * x) (zero outside the
// box) is staged in a 4-plane LDS ring, each word holding the point and its
// east neighbour, so that two words two apart are the four points x-1 .. x+2.
// One K = 16 MFMA per dz: lane group grp takes dy = grp - 1 (the fourth group is
// zero), its four K slots dx = -1, 0, 1 (the fourth is zero): one LDS
// instruction per operand, where 27 taps laid along K took eight 2-byte reads
// and their packing.
template <typename TIN, int EPI>
__global__ __launch_bounds__(256) void k_conv_in_tile(const TIN *__restrict__ x, float scale,
                                                      const uint16_t *__restrict__ Wfi,
                                                      const float *__restrict__ bias, const float *__restrict__ aux,
                                                      float *__restrict__ Zout, uint16_t *__restrict__ Aout, Geom g,
                                                      int zc) {
  constexpr int LXW = CTX + 4;  // words per row: x0-1 .. x0+CTX (+ padding)
  // one row more than the tile and its halo, for the reads of the fourth lane group
  __shared__ uint32_t sx[4][CLY + 1][LXW];
  const ConvTile T = conv_tile(g, CTX, CTY, zc);
  const int x0 = T.x0, y0 = T.y0, z0 = T.z0, z1 = T.z1;
  const size_t box = (size_t)g.nx * g.ny * g.nz;
  const TIN *xb = x + (size_t)T.b * box;
  const int lane = threadIdx.x & 63, w = wave_ix(), m = lane & 15, grp = lane >> 4;
  constexpr int NPT = CLY * CLX, NLD = (NPT + 255) / 256;
  TIN reg[NLD];
  size_t off[NLD];
  unsigned in = 0;
  int lds[NLD];
#pragma unroll
  for (int q = 0; q < NLD; q++) {
    const int idx = (int)threadIdx.x + q * 256;
    const int ly = idx / CLX, lx = idx % CLX, gx = x0 - 1 + lx, gy = y0 - 1 + ly;
    const bool ok = idx < NPT && gx >= 0 && gx < g.nx && gy >= 0 && gy < g.ny;
    off[q] = ok ? (size_t)gy * g.nx + gx : 0;
    in |= (unsigned)ok << q;
    lds[q] = idx < NPT ? ly * LXW + lx : -1;
  }
  for (int q = (int)threadIdx.x; q < 4 * (CLY + 1) * LXW; q += 256) (&sx[0][0][0])[q] = 0u;
  __syncthreads();
  const size_t plane = (size_t)g.nx * g.ny;
  auto fetch = [&](int k) {
    const TIN *xk = xb + (k >= 0 && k < g.nz ? (size_t)k * plane : 0);
#pragma unroll
    for (int q = 0; q < NLD; q++) reg[q] = xk[off[q]];
  };
  auto store = [&](int k) {
    uint16_t *S = (uint16_t *)&sx[k & 3][0][0];
    const bool kin = k >= 0 && k < g.nz;
#pragma unroll
    for (int q = 0; q < NLD; q++) {
      if (lds[q] < 0) continue;
      uint16_t v;
      if constexpr (std::is_same<TIN, float>::value) v = (uint16_t)pk_bf16(reg[q] * scale, 0.f);
      else v = reg[q];
      if (!(kin && ((in >> q) & 1))) v = 0;
      S[2 * lds[q]] = v;                              // low half of its own word
      if (lds[q] % LXW > 0) S[2 * lds[q] - 1] = v;    // high half of the west neighbour's
    }
  };
  bf16x4 bw[3];
#pragma unroll
  for (int d = 0; d < 3; d++) bw[d] = *(const bf16x4 *)(Wfi + ((size_t)d * 64 + lane) * 4);
  const floatx4 bm = EPI == 2 ? floatx4{0.f, 0.f, 0.f, 0.f} : *(const floatx4 *)(bias + 4 * grp);
  const uint32_t live = grp < 3 ? ~0u : 0u;
  fetch(z0 - 1);
  store(z0 - 1);
  fetch(z0);
  store(z0);
  fetch(z0 + 1);
  store(z0 + 1);
  fetch(z0 + 2);
  __syncthreads();
  for (int z = z0; z < z1; z++) {
    store(z + 2);
    fetch(z + 3);
#pragma unroll
    for (int q = 0; q < 4; q++) {
      const int r = 2 * w + (q >> 1), sg = q & 1, y = y0 + r, xs = x0 + 16 * sg;
      if (y >= g.ny || xs >= g.nx) continue;  // uniform per wave
      const int npts = min(16, g.nx - xs);
      const size_t row = (size_t)T.b * box + ((size_t)z * g.ny + y) * g.nx + xs;
      const floatx4 ax = conv_aux<EPI>(aux, row, npts);
      floatx4 acc = bm;
#pragma unroll
      for (int d = 0; d < 3; d++) {
        // LDS column lx is the point x0 - 1 + lx: the four points from x-1 on
        const uint32_t *S = &sx[(z + d - 1) & 3][r + grp][16 * sg + m];
        const uint32_t aw[2] = {S[0] & live, S[2] & live & 0xffffu};
        bf16x4 a;
        __builtin_memcpy(&a, aw, 8);
        acc = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(bw[d], a, acc, 0, 0, 0);
      }
      conv_epilogue<EPI>(acc, ax, Zout, Aout, row, npts);
    }
    __syncthreads();
  }
}

// The last layer (16 -> 1): out[q] = sum_tap G[q + off(tap)][tap] with
// G[p][tap] = sum_ci A[p][ci] w3[ci][tap], a product of every point's 16
// channels with the 16 x 27 weights: two K = 16 MFMAs per 16 points instead
// of the 14 of K = 32 that padding the single output channel to 16 takes, and
// the activations go from global memory straight into the operand registers
// (each input point is read once per tile, 8 bytes a lane, contiguous).  G of
// one input plane (OIX x OIY points) lies in LDS tap by tap; every output
// column then adds its 27 values to the three running sums of the output
// planes z-1, z, z+1.  At 257^3: 0.34 -> 0.20 ms.
constexpr int OIX = 32, OIY = 10, OTX = OIX - 2, OTY = OIY - 2;
constexpr int OPTS = OIX * OIY, OSEG = OPTS / 16 / 4;  // segments per wave
constexpr int OSTR = OPTS + 4;                         // LDS words per tap (4 mod 64: 16 taps on 64 banks)
static_assert(OIX * OTY == 256 && OSTR % 64 == 4, "one output column per thread");
static_assert(OPTS % 64 == 0, "whole segments per wave");
__global__ __launch_bounds__(256) void k_conv_out_tile(const uint16_t *__restrict__ X,
                                                       const uint16_t *__restrict__ Wo,
                                                       const float *__restrict__ bias, float *__restrict__ out, Geom g,
                                                       int zc) {
  __shared__ float sG[NTAP * OSTR];
  const ConvTile T = conv_tile(g, OTX, OTY, zc);
  const size_t box = (size_t)g.nx * g.ny * g.nz;
  const uint16_t *Xb = X + (size_t)T.b * box * NC;
  const int lane = threadIdx.x & 63, w = wave_ix(), m = lane & 15, grp = lane >> 4;
  // input segment s of this wave: 16 points of row (w * OSEG + s) / 2
  uint2 regA[OSEG], regB[OSEG];
  size_t off[OSEG];
  unsigned in = 0;
#pragma unroll
  for (int s = 0; s < OSEG; s++) {
    const int seg = w * OSEG + s, gy = T.y0 - 1 + seg / 2, gx = T.x0 - 1 + 16 * (seg & 1) + m;
    const bool ok = gx >= 0 && gx < g.nx && gy >= 0 && gy < g.ny;
    off[s] = ok ? ((size_t)gy * g.nx + gx) * NC + 4 * grp : 0;
    in |= (unsigned)ok << s;
  }
  const size_t plane = (size_t)g.nx * g.ny * NC;
  auto fetch = [&](int k, uint2 (&reg)[OSEG]) {
    const uint16_t *Xk = Xb + (k >= 0 && k < g.nz ? (size_t)k * plane : 0);
#pragma unroll
    for (int s = 0; s < OSEG; s++) reg[s] = *(const uint2 *)(Xk + off[s]);
  };
  const bf16x4 w0 = *(const bf16x4 *)(Wo + (size_t)lane * 4), w1 = *(const bf16x4 *)(Wo + (size_t)(64 + lane) * 4);
  // output columns of this thread
  // (a row of 32 lanes has 30 columns: neighbouring lanes read neighbouring words)
  const int ox = (int)threadIdx.x % OIX, oy = (int)threadIdx.x / OIX;
  const bool mine = ox < OTX && T.x0 + ox < g.nx && T.y0 + oy < g.ny;
  const float *G = &sG[(oy + 1) * OIX + (ox < OTX ? ox : 0) + 1];
  float *o = out + (size_t)T.b * box + (mine ? (size_t)(T.y0 + oy) * g.nx + T.x0 + ox : 0);
  const size_t oplane = (size_t)g.nx * g.ny;
  float sum[3] = {0.f, 0.f, 0.f};
  const float b0 = bias[0];
  // two planes in flight: a step is shorter than a load's way from memory
  auto step = [&](int k, uint2 (&reg)[OSEG]) {
    const bool kin = k >= 0 && k < g.nz;
    bf16x4 a[OSEG];
#pragma unroll
    for (int s = 0; s < OSEG; s++) {
      const uint2 v = kin && ((in >> s) & 1) ? reg[s] : make_uint2(0u, 0u);
      __builtin_memcpy(&a[s], &v, 8);
    }
    if (k + 1 < T.z1) fetch(k + 2, reg);
    __syncthreads();  // the sums of the plane before have read sG
#pragma unroll
    for (int s = 0; s < OSEG; s++) {
      const floatx4 zero = {0.f, 0.f, 0.f, 0.f};
      const floatx4 g0 = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a[s], w0, zero, 0, 0, 0);
      const floatx4 g1 = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a[s], w1, zero, 0, 0, 0);
      // lane (m, grp): points 4grp .. 4grp+3 of taps m and 16 + m
      float *S = &sG[m * OSTR + (w * OSEG + s) * 16 + 4 * grp];
      *(floatx4 *)S = g0;
      if (16 + m < NTAP) *(floatx4 *)(S + 16 * OSTR) = g1;
    }
    __syncthreads();
    // input plane k is at dz = +1 of output plane k-1, 0 of k, -1 of k+1
#pragma unroll
    for (int dz = -1; dz <= 1; dz++) {
      float v = sum[1 - dz];
#pragma unroll
      for (int dy = -1; dy <= 1; dy++)
#pragma unroll
        for (int dx = -1; dx <= 1; dx++) v += G[((dz + 1) * 9 + (dy + 1) * 3 + dx + 1) * OSTR + dy * OIX + dx];
      sum[1 - dz] = v;
    }
    if (mine && k - 1 >= T.z0) o[(size_t)(k - 1) * oplane] = sum[0] + b0;  // plane k-1 is complete
    sum[0] = sum[1];
    sum[1] = sum[2];
    sum[2] = 0.f;
  };
  fetch(T.z0 - 1, regA);
  fetch(T.z0, regB);
  for (int k = T.z0 - 1; k <= T.z1; k += 2) {
    step(k, regA);
    if (k + 1 <= T.z1) step(k + 1, regB);
  }
}

// ---------------------------------------------------------------------------
// Weight gradients: dW[tap][ci][co] = sum_p X[p+off(tap)][ci] * dZ[p][co], and
// the bias gradient sum_p dZ[p][co] as row 27.  A GEMM per tap with the points
// along K.  A block owns a WTX x WTY tile of (x, y) columns and marches zc
// planes, one 32-point row of dZ per wave and step against the 9 rows of X
// around it, all 27 taps accumulated in registers -- so every point of X and
// dZ is read from memory once per tile, where one workgroup per tap read
// both 28 times, 2 bytes at a time (0.70 -> 0.035 ms for 16 crops of 32^3).
// The operands want 8 consecutive points of one channel per lane, the arrays
// are channel-last: the planes are transposed on their way into LDS
// ([row][channel][x], two points per word).  The taps dx = -1 and +1 of a row
// come from the aligned 8 points and their outer neighbours by five funnel
// shifts.  Row strides of 28 and 20 words spread the 16 channels over the
// banks.  The waves' sums are added in wave order, one partial per block.
//   XCH: 16 -- X is BF16 [P][16]; 1 -- X is FP32 [P] (the network's input,
//   rounded to BF16): the taps themselves are the rows of A (27 of 32, row 27
//   all ones for the bias), one LDS row per point row and dx.
//   ZCH: 16 -- dZ is BF16 [P][16]; 1 -- BF16 [P], the single output channel.
// ---------------------------------------------------------------------------
constexpr int WTX = 32, WTY = 8, WLY = WTY + 2;
constexpr int WGT = 512;  // threads: a wave per tile row, two waves a SIMD (the accumulators' registers)
constexpr int WXS = 56, WZS = 40;  // 2-byte elements per (row, channel) of the X and dZ planes

// the ci * 16 + co of entry e of a row of a block's partial (lane order: lane
// l = 16 grp + m holds ci = 4grp + i, co = m as entries 4 l + i)
__device__ __forceinline__ int wgrad_entry(int e) { return (4 * (e >> 6) + (e & 3)) * 16 + ((e >> 2) & 15); }

// words of channels c .. c+7 of two neighbouring points, one word per channel
__device__ __forceinline__ void put_pair(uint16_t *S, int stride, const uint4 &p, const uint4 &q) {
  const unsigned pw[4] = {p.x, p.y, p.z, p.w}, qw[4] = {q.x, q.y, q.z, q.w};
#pragma unroll
  for (int c = 0; c < 4; c++) {
    *(unsigned *)(S + (2 * c) * stride) = __builtin_amdgcn_perm(qw[c], pw[c], 0x05040100u);
    *(unsigned *)(S + (2 * c + 1) * stride) = __builtin_amdgcn_perm(qw[c], pw[c], 0x07060302u);
  }
}

template <int ZCH>
__global__ __launch_bounds__(WGT) void k_wgrad_tile(const uint16_t *__restrict__ X, const uint16_t *__restrict__ dZ,
                                                    float *__restrict__ partial, Geom g, int zc) {
  // X planes k-1, k, k+1 and the plane being filled share 4 slots
  extern __shared__ __align__(16) unsigned char wsm[];
  uint16_t *sX = (uint16_t *)wsm;                          // [4][WLY][16][WXS]
  uint16_t *sZ = sX + 4 * WLY * NC * WXS;                  // [2][WTY][16][WZS]
  const ConvTile T = conv_tile(g, WTX, WTY, zc);
  const size_t box = (size_t)g.nx * g.ny * g.nz;
  const uint16_t *Xb = X + (size_t)T.b * box * NC;
  const uint16_t *Zb = dZ + (size_t)T.b * box * ZCH;
  const int lane = threadIdx.x & 63, w = wave_ix(), m = lane & 15, grp = lane >> 4;
  const uint4 zero4 = make_uint4(0u, 0u, 0u, 0u);
  // staging tasks: a pair of points (x even relative to the tile) of one row, 8 channels
  constexpr int XPAIR = WTX / 2 + 2;
  static_assert(WLY * XPAIR * 2 <= WGT && WTX * WTY == 256, "one task per thread");
  struct Pair {
    uint4 p, q;
  };
  auto fetch_x = [&](int k) {
    const int idx = (int)threadIdx.x, h = idx & 1, pr = (idx >> 1) % XPAIR, row = (idx >> 1) / XPAIR;
    const int gy = T.y0 - 1 + row, gx = T.x0 - 2 + 2 * pr;
    const bool ok = k >= 0 && k < g.nz && row < WLY && gy >= 0 && gy < g.ny;
    const size_t at = ok ? (((size_t)k * g.ny + gy) * g.nx) * NC + 8 * h : 0;
    return Pair{ok && gx >= 0 && gx < g.nx ? *(const uint4 *)(Xb + at + (size_t)gx * NC) : zero4,
                ok && gx + 1 >= 0 && gx + 1 < g.nx ? *(const uint4 *)(Xb + at + (size_t)(gx + 1) * NC) : zero4};
  };
  auto store_x = [&](int k, const Pair &v) {
    uint16_t *S = sX + (size_t)(k & 3) * WLY * NC * WXS;
    const int idx = (int)threadIdx.x, h = idx & 1, pr = (idx >> 1) % XPAIR, row = (idx >> 1) / XPAIR;
    if (row < WLY) put_pair(S + ((size_t)row * NC + 8 * h) * WXS + 6 + 2 * pr, WXS, v.p, v.q);
  };
  // dZ: the last 256 threads (those with the fewest X tasks)
  const int zt = (int)threadIdx.x - (WGT - 256);
  auto fetch_z = [&](int k) {
    Pair v{zero4, zero4};
    if (zt < 0) return v;
    if constexpr (ZCH == 16) {
      const int h = zt & 1, pr = (zt >> 1) % (WTX / 2), row = (zt >> 1) / (WTX / 2);
      const int gy = T.y0 + row, gx = T.x0 + 2 * pr;
      const bool ok = k < T.z1 && gy < g.ny;
      const size_t at = ok ? (((size_t)k * g.ny + gy) * g.nx) * NC + 8 * h : 0;
      if (ok && gx < g.nx) v.p = *(const uint4 *)(Zb + at + (size_t)gx * NC);
      if (ok && gx + 1 < g.nx) v.q = *(const uint4 *)(Zb + at + (size_t)(gx + 1) * NC);
    } else {
      const int gy = T.y0 + zt / WTX, gx = T.x0 + zt % WTX;
      if (k < T.z1 && gy < g.ny && gx < g.nx) v.p.x = Zb[((size_t)k * g.ny + gy) * g.nx + gx];
    }
    return v;
  };
  auto store_z = [&](int k, const Pair &v) {
    if (zt < 0) return;
    uint16_t *S = sZ + (size_t)(k & 1) * WTY * NC * WZS;
    if constexpr (ZCH == 16) {
      const int h = zt & 1, pr = (zt >> 1) % (WTX / 2), row = (zt >> 1) / (WTX / 2);
      put_pair(S + ((size_t)row * NC + 8 * h) * WZS + 2 * pr, WZS, v.p, v.q);
    } else {
      S[(size_t)(zt / WTX) * NC * WZS + zt % WTX] = (uint16_t)v.p.x;
    }
  };
  floatx4 acc[NTAP + 1];
#pragma unroll
  for (int t = 0; t <= NTAP; t++) acc[t] = floatx4{0.f, 0.f, 0.f, 0.f};
  bf16x8 ones = {};
  if (m == 0)
    for (int j = 0; j < 8; j++) ones[j] = (__bf16)1.0f;
  auto u4 = [](unsigned a, unsigned b, unsigned c, unsigned d) {
    const unsigned v[4] = {a, b, c, d};
    bf16x8 r;
    __builtin_memcpy(&r, v, 16);
    return r;
  };
  {
    const Pair xa = fetch_x(T.z0 - 1), xb_ = fetch_x(T.z0), xc = fetch_x(T.z0 + 1), za = fetch_z(T.z0);
    store_x(T.z0 - 1, xa);
    store_x(T.z0, xb_);
    store_x(T.z0 + 1, xc);
    store_z(T.z0, za);
  }
  __syncthreads();
  for (int k = T.z0; k < T.z1; k++) {
    // the next planes' loads are in flight through this step's products and go
    // into slots that no wave reads in it (requesting them two steps ahead
    // measured 10 % slower)
    const Pair xn = fetch_x(k + 2), zn = fetch_z(k + 1);
    {
      const int row = w;
      bf16x8 bz = *(const bf16x8 *)(sZ + ((size_t)((k & 1) * WTY + row) * NC + (ZCH == 16 ? m : 0)) * WZS + 8 * grp);
      if (ZCH == 1 && m != 0) bz = bf16x8{};
      acc[NTAP] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ones, bz, acc[NTAP], 0, 0, 0);
#pragma unroll
      for (int dzy = 0; dzy < 9; dzy++) {
        const int slot = (k + dzy / 3 - 1) & 3, xr = row + dzy % 3;
        const uint16_t *S = sX + ((size_t)(slot * WLY + xr) * NC + m) * WXS + 8 + 8 * grp;
        const uint4 v = *(const uint4 *)S;
        const unsigned wl = *(const unsigned *)(S - 2), wr = *(const unsigned *)(S + 8);
        const unsigned a0 = __builtin_amdgcn_alignbit(v.x, wl, 16), a1 = __builtin_amdgcn_alignbit(v.y, v.x, 16),
                       a2 = __builtin_amdgcn_alignbit(v.z, v.y, 16), a3 = __builtin_amdgcn_alignbit(v.w, v.z, 16),
                       a4 = __builtin_amdgcn_alignbit(wr, v.w, 16);
        acc[3 * dzy] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(u4(a0, a1, a2, a3), bz, acc[3 * dzy], 0, 0, 0);
        acc[3 * dzy + 1] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(u4(v.x, v.y, v.z, v.w), bz, acc[3 * dzy + 1], 0, 0, 0);
        acc[3 * dzy + 2] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(u4(a1, a2, a3, a4), bz, acc[3 * dzy + 2], 0, 0, 0);
      }
    }
    store_x(k + 2, xn);
    store_z(k + 1, zn);
    __syncthreads();
  }
  // lane holds D[ci = 4grp + i][co = m]: entry 4 lane + i of a tap's 256.  The
  // waves' sums meet in LDS a quarter of the rows at a time and are added in
  // wave order, wave w taking row t0 + w.
  constexpr int NW = WGT / kWave, QT = (NTAP + 1) / 4;
  floatx4 *red = (floatx4 *)wsm;
  float *out = partial + (size_t)blockIdx.x * LAYER_FLOATS;
#pragma unroll
  for (int h = 0; h < 4; h++) {
#pragma unroll
    for (int t = 0; t < QT; t++) red[(t * NW + w) * kWave + lane] = acc[h * QT + t];
    __syncthreads();
    if (w < QT) {
      floatx4 v = red[w * NW * kWave + lane];
      for (int ww = 1; ww < NW; ww++) v += red[(w * NW + ww) * kWave + lane];
      *(floatx4 *)(out + (h * QT + w) * 256 + 4 * lane) = v;
    }
    __syncthreads();
  }
}
constexpr size_t kWgradLds = (4 * (size_t)WLY * NC * WXS + 2 * (size_t)WTY * NC * WZS) * sizeof(uint16_t);
static_assert(kWgradLds >= (NTAP + 1) / 4 * (WGT / kWave) * kWave * 16, "the wave sums reuse the planes' LDS");
static_assert((NTAP + 1) % 4 == 0 && WGT / kWave == WTY, "one tile row per wave");

// layer 1: the taps are the rows of A (two MFMAs per 32 points)
__global__ __launch_bounds__(256) void k_wgrad_in_tile(const float *__restrict__ x, const uint16_t *__restrict__ dZ,
                                                       float *__restrict__ partial, Geom g, int zc) {
  constexpr int XS = 40;  // elements per row; copy d holds the points shifted by d - 1
  __shared__ __align__(16) uint16_t sX[4][3][WLY][XS];
  __shared__ __align__(16) uint16_t sZ[2][WTY][NC][WZS];
  __shared__ float red[2 * 256];
  const ConvTile T = conv_tile(g, WTX, WTY, zc);
  const size_t box = (size_t)g.nx * g.ny * g.nz;
  const float *xb = x + (size_t)T.b * box;
  const uint16_t *Zb = dZ + (size_t)T.b * box * NC;
  const int lane = threadIdx.x & 63, w = wave_ix(), m = lane & 15, grp = lane >> 4;
  const uint4 zero4 = make_uint4(0u, 0u, 0u, 0u);
  constexpr int LXP = WTX + 2, NXT = (WLY * LXP + 255) / 256;
  struct Vals {
    float v[NXT];
  };
  auto fetch_x = [&](int k) {
    Vals r;
#pragma unroll
    for (int t = 0; t < NXT; t++) {
      const int idx = (int)threadIdx.x + t * 256, row = idx / LXP, gy = T.y0 - 1 + row, gx = T.x0 - 1 + idx % LXP;
      r.v[t] = k >= 0 && k < g.nz && row < WLY && gy >= 0 && gy < g.ny && gx >= 0 && gx < g.nx
                   ? xb[((size_t)k * g.ny + gy) * g.nx + gx] : 0.f;
    }
    return r;
  };
  auto store_x = [&](int k, const Vals &r) {
#pragma unroll
    for (int t = 0; t < NXT; t++) {
      const int idx = (int)threadIdx.x + t * 256, row = idx / LXP, lx = idx % LXP;
      if (row >= WLY) continue;
      const uint16_t h = (uint16_t)pk_bf16(r.v[t], 0.f);
      // the point x0 - 1 + lx is element p + (d - 1) of copy d at p = lx - d
#pragma unroll
      for (int d = 0; d < 3; d++)
        if (lx - d >= 0 && lx - d < WTX) sX[k & 3][d][row][lx - d] = h;
    }
  };
  struct Pair {
    uint4 p, q;
  };
  const int zh = threadIdx.x & 1, zpr = (threadIdx.x >> 1) % (WTX / 2), zrow = (threadIdx.x >> 1) / (WTX / 2);
  auto fetch_z = [&](int k) {
    const int gy = T.y0 + zrow, gx = T.x0 + 2 * zpr;
    const bool ok = k < T.z1 && gy < g.ny;
    const size_t at = ok ? (((size_t)k * g.ny + gy) * g.nx) * NC + 8 * zh : 0;
    return Pair{ok && gx < g.nx ? *(const uint4 *)(Zb + at + (size_t)gx * NC) : zero4,
                ok && gx + 1 < g.nx ? *(const uint4 *)(Zb + at + (size_t)(gx + 1) * NC) : zero4};
  };
  auto store_z = [&](int k, const Pair &v) { put_pair(&sZ[k & 1][zrow][8 * zh][2 * zpr], WZS, v.p, v.q); };
  floatx4 acc[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
  bf16x8 ones;
  for (int j = 0; j < 8; j++) ones[j] = (__bf16)1.0f;
  {
    const Vals xa = fetch_x(T.z0 - 1), xb_ = fetch_x(T.z0), xc = fetch_x(T.z0 + 1);
    const Pair za = fetch_z(T.z0);
    store_x(T.z0 - 1, xa);
    store_x(T.z0, xb_);
    store_x(T.z0 + 1, xc);
    store_z(T.z0, za);
  }
  __syncthreads();
  for (int k = T.z0; k < T.z1; k++) {
    const Vals xn = fetch_x(k + 2);
    const Pair zn = fetch_z(k + 1);
#pragma unroll
    for (int rr = 0; rr < WTY / 4; rr++) {
      const int row = w * (WTY / 4) + rr;
      const bf16x8 bz = *(const bf16x8 *)&sZ[k & 1][row][m][8 * grp];
#pragma unroll
      for (int h = 0; h < 2; h++) {
        const int tap = 16 * h + m, tp = tap < NTAP ? tap : 0;
        bf16x8 a = *(const bf16x8 *)&sX[(k + tp / 9 - 1) & 3][tp % 3][row + (tp / 3) % 3][8 * grp];
        if (tap >= NTAP) a = tap == NTAP ? ones : bf16x8{};
        acc[h] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, bz, acc[h], 0, 0, 0);
      }
    }
    store_x(k + 2, xn);
    store_z(k + 1, zn);
    __syncthreads();
  }
  for (int ww = 0; ww < 4; ww++) {
    if (w == ww)
#pragma unroll
      for (int h = 0; h < 2; h++)
#pragma unroll
        for (int i = 0; i < 4; i++) {
          float *r = red + (16 * h + 4 * grp + i) * 16 + m;
          *r = ww == 0 ? acc[h][i] : *r + acc[h][i];
        }
    __syncthreads();
  }
  // only input channel 0 (row 0 of every tap, and the bias row) has gradients
  float *out = partial + (size_t)blockIdx.x * LAYER_FLOATS;
  for (int e = threadIdx.x; e < LAYER_FLOATS; e += 256) {
    const int q = wgrad_entry(e % 256);
    out[e] = q < 16 ? red[(e / 256) * 16 + q] : 0.f;
  }
}

// fold of the blocks' partials -> grad[28][256]: a block takes 64 entries, its
// 16 waves every 16th partial (64 neighbouring words a load), then the waves'
// sums in order (deterministic for a fixed launch shape)
__global__ __launch_bounds__(1024) void k_fold_wgrad(const float *__restrict__ partial, float *__restrict__ grad,
                                                     int nblk) {
  __shared__ float red[16][64];
  const int e = blockIdx.x * 64 + (threadIdx.x & 63), w = threadIdx.x >> 6;
  float s = 0.f;
  for (int c = w; c < nblk; c += 16) s += partial[(size_t)c * LAYER_FLOATS + e];
  red[w][threadIdx.x & 63] = s;
  __syncthreads();
  if (w == 0) {
    for (int c = 1; c < 16; c++) s += red[c][threadIdx.x];
    grad[e / 256 * 256 + wgrad_entry(e % 256)] = s;
  }
}

// loss = 0.5 * mean over counted points of (Y[p] - T[p])^2; dY[p] =
// (Y - T)/count (bf16).  Points within `margin` of a box
// face are not counted.  Per-block partial sums of the squared error.
__global__ __launch_bounds__(256) void k_loss(const float *__restrict__ Y, const float *__restrict__ T,
                                              const float *__restrict__ W, const double *__restrict__ wcount,
                                              uint16_t *__restrict__ dY, double *__restrict__ part,
                                              Geom g, int margin, double inv_count) {
  // W (optional): per-point weights 0/1 on top of the margin rule; the
  // mean then runs over the weighted points, whose count *wcount holds
  __shared__ double red[256];
  const size_t box = (size_t)g.nx * g.ny * g.nz;
  const size_t p = (size_t)blockIdx.x * 256 + threadIdx.x;
  if (wcount) inv_count = *wcount > 0 ? 1.0 / *wcount : 0.0;
  double e2 = 0.0;
  if (p < box * g.nb) {
    const size_t q = p % box;
    const int x = (int)(q % g.nx), y = (int)((q / g.nx) % g.ny), z = (int)(q / ((size_t)g.nx * g.ny));
    bool on = x >= margin && x < g.nx - margin && y >= margin && y < g.ny - margin &&
              z >= margin && z < g.nz - margin;
    if (W) on = on && W[p] != 0.f;
    float d = 0.f;
    if (on) {
      d = Y[p] - T[p];
      e2 = (double)d * (double)d;
    }
    dY[p] = f2bf((float)(d * inv_count));
  }
  red[threadIdx.x] = e2;
  __syncthreads();
  for (int s = 128; s > 0; s >>= 1) {
    if (threadIdx.x < s) red[threadIdx.x] += red[threadIdx.x + s];
    __syncthreads();
  }
  if (threadIdx.x == 0) part[blockIdx.x] = red[0];
}

// partial counts of the weighted points (margin rule and W != 0), one per block
__global__ __launch_bounds__(256) void k_wcount(const float *__restrict__ W, Geom g, int margin,
                                                double *__restrict__ part) {
  __shared__ double red[256];
  const size_t box = (size_t)g.nx * g.ny * g.nz;
  const size_t p = (size_t)blockIdx.x * 256 + threadIdx.x;
  double v = 0.0;
  if (p < box * g.nb) {
    const size_t q = p % box;
    const int x = (int)(q % g.nx), y = (int)((q / g.nx) % g.ny), z = (int)(q / ((size_t)g.nx * g.ny));
    if (x >= margin && x < g.nx - margin && y >= margin && y < g.ny - margin && z >= margin &&
        z < g.nz - margin && W[p] != 0.f)
      v = 1.0;
  }
  red[threadIdx.x] = v;
  __syncthreads();
  for (int s = 128; s > 0; s >>= 1) {
    if (threadIdx.x < s) red[threadIdx.x] += red[threadIdx.x + s];
    __syncthreads();
  }
  if (threadIdx.x == 0) part[blockIdx.x] = red[0];
}

__global__ __launch_bounds__(256) void k_fold_d(const double *__restrict__ part, int n, double *out) {
  __shared__ double red[256];
  double s = 0.0;
  for (int i = threadIdx.x; i < n; i += 256) s += part[i];
  red[threadIdx.x] = s;
  __syncthreads();
  for (int k = 128; k > 0; k >>= 1) {
    if (threadIdx.x < k) red[threadIdx.x] += red[threadIdx.x + k];
    __syncthreads();
  }
  if (threadIdx.x == 0) out[0] = red[0];
}

// Adam on FP32 master weights (only the entries `mask` marks trainable)
__global__ __launch_bounds__(256) void k_adam(float *__restrict__ w, float *__restrict__ m1,
                                              float *__restrict__ m2, const float *__restrict__ gr,
                                              const uint8_t *__restrict__ mask, int n, float lr,
                                              float b1, float b2, float c1, float c2, float eps) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i >= n || !mask[i]) return;
  const float g = gr[i];
  const float a = b1 * m1[i] + (1.f - b1) * g;
  const float b = b2 * m2[i] + (1.f - b2) * g * g;
  m1[i] = a;
  m2[i] = b;
  w[i] -= lr * (a / c1) / (sqrtf(b / c2) + eps);
}

// MFMA weight fragments of all three layers, packed by one launch
// (lane l: m = l%16, grp = l/16):
//   wfi   layer 1, one input channel (K = 16 per dz): [dz][lane][j] =
//         W1[tap (dx = j-1, dy = grp-1, dz)][ci 0][co m], 0 for j = 3 or grp = 3
//   wbi   backward data of layer 3, the same with flipped taps and the single
//         output channel as input: W3[26 - tap][ci m][co 0]
//   wp2   layer 2, tap pairs (K = 32): [pr][lane][j] =
//         W2[2 pr + grp/2][ci 8(grp%2) + j][co m], 0 past tap 26
//   wpb2  its backward data: W2[26 - tap][ci m][co 8(grp%2) + j]
//   wo3   layer 3 with the taps as columns (K = 16 channels): [h][lane][j] =
//         W3[tap 16 h + m][ci 4 grp + j][co 0], 0 past tap 26
constexpr int FR_IN = 3 * 64 * 4, FR_PAIR = NPAIR * 64 * 8, FR_OUT = 2 * 64 * 4;
constexpr int FR_WFI = 0, FR_WBI = FR_WFI + FR_IN, FR_WP2 = FR_WBI + FR_IN, FR_WPB2 = FR_WP2 + FR_PAIR,
              FR_WO3 = FR_WPB2 + FR_PAIR, FR_TOTAL = FR_WO3 + FR_OUT;
__global__ __launch_bounds__(256) void k_pack_frags(const float *__restrict__ W, uint16_t *__restrict__ F) {
  const int idx = blockIdx.x * 256 + threadIdx.x;
  if (idx >= FR_TOTAL) return;
  const float *W1 = W, *W2 = W + LAYER_FLOATS, *W3 = W + 2 * LAYER_FLOATS;
  float v = 0.f;
  if (idx < FR_WP2) {
    const int q = idx % FR_IN, d = q / 256, lane = (q / 4) % 64, j = q % 4, m = lane & 15, grp = lane >> 4;
    const int tap = d * 9 + grp * 3 + j;
    if (j < 3 && grp < 3) v = idx < FR_WBI ? W1[tap * 256 + m] : W3[(26 - tap) * 256 + m * 16];
  } else if (idx < FR_WO3) {
    const int q = (idx - FR_WP2) % FR_PAIR, pr = q / 512, lane = (q / 8) % 64, j = q % 8, m = lane & 15, grp = lane >> 4;
    const int tap = 2 * pr + (grp >> 1), k = 8 * (grp & 1) + j;
    if (tap < NTAP) v = idx < FR_WPB2 ? W2[tap * 256 + k * 16 + m] : W2[(26 - tap) * 256 + m * 16 + k];
  } else {
    const int q = idx - FR_WO3, h = q / 256, lane = (q / 4) % 64, j = q % 4, m = lane & 15, grp = lane >> 4;
    const int tap = 16 * h + m;
    if (tap < NTAP) v = W3[tap * 256 + (4 * grp + j) * 16];
  }
  F[idx] = f2bf(v);
}

// u += coef * Z[p * STRIDE] at interior points of the grid (box = the grid)
template <typename TU, int STRIDE>
__global__ __launch_bounds__(256) void k_apply_correction(TU *__restrict__ u, const float *__restrict__ Z,
                                                          int nx, int ny, int nz, double coef) {
  const int i = blockIdx.x * 64 + (int)(threadIdx.x % 64);
  const int j = blockIdx.y * 4 + (int)(threadIdx.x / 64);
  const int k = blockIdx.z;
  if (i < 1 || j < 1 || k < 1 || i >= nx - 1 || j >= ny - 1 || k >= nz - 1) return;
  const size_t p = ix3(i, j, k, nx, ny);
  u[p] = u[p] + (TU)(coef * (double)Z[p * STRIDE]);
}

}  // namespace

// ===========================================================================
// network object
// ===========================================================================
struct pmg_net {
  int hidden = 16;
  float *w = nullptr;       // 3 layers * LAYER_FLOATS master weights (device)
  float *m1 = nullptr, *m2 = nullptr, *grad = nullptr;
  uint8_t *mask = nullptr;  // trainable entries
  uint16_t *fr = nullptr;   // weight fragments (k_pack_frags)
  int adam_t = 0;
  // training buffers (grown on demand): activations and their gradients (BF16
  // [P][16]), pre-activations (FP32 [P][16]), output (FP32 [P]) and its
  // gradient (BF16 [P])
  size_t cap = 0;
  uint16_t *a1 = nullptr, *a2 = nullptr, *d16 = nullptr, *d16b = nullptr, *dy = nullptr;
  float *z1 = nullptr, *z2 = nullptr, *yt = nullptr;
  // inference buffers (their own capacity: inference allocates no training buffers)
  size_t icap = 0;
  uint16_t *ia1 = nullptr, *ia2 = nullptr;  // bf16 [P][16]
  float *y = nullptr;                       // output, one FP32 per point
  float *partial = nullptr;
  size_t partial_cap = 0;
  double *lpart = nullptr, *lsum = nullptr;
  size_t lpart_cap = 0;
  hipStream_t stream = nullptr;
  bool frags_valid = false;
};

namespace {

int net_ensure(pmg_net *N, size_t P) {
  if (P <= N->cap) return 0;
  PMG_HOST_CHECK(hipStreamSynchronize(N->stream));
  N->cap = 0;
  for (void **p : {(void **)&N->a1, (void **)&N->a2, (void **)&N->d16, (void **)&N->d16b, (void **)&N->dy,
                   (void **)&N->z1, (void **)&N->z2, (void **)&N->yt}) {
    if (*p) PMG_HOST_CHECK(hipFree(*p));
    *p = nullptr;
  }
  const size_t b16 = P * NC * sizeof(uint16_t), b32 = P * NC * sizeof(float);
  PMG_HOST_CHECK(hipMalloc(&N->a1, b16));
  PMG_HOST_CHECK(hipMalloc(&N->a2, b16));
  PMG_HOST_CHECK(hipMalloc(&N->d16, b16));
  PMG_HOST_CHECK(hipMalloc(&N->d16b, b16));
  PMG_HOST_CHECK(hipMalloc(&N->dy, P * sizeof(uint16_t)));
  PMG_HOST_CHECK(hipMalloc(&N->z1, b32));
  PMG_HOST_CHECK(hipMalloc(&N->z2, b32));
  PMG_HOST_CHECK(hipMalloc(&N->yt, P * sizeof(float)));
  N->cap = P;
  return 0;
}

int net_ensure_infer(pmg_net *N, size_t P) {
  if (P <= N->icap) return 0;
  PMG_HOST_CHECK(hipStreamSynchronize(N->stream));
  for (void *p : {(void *)N->ia1, (void *)N->ia2, (void *)N->y})
    if (p) PMG_HOST_CHECK(hipFree(p));
  PMG_HOST_CHECK(hipMalloc(&N->ia1, P * NC * sizeof(uint16_t)));
  PMG_HOST_CHECK(hipMalloc(&N->ia2, P * NC * sizeof(uint16_t)));
  PMG_HOST_CHECK(hipMalloc(&N->y, P * sizeof(float)));
  N->icap = P;
  return 0;
}

int net_frags(pmg_net *N) {
  if (N->frags_valid) return 0;
  hipLaunchKernelGGL(k_pack_frags, dim3((FR_TOTAL + 255) / 256), dim3(256), 0, N->stream, N->w, N->fr);
  PMG_HOST_CHECK(hipGetLastError());
  N->frags_valid = true;
  return 0;
}

const float *net_bias(const pmg_net *N, int layer) { return N->w + (size_t)layer * LAYER_FLOATS + NTAP * 256; }

// z planes one block of a tiled kernel marches: long marches re-read fewer
// halo planes, short ones give a small batch enough workgroups -- the longest
// of 16, 8, 4 that still makes `want` of them
int conv_zc(const Geom &g, int tx, int ty, unsigned want) {
  int zc = 16;
  while (zc > 4 && conv_blocks(g, tx, ty, zc) < want) zc /= 2;
  return zc;
}
constexpr unsigned kConvBlocks = 768;  // three workgroups a CU, what the hidden layer's LDS allows
constexpr unsigned kWgradBlocks = 256;  // one workgroup a CU (their planes take 92 KB of LDS)

// inference: N(scale * x) into y (one FP32 per point).  Layer 1 reads x
// directly, the hidden layer keeps only the BF16 activations, the last layer
// writes its one channel -- no pre-activations are stored
int net_infer(pmg_net *N, const float *x, float scale, float *y, const Geom &g) {
  int rc;
  if ((rc = net_frags(N))) return rc;
  const int zc = conv_zc(g, CTX, CTY, kConvBlocks), zo = conv_zc(g, OTX, OTY, kConvBlocks);
  const dim3 gt(conv_blocks(g, CTX, CTY, zc)), blk(256);
  hipLaunchKernelGGL((k_conv_in_tile<float, 3>), gt, blk, 0, N->stream, x, scale, N->fr + FR_WFI, net_bias(N, 0),
                     (const float *)nullptr, (float *)nullptr, N->ia1, g, zc);
  hipLaunchKernelGGL(k_conv16_tile<3>, gt, blk, 0, N->stream, N->ia1, N->fr + FR_WP2, net_bias(N, 1),
                     (const float *)nullptr, (float *)nullptr, N->ia2, g, zc);
  hipLaunchKernelGGL(k_conv_out_tile, dim3(conv_blocks(g, OTX, OTY, zo)), blk, 0, N->stream, N->ia2, N->fr + FR_WO3,
                     net_bias(N, 2), y, g, zo);
  PMG_HOST_CHECK(hipGetLastError());
  return 0;
}

// training forward of the 3 layers on x into y, keeping pre-activations and
// activations
int net_forward(pmg_net *N, const float *x, float *y, const Geom &g) {
  int rc;
  if ((rc = net_frags(N))) return rc;
  const int zc = conv_zc(g, CTX, CTY, kConvBlocks), zo = conv_zc(g, OTX, OTY, kConvBlocks);
  const dim3 gt(conv_blocks(g, CTX, CTY, zc)), blk(256);
  hipLaunchKernelGGL((k_conv_in_tile<float, 0>), gt, blk, 0, N->stream, x, 1.0f, N->fr + FR_WFI, net_bias(N, 0),
                     (const float *)nullptr, N->z1, N->a1, g, zc);
  hipLaunchKernelGGL(k_conv16_tile<0>, gt, blk, 0, N->stream, N->a1, N->fr + FR_WP2, net_bias(N, 1),
                     (const float *)nullptr, N->z2, N->a2, g, zc);
  hipLaunchKernelGGL(k_conv_out_tile, dim3(conv_blocks(g, OTX, OTY, zo)), blk, 0, N->stream, N->a2, N->fr + FR_WO3,
                     net_bias(N, 2), y, g, zo);
  PMG_HOST_CHECK(hipGetLastError());
  return 0;
}

// weight gradients of layer l (0, 1, 2) into N->grad
int net_wgrad(pmg_net *N, const Geom &g, int l, const float *x) {
  const int zc = conv_zc(g, WTX, WTY, kWgradBlocks);
  const unsigned nblk = conv_blocks(g, WTX, WTY, zc);
  const size_t need = (size_t)nblk * LAYER_FLOATS;
  if (need > N->partial_cap) {
    PMG_HOST_CHECK(hipStreamSynchronize(N->stream));
    N->partial_cap = 0;
    if (N->partial) PMG_HOST_CHECK(hipFree(N->partial));
    N->partial = nullptr;
    PMG_HOST_CHECK(hipMalloc(&N->partial, need * sizeof(float)));
    N->partial_cap = need;
  }
  if (l == 0) {
    hipLaunchKernelGGL(k_wgrad_in_tile, dim3(nblk), dim3(256), 0, N->stream, x, N->d16, N->partial, g, zc);
  } else if (l == 1) {
    hipLaunchKernelGGL(k_wgrad_tile<16>, dim3(nblk), dim3(WGT), kWgradLds, N->stream, N->a1, N->d16b, N->partial, g,
                       zc);
  } else {
    hipLaunchKernelGGL(k_wgrad_tile<1>, dim3(nblk), dim3(WGT), kWgradLds, N->stream, N->a2, N->dy, N->partial, g, zc);
  }
  PMG_HOST_CHECK(hipGetLastError());
  hipLaunchKernelGGL(k_fold_wgrad, dim3(LAYER_FLOATS / 64), dim3(1024), 0, N->stream, N->partial,
                     N->grad + (size_t)l * LAYER_FLOATS, (int)nblk);
  PMG_HOST_CHECK(hipGetLastError());
  return 0;
}

// forward + loss + backward; gradients into N->grad (3 * LAYER_FLOATS)
int net_loss_backward(pmg_net *N, const Geom &g, const float *x, const float *T, const float *W, int margin,
                      double *loss_out) {
  int rc;
  if ((rc = net_forward(N, x, N->yt, g))) return rc;
  const size_t total = (size_t)g.nx * g.ny * g.nz * g.nb;
  const int nblk = (int)((total + 255) / 256);
  if ((size_t)nblk > N->lpart_cap) {
    PMG_HOST_CHECK(hipStreamSynchronize(N->stream));
    if (N->lpart) PMG_HOST_CHECK(hipFree(N->lpart));
    PMG_HOST_CHECK(hipMalloc(&N->lpart, (size_t)nblk * sizeof(double)));
    N->lpart_cap = nblk;
  }
  const long long cx = g.nx - 2 * margin, cy = g.ny - 2 * margin, cz = g.nz - 2 * margin;
  double count = (double)(cx > 0 ? cx : 0) * (cy > 0 ? cy : 0) * (cz > 0 ? cz : 0) * g.nb;
  if (W) {
    // the weighted count, folded on the device into lsum[1] before the loss uses it
    hipLaunchKernelGGL(k_wcount, dim3(nblk), dim3(256), 0, N->stream, W, g, margin, N->lpart);
    hipLaunchKernelGGL(k_fold_d, dim3(1), dim3(256), 0, N->stream, N->lpart, nblk, N->lsum + 1);
  }
  hipLaunchKernelGGL(k_loss, dim3(nblk), dim3(256), 0, N->stream, N->yt, T, W, W ? N->lsum + 1 : (const double *)nullptr,
                     N->dy, N->lpart, g, margin, 1.0 / count);
  hipLaunchKernelGGL(k_fold_d, dim3(1), dim3(256), 0, N->stream, N->lpart, nblk, N->lsum);
  PMG_HOST_CHECK(hipGetLastError());
  const int zc = conv_zc(g, CTX, CTY, kConvBlocks);
  const dim3 gt(conv_blocks(g, CTX, CTY, zc)), blk(256);
  // layer 3: dW3 from A2 and dY; dZ2 = conv^T(dY) * gelu'(Z2)
  if ((rc = net_wgrad(N, g, 2, nullptr))) return rc;
  hipLaunchKernelGGL((k_conv_in_tile<uint16_t, 2>), gt, blk, 0, N->stream, N->dy, 1.0f, N->fr + FR_WBI,
                     (const float *)nullptr, N->z2, (float *)nullptr, N->d16b, g, zc);
  // layer 2
  if ((rc = net_wgrad(N, g, 1, nullptr))) return rc;
  hipLaunchKernelGGL(k_conv16_tile<2>, gt, blk, 0, N->stream, N->d16b, N->fr + FR_WPB2, (const float *)nullptr, N->z1,
                     (float *)nullptr, N->d16, g, zc);
  // layer 1
  if ((rc = net_wgrad(N, g, 0, x))) return rc;
  if (loss_out) {
    double l[2];
    PMG_HOST_CHECK(hipMemcpyAsync(l, N->lsum, 2 * sizeof(double), hipMemcpyDeviceToHost, N->stream));
    PMG_HOST_CHECK(hipStreamSynchronize(N->stream));
    if (W) count = l[1];
    *loss_out = count > 0 ? 0.5 * l[0] / count : 0.0;
  }
  return 0;
}

}  // namespace

extern "C" {

int pmg_net_mfma32_selftest(const float *A, const float *B, float *D_out) {
  // host A (16x32), B (32x16) rounded to bf16; D_out = A*B from one K = 32 MFMA
  std::vector<uint16_t> ha(512), hb(512);
  for (int i = 0; i < 512; i++) { ha[i] = f2bf(A[i]); hb[i] = f2bf(B[i]); }
  uint16_t *dA, *dB;
  float *dD;
  PMG_HOST_CHECK(hipMalloc(&dA, 1024));
  PMG_HOST_CHECK(hipMalloc(&dB, 1024));
  PMG_HOST_CHECK(hipMalloc(&dD, 1024));
  PMG_HOST_CHECK(hipMemcpy(dA, ha.data(), 1024, hipMemcpyHostToDevice));
  PMG_HOST_CHECK(hipMemcpy(dB, hb.data(), 1024, hipMemcpyHostToDevice));
  hipLaunchKernelGGL(k_mfma32_probe, dim3(1), dim3(64), 0, 0, dA, dB, dD);
  PMG_HOST_CHECK(hipGetLastError());
  PMG_HOST_CHECK(hipMemcpy(D_out, dD, 1024, hipMemcpyDeviceToHost));
  (void)hipFree(dA);
  (void)hipFree(dB);
  (void)hipFree(dD);
  return 0;
}

int pmg_net_mfma_selftest(const float *A, const float *B, float *D_out) {
  // host A (16x16), B (16x16) rounded to bf16; D_out = A*B from one MFMA
  std::vector<uint16_t> ha(256), hb(256);
  for (int i = 0; i < 256; i++) { ha[i] = f2bf(A[i]); hb[i] = f2bf(B[i]); }
  uint16_t *dA, *dB;
  float *dD;
  PMG_HOST_CHECK(hipMalloc(&dA, 512));
  PMG_HOST_CHECK(hipMalloc(&dB, 512));
  PMG_HOST_CHECK(hipMalloc(&dD, 1024));
  PMG_HOST_CHECK(hipMemcpy(dA, ha.data(), 512, hipMemcpyHostToDevice));
  PMG_HOST_CHECK(hipMemcpy(dB, hb.data(), 512, hipMemcpyHostToDevice));
  hipLaunchKernelGGL(k_mfma_probe, dim3(1), dim3(64), 0, 0, dA, dB, dD);
  PMG_HOST_CHECK(hipGetLastError());
  PMG_HOST_CHECK(hipMemcpy(D_out, dD, 1024, hipMemcpyDeviceToHost));
  (void)hipFree(dA);
  (void)hipFree(dB);
  (void)hipFree(dD);
  return 0;
}

pmg_net *pmg_net_create(int hidden, unsigned long long seed) {
  if (hidden != 16) return nullptr;
  pmg_net *N = new pmg_net();
  if (hipStreamCreate(&N->stream) != hipSuccess) { delete N; return nullptr; }
  const size_t nf = 3 * (size_t)LAYER_FLOATS;
  std::vector<float> w(nf, 0.f);
  std::vector<uint8_t> mask(nf, 0);
  // splitmix64-driven uniform init, He-like scale; padding stays zero
  unsigned long long st = seed;
  auto rnd = [&]() {
    st += 0x9E3779B97F4A7C15ull;
    unsigned long long z = st;
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    z ^= z >> 31;
    return (double)(z >> 11) * (1.0 / 9007199254740992.0);
  };
  const int cin[3] = {1, 16, 16}, cout[3] = {16, 16, 1};
  for (int l = 0; l < 3; l++) {
    const double sc = std::sqrt(3.0 / (27.0 * cin[l]));
    for (int t = 0; t < NTAP; t++)
      for (int ci = 0; ci < cin[l]; ci++)
        for (int co = 0; co < cout[l]; co++) {
          const size_t idx = (size_t)l * LAYER_FLOATS + t * 256 + ci * 16 + co;
          w[idx] = (float)((2.0 * rnd() - 1.0) * sc);
          mask[idx] = 1;
        }
    for (int co = 0; co < cout[l]; co++) mask[(size_t)l * LAYER_FLOATS + NTAP * 256 + co] = 1;
  }
  bool ok = hipMalloc(&N->w, nf * 4) == hipSuccess && hipMalloc(&N->m1, nf * 4) == hipSuccess &&
            hipMalloc(&N->m2, nf * 4) == hipSuccess && hipMalloc(&N->grad, nf * 4) == hipSuccess &&
            hipMalloc(&N->mask, nf) == hipSuccess &&
            hipMalloc(&N->fr, FR_TOTAL * sizeof(uint16_t)) == hipSuccess &&
            hipMalloc(&N->lsum, 2 * sizeof(double)) == hipSuccess;
  // the weight gradients' planes take more LDS than a kernel gets by default
  for (const void *k : {reinterpret_cast<const void *>(&k_wgrad_tile<1>), reinterpret_cast<const void *>(&k_wgrad_tile<16>)})
    ok = ok && hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)kWgradLds) == hipSuccess;
  if (!ok) { pmg_net_destroy(N); return nullptr; }
  (void)hipMemcpy(N->w, w.data(), nf * 4, hipMemcpyHostToDevice);
  (void)hipMemcpy(N->mask, mask.data(), nf, hipMemcpyHostToDevice);
  (void)hipMemset(N->m1, 0, nf * 4);
  (void)hipMemset(N->m2, 0, nf * 4);
  (void)hipMemset(N->grad, 0, nf * 4);
  return N;
}

void pmg_net_destroy(pmg_net *N) {
  if (!N) return;
  if (N->stream) (void)hipStreamSynchronize(N->stream);
  for (void *p : {(void *)N->w, (void *)N->m1, (void *)N->m2, (void *)N->grad, (void *)N->mask, (void *)N->fr,
                  (void *)N->a1, (void *)N->a2, (void *)N->d16, (void *)N->d16b, (void *)N->dy, (void *)N->z1,
                  (void *)N->z2, (void *)N->yt, (void *)N->ia1, (void *)N->ia2, (void *)N->y, (void *)N->partial,
                  (void *)N->lpart, (void *)N->lsum})
    if (p) (void)hipFree(p);
  if (N->stream) (void)hipStreamDestroy(N->stream);
  delete N;
}

// Weights in the oracle's layout (oracle/mg_oracle.h): w1[16][1][27], b1[16],
// w2[16][16][27], b2[16], w3[1][16][27], b3[1]; FP64 on the host.
int pmg_net_set_weights(pmg_net *N, const double *w1, const double *b1, const double *w2,
                        const double *b2, const double *w3, const double *b3) {
  if (!N) return -1;
  std::vector<float> w(3 * (size_t)LAYER_FLOATS, 0.f);
  for (int co = 0; co < 16; co++) {
    for (int t = 0; t < NTAP; t++) {
      w[0 * LAYER_FLOATS + t * 256 + 0 * 16 + co] = (float)w1[co * 27 + t];
      for (int ci = 0; ci < 16; ci++)
        w[1 * LAYER_FLOATS + t * 256 + ci * 16 + co] = (float)w2[(co * 16 + ci) * 27 + t];
    }
    w[0 * LAYER_FLOATS + NTAP * 256 + co] = (float)b1[co];
    w[1 * LAYER_FLOATS + NTAP * 256 + co] = (float)b2[co];
  }
  for (int ci = 0; ci < 16; ci++)
    for (int t = 0; t < NTAP; t++) w[2 * LAYER_FLOATS + t * 256 + ci * 16 + 0] = (float)w3[ci * 27 + t];
  w[2 * LAYER_FLOATS + NTAP * 256 + 0] = (float)b3[0];
  PMG_HOST_CHECK(hipMemcpy(N->w, w.data(), w.size() * 4, hipMemcpyHostToDevice));
  N->frags_valid = false;
  return 0;
}

static void from_master(const std::vector<float> &w, double *w1, double *b1, double *w2, double *b2,
                        double *w3, double *b3) {
  for (int co = 0; co < 16; co++) {
    for (int t = 0; t < NTAP; t++) {
      w1[co * 27 + t] = w[0 * LAYER_FLOATS + t * 256 + co];
      for (int ci = 0; ci < 16; ci++) w2[(co * 16 + ci) * 27 + t] = w[1 * LAYER_FLOATS + t * 256 + ci * 16 + co];
    }
    b1[co] = w[0 * LAYER_FLOATS + NTAP * 256 + co];
    b2[co] = w[1 * LAYER_FLOATS + NTAP * 256 + co];
  }
  for (int ci = 0; ci < 16; ci++)
    for (int t = 0; t < NTAP; t++) w3[ci * 27 + t] = w[2 * LAYER_FLOATS + t * 256 + ci * 16];
  b3[0] = w[2 * LAYER_FLOATS + NTAP * 256];
}

int pmg_net_get_weights(pmg_net *N, double *w1, double *b1, double *w2, double *b2, double *w3,
                        double *b3) {
  if (!N) return -1;
  std::vector<float> w(3 * (size_t)LAYER_FLOATS);
  PMG_HOST_CHECK(hipStreamSynchronize(N->stream));
  PMG_HOST_CHECK(hipMemcpy(w.data(), N->w, w.size() * 4, hipMemcpyDeviceToHost));
  from_master(w, w1, b1, w2, b2, w3, b3);
  return 0;
}

// Forward on nb boxes of nx*ny*nz points: x (device fp32 [nb][P]) -> y
// (device fp32 [nb][P]).
int pmg_net_forward(pmg_net *N, const float *x, float *y, int nx, int ny, int nz, int nb) {
  if (!N || !x || !y || nx < 1 || ny < 1 || nz < 1 || nb < 1) return -1;
  const size_t P = (size_t)nx * ny * nz * nb;
  if (net_ensure(N, P)) return -1;
  Geom g{nx, ny, nz, nb};
  int rc = net_forward(N, x, y, g);
  if (rc) return rc;
  PMG_HOST_CHECK(hipStreamSynchronize(N->stream));
  return 0;
}

// Loss and gradients (oracle layout, host FP64) for inputs x and targets t
// (device fp32 [nb][P]); margin = points near box faces excluded from the loss.
int pmg_net_loss_grad(pmg_net *N, const float *x, const float *t, int nx, int ny, int nz, int nb,
                      int margin, double *loss, double *gw1, double *gb1, double *gw2, double *gb2,
                      double *gw3, double *gb3) {
  if (!N || !x || !t) return -1;
  const size_t P = (size_t)nx * ny * nz * nb;
  if (net_ensure(N, P)) return -1;
  Geom g{nx, ny, nz, nb};
  int rc = net_loss_backward(N, g, x, t, nullptr, margin, loss);
  if (rc) return rc;
  std::vector<float> gr(3 * (size_t)LAYER_FLOATS);
  PMG_HOST_CHECK(hipMemcpy(gr.data(), N->grad, gr.size() * 4, hipMemcpyDeviceToHost));
  from_master(gr, gw1, gb1, gw2, gb2, gw3, gb3);
  return 0;
}

// Loss and gradients as pmg_net_loss_grad, the mean taken over the points
// with w != 0 (w: device fp32 [nb][P]) that also satisfy the margin rule.
int pmg_net_loss_grad_w(pmg_net *N, const float *x, const float *t, const float *w, int nx, int ny, int nz,
                        int nb, int margin, double *loss, double *gw1, double *gb1, double *gw2, double *gb2,
                        double *gw3, double *gb3) {
  if (!N || !x || !t || !w) return -1;
  const size_t P = (size_t)nx * ny * nz * nb;
  if (net_ensure(N, P)) return -1;
  Geom g{nx, ny, nz, nb};
  int rc = net_loss_backward(N, g, x, t, w, margin, loss);
  if (rc) return rc;
  std::vector<float> gr(3 * (size_t)LAYER_FLOATS);
  PMG_HOST_CHECK(hipMemcpy(gr.data(), N->grad, gr.size() * 4, hipMemcpyDeviceToHost));
  from_master(gr, gw1, gb1, gw2, gb2, gw3, gb3);
  return 0;
}

// One Adam step on a batch (device fp32 inputs/targets; w optional weights
// as in pmg_net_loss_grad_w, NULL for every point past the margin).
int pmg_net_train_step_w(pmg_net *N, const float *x, const float *t, const float *w, int nx, int ny, int nz,
                         int nb, int margin, float lr, double *loss) {
  if (!N || !x || !t) return -1;
  const size_t P = (size_t)nx * ny * nz * nb;
  if (net_ensure(N, P)) return -1;
  Geom g{nx, ny, nz, nb};
  int rc = net_loss_backward(N, g, x, t, w, margin, loss);
  if (rc) return rc;
  N->adam_t++;
  const float b1 = 0.9f, b2 = 0.999f;
  const float c1 = 1.f - std::pow(b1, (float)N->adam_t), c2 = 1.f - std::pow(b2, (float)N->adam_t);
  const int nf = 3 * LAYER_FLOATS;
  hipLaunchKernelGGL(k_adam, dim3((nf + 255) / 256), dim3(256), 0, N->stream, N->w, N->m1, N->m2, N->grad,
                     N->mask, nf, lr, b1, b2, c1, c2, 1e-8f);
  PMG_HOST_CHECK(hipGetLastError());
  N->frags_valid = false;
  return 0;
}

// One Adam step on a batch (device fp32 inputs/targets).
int pmg_net_train_step(pmg_net *N, const float *x, const float *t, int nx, int ny, int nz, int nb,
                       int margin, float lr, double *loss) {
  if (!N || !x || !t) return -1;
  const size_t P = (size_t)nx * ny * nz * nb;
  if (net_ensure(N, P)) return -1;
  Geom g{nx, ny, nz, nb};
  int rc = net_loss_backward(N, g, x, t, nullptr, margin, loss);
  if (rc) return rc;
  N->adam_t++;
  const float b1 = 0.9f, b2 = 0.999f;
  const float c1 = 1.f - std::pow(b1, (float)N->adam_t), c2 = 1.f - std::pow(b2, (float)N->adam_t);
  const int nf = 3 * LAYER_FLOATS;
  hipLaunchKernelGGL(k_adam, dim3((nf + 255) / 256), dim3(256), 0, N->stream, N->w, N->m1, N->m2, N->grad,
                     N->mask, nf, lr, b1, b2, c1, c2, 1e-8f);
  PMG_HOST_CHECK(hipGetLastError());
  N->frags_valid = false;
  return 0;
}

void *pmg_net_stream(pmg_net *N) { return N ? (void *)N->stream : nullptr; }

// Learned correction on one grid, on the caller's stream: y = N(scale * x)
// (x device FP32, e.g. the negated defect the mixed solver keeps), then
// u += coef * y at interior points.  The output stays in the network's
// buffer so pmg_net_recorrect can undo or repeat the step.
int pmg_net_correct(pmg_net *N, const float *x, float scale, double *u, double coef, int nx,
                    int ny, int nz, void *stream) {
  if (!N || !x || !u) return -1;
  hipStream_t st = (hipStream_t)stream;
  const size_t P = (size_t)nx * ny * nz;
  if (net_ensure_infer(N, P)) return -1;
  hipStream_t keep = N->stream;
  N->stream = st;
  int rc = net_infer(N, x, scale, N->y, Geom{nx, ny, nz, 1});
  N->stream = keep;
  if (rc) return rc;
  hipLaunchKernelGGL((k_apply_correction<double, 1>), dim3((nx + 63) / 64, (ny + 3) / 4, nz), dim3(256), 0, st, u,
                     N->y, nx, ny, nz, coef);
  PMG_HOST_CHECK(hipGetLastError());
  return 0;
}

int pmg_net_recorrect(pmg_net *N, double *u, double coef, int nx, int ny, int nz, void *stream) {
  if (!N || !u || (size_t)nx * ny * nz > N->icap) return -1;
  hipLaunchKernelGGL((k_apply_correction<double, 1>), dim3((nx + 63) / 64, (ny + 3) / 4, nz), dim3(256), 0,
                     (hipStream_t)stream, u, N->y, nx, ny, nz, coef);
  PMG_HOST_CHECK(hipGetLastError());
  return 0;
}

int pmg_net_reserve(pmg_net *N, long long points) {
  if (!N || points < 1) return -1;
  if (net_ensure_infer(N, (size_t)points)) return -1;
  if (net_frags(N)) return -1;
  PMG_HOST_CHECK(hipStreamSynchronize(N->stream));
  return 0;
}

// y = N(scale * x) on nb boxes, enqueued on `stream` with no host
// synchronisation (capturable in a graph once pmg_net_reserve has sized the
// buffers and packed the weights: then nothing is allocated or packed
// here).  Returns the network-owned output buffer (fp32 [nb][P], valid until
// the next inference), or NULL on error.
float *pmg_net_infer_async(pmg_net *N, const float *x, float scale, int nx, int ny, int nz, int nb, void *stream) {
  if (!N || !x || nx < 1 || ny < 1 || nz < 1 || nb < 1) return nullptr;
  const size_t P = (size_t)nx * ny * nz * nb;
  if (net_ensure_infer(N, P)) return nullptr;
  hipStream_t keep = N->stream;
  N->stream = (hipStream_t)stream;
  const int rc = net_infer(N, x, scale, N->y, Geom{nx, ny, nz, nb});
  N->stream = keep;
  return rc ? nullptr : N->y;
}

int pmg_net_infer(pmg_net *N, const float *x, float scale, float *y, int nx, int ny, int nz, int nb) {
  if (!N || !x || !y || nx < 1 || ny < 1 || nz < 1 || nb < 1) return -1;
  const size_t P = (size_t)nx * ny * nz * nb;
  if (net_ensure_infer(N, P)) return -1;
  int rc = net_infer(N, x, scale, y, Geom{nx, ny, nz, nb});
  if (rc) return rc;
  PMG_HOST_CHECK(hipStreamSynchronize(N->stream));
  return 0;
}

// Crops for training: out[c][z][y][x] = scale * (a[p] - b[p]) (b may be
// NULL) for cubes of side `side` at host-given origins (ox, oy, oz).
__global__ void k_gather_crops(const double *__restrict__ a, const double *__restrict__ b, int nx, int ny,
                               const int *__restrict__ org, int side, double scale, float *__restrict__ out) {
  const int c = blockIdx.y;
  const size_t n = (size_t)side * side * side;
  const size_t q = (size_t)blockIdx.x * 256 + threadIdx.x;
  if (q >= n) return;
  const int x = (int)(q % side), y = (int)((q / side) % side), z = (int)(q / ((size_t)side * side));
  const size_t p = ix3(org[3 * c] + x, org[3 * c + 1] + y, org[3 * c + 2] + z, nx, ny);
  const double v = b ? a[p] - b[p] : a[p];
  out[(size_t)c * n + q] = (float)(scale * v);
}

int pmg_gather_crops(const double *a, const double *b, int nx, int ny, int nz, const int *origins_host,
                     int ncrop, int side, double scale, float *out, void *stream) {
  if (!a || !out || ncrop < 1 || side < 1) return -1;
  for (int c = 0; c < ncrop; c++)
    for (int d = 0; d < 3; d++) {
      const int o = origins_host[3 * c + d], n = d == 0 ? nx : (d == 1 ? ny : nz);
      if (o < 0 || o + side > n) return -1;
    }
  int *dorg;
  PMG_HOST_CHECK(hipMalloc(&dorg, sizeof(int) * 3 * ncrop));
  PMG_HOST_CHECK(hipMemcpyAsync(dorg, origins_host, sizeof(int) * 3 * ncrop, hipMemcpyHostToDevice,
                                (hipStream_t)stream));
  const size_t n = (size_t)side * side * side;
  hipLaunchKernelGGL(k_gather_crops, dim3((unsigned)((n + 255) / 256), ncrop), dim3(256), 0, (hipStream_t)stream,
                     a, b, nx, ny, dorg, side, scale, out);
  PMG_HOST_CHECK(hipGetLastError());
  PMG_HOST_CHECK(hipStreamSynchronize((hipStream_t)stream));
  PMG_HOST_CHECK(hipFree(dorg));
  return 0;
}

}  // extern "C"
