// Kernels of the warm-start network: 3x3x3 convolutions as implicit GEMMs
// on the gfx950 matrix cores (v_mfma_f32_16x16x32_bf16: BF16 operands,
// FP32 accumulation), average pooling, nearest upsampling, skip additions,
// ReLU, the MSE loss and Adam.
//
// Tensors are voxel-major with channels fastest: T[v*C + c], v = x + X*(y +
// Y*z) -- the same order as the solver's packed vectors (r, theta, phi).
// Activations are BF16 (raw bits in uint16); gradients are FP32; weights
// are kept in FP32 (Adam state) with a BF16 copy [tap][c_out][c_in] for the
// matrix cores.  The z axis (phi) is periodic, x and y are zero-padded.
//
// MFMA 16x16x32 operand layout (lane l of a wave64): A row l%16 and B column
// l%16, each with the eight k of group l/16 (the order of the k does not
// matter as long as A and B agree); D (16 x 16): lane holds D[4*(l/16) ..
// 4*(l/16)+3][l%16].  p3d_nn_mfma_check is there to compare it, and the
// transposing LDS read, with a host matmul.
//
// Every BF16 tensor is preceded by kZeroFront zero bytes (the allocation's
// first ones): a tap that falls outside the grid reads those.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>

#include "p3d_nn.hpp"

namespace p3d {
namespace nn {

typedef short bf16x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ uint16_t f2bf(float f) {
  uint32_t u = __float_as_uint(f);
  if ((u & 0x7f800000u) == 0x7f800000u) return (uint16_t)(u >> 16);  // inf/nan
  u += 0x7fffu + ((u >> 16) & 1u);  // round to nearest even
  return (uint16_t)(u >> 16);
}
__device__ __forceinline__ float bf2f(uint16_t b) { return __uint_as_float((uint32_t)b << 16); }

__device__ __forceinline__ f32x4 mfma32(u32x4 a, u32x4 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a),
                                                 __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}
__device__ __forceinline__ unsigned pack2(float lo, float hi) {
  return (unsigned)f2bf(lo) | ((unsigned)f2bf(hi) << 16);
}
// the two BF16 values of a word
__device__ __forceinline__ float lo2f(unsigned w) { return __uint_as_float(w << 16); }
__device__ __forceinline__ float hi2f(unsigned w) { return __uint_as_float(w & 0xffff0000u); }

struct Dims {
  int X, Y, Z;
  int V;
};

// Tap t = (dx+1) + 3*(dy+1) + 9*(dz+1).
__device__ __forceinline__ void coords(const Dims& d, int v, int& x, int& y, int& z) {
  x = v % d.X;
  const int r = v / d.X;
  y = r % d.Y;
  z = r / d.Y;
}

// ---------------------------------------------------------------------------
// y[v][co] = act( sum_t sum_ci x[nb(v,t)][ci] w[t][co][ci] + bias[co] )
// One wave: MT x 16 voxels times NB x 16 output channels; grid (voxels / (64
// MT), Cout / (16 NB)), block 256.  The weights are the MFMA's A operand and
// the voxels its B operand, so a lane ends with four channels of one voxel.
// DIR -1 mirrors the taps' shifts (input gradients).
// K runs over 32 channels of a tap; with 16 channels over two taps at a time
// (lanes 0-31 the even, 32-63 the odd one; the 28th tap is empty).
//
// What bounds it: the voxel operand, 16 bytes a lane read from L1/L2 once per
// tap and 32 channels (27 times the tensor), and the index arithmetic before
// it.  MT tiles share a weight fragment and give the loads of one step
// something to overlap with.  The eight convolutions of a forward pass at
// 51x91x181: 1123 us with one 16 x 16 tile a wave and 8-byte operands, 394 us
// with this kernel alone, 296 us with k_conv_lds for 32 channels and more and
// DIR known to the compiler (the three of 16 channels here 38, 38 and 13 us).
struct ConvOut {
  uint16_t* y;        // BF16 result (after the ReLU), or null
  const uint16_t* e;  // BF16 skip input, or null
  uint16_t* s;        // with e: the BF16 sum y + e
  float* yf;          // FP32 result, all channels, or null
  float* y1;          // FP32 result, channel 0 alone, or null
  const float* bias;  // or null
  int relu;
};

// The results of a wave: four channels of a voxel per lane and tile.
template <int NB, int MT>
__device__ __forceinline__ void conv_store(const Dims& d, int Cout, const ConvOut& o,
                                           const f32x4 (&acc)[NB][MT], int v0, int co0, int m,
                                           int kb) {
#pragma unroll
  for (int n = 0; n < NB; n++) {
    const int co = co0 + n * 16 + 4 * kb;
    f32x4 bias = {0.f, 0.f, 0.f, 0.f};
    if (o.bias) bias = *(const f32x4*)(o.bias + co);
#pragma unroll
    for (int t = 0; t < MT; t++) {
      const int v = v0 + t * 16 + m;
      if (v >= d.V) continue;
      f32x4 r = acc[n][t] + bias;
      if (o.relu)
#pragma unroll
        for (int i = 0; i < 4; i++) r[i] = r[i] < 0.f ? 0.f : r[i];
      const size_t at = (size_t)v * Cout + co;
      if (o.y) {
        const uint2 y = make_uint2(pack2(r[0], r[1]), pack2(r[2], r[3]));
        *(uint2*)(o.y + at) = y;
        if (o.e) {
          const uint2 e = *(const uint2*)(o.e + at);
          *(uint2*)(o.s + at) =
              make_uint2(pack2(lo2f(y.x) + lo2f(e.x), hi2f(y.x) + hi2f(e.x)),
                         pack2(lo2f(y.y) + lo2f(e.y), hi2f(y.y) + hi2f(e.y)));
        }
      }
      if (o.yf) *(f32x4*)(o.yf + at) = r;
      if (o.y1 && co == 0) o.y1[v] = r[0];
    }
  }
}

template <int CIN, int NB, int MT, int DIR>
__global__ void __launch_bounds__(256)
    k_conv(Dims d, int Cout, const uint16_t* __restrict__ x, const uint16_t* __restrict__ w,
           ConvOut o) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int m = lane & 15, kb = lane >> 4, h = kb >> 1;
  // a contiguous range of voxels per XCD (workgroups go round the 8 XCDs):
  // a tensor's neighbouring planes then meet in one L2
  const int per = (int)gridDim.x / 8;
  const int blk = (int)blockIdx.x < 8 * per
                      ? ((int)blockIdx.x & 7) * per + ((int)blockIdx.x >> 3)
                      : (int)blockIdx.x;
  const int v0 = (blk * 4 + wave) * (16 * MT);
  const int co0 = blockIdx.y * (16 * NB);
  constexpr unsigned kQ = CIN / 8;  // 16-byte words of a voxel
  const u32x4* xq = (const u32x4*)x - kZeroFront / 16;
  const unsigned lane_q = kZeroFront / 16 + (CIN == 16 ? (unsigned)(kb & 1) : (unsigned)kb);
  constexpr bool fw = DIR > 0;
  const unsigned XQ = (unsigned)DIR * kQ * (unsigned)d.X, PQ = kQ * (unsigned)d.X * (unsigned)d.Y;
  unsigned base[MT], zlo[MT], zhi[MT];
  bool in[MT], xm[MT], xp[MT], ym[MT], yp[MT];
#pragma unroll
  for (int t = 0; t < MT; t++) {
    const int v = v0 + t * 16 + m;
    int vx = 0, vy = 0, vz = 0;
    in[t] = v < d.V;
    if (in[t]) coords(d, v, vx, vy, vz);
    base[t] = lane_q + kQ * (unsigned)(in[t] ? v : 0);
    const unsigned zl = vz > 0 ? 0u - PQ : PQ * (unsigned)(d.Z - 1);
    const unsigned zh = vz < d.Z - 1 ? PQ : 0u - PQ * (unsigned)(d.Z - 1);
    zlo[t] = fw ? zl : zh;
    zhi[t] = fw ? zh : zl;
    xm[t] = in[t] && (fw ? vx > 0 : vx < d.X - 1);
    xp[t] = in[t] && (fw ? vx < d.X - 1 : vx > 0);
    ym[t] = fw ? vy > 0 : vy < d.Y - 1;
    yp[t] = fw ? vy < d.Y - 1 : vy > 0;
  }
  // index and validity of tap t (a constant) for tile q
  auto tap_ok = [&](int q, int t) {
    const int dx = t % 3, dy = (t / 3) % 3;
    const bool vx = dx == 0 ? xm[q] : (dx == 2 ? xp[q] : in[q]);
    return t < 27 && vx && (dy == 0 ? ym[q] : (dy == 2 ? yp[q] : true));
  };
  auto tap_off = [&](int q, int t) {
    const int dx = t % 3 - 1, dy = (t / 3) % 3 - 1, dz = t / 9;
    return (unsigned)(dx * DIR * (int)kQ) + (unsigned)dy * XQ +
           (dz == 0 ? zlo[q] : (dz == 2 ? zhi[q] : 0u));
  };
  f32x4 acc[NB][MT];
#pragma unroll
  for (int n = 0; n < NB; n++)
#pragma unroll
    for (int t = 0; t < MT; t++) acc[n][t] = f32x4{0.f, 0.f, 0.f, 0.f};
  const u32x4 zero = {0u, 0u, 0u, 0u};
  if constexpr (CIN == 16) {
    const u32x4* wq = (const u32x4*)w + (size_t)(co0 + m) * kQ + (kb & 1);
    const size_t wt = (size_t)Cout * kQ;
#pragma unroll
    for (int s = 0; s < 14; s++) {
      u32x4 av[NB], bv[MT];
#pragma unroll
      for (int n = 0; n < NB; n++) {
        const u32x4* p = wq + (size_t)n * 16 * kQ;
        av[n] = p[wt * (size_t)(h && s < 13 ? 2 * s + 1 : 2 * s)];
        if (s == 13 && h) av[n] = zero;
      }
#pragma unroll
      for (int t = 0; t < MT; t++) {
        const bool ok = h ? tap_ok(t, 2 * s + 1) : tap_ok(t, 2 * s);
        const unsigned off = h ? tap_off(t, 2 * s + 1) : tap_off(t, 2 * s);
        bv[t] = xq[ok ? base[t] + off : lane_q - kZeroFront / 16];
      }
#pragma unroll
      for (int n = 0; n < NB; n++)
#pragma unroll
        for (int t = 0; t < MT; t++) acc[n][t] = mfma32(av[n], bv[t], acc[n][t]);
    }
  } else {
    const u32x4* wq = (const u32x4*)w + (size_t)(co0 + m) * kQ + kb;
    const size_t wt = (size_t)Cout * kQ;
#pragma unroll 1
    for (int dz = 0; dz < 3; dz++) {
      unsigned bz[MT];
#pragma unroll
      for (int t = 0; t < MT; t++)
        bz[t] = base[t] + (dz == 0 ? zlo[t] : (dz == 2 ? zhi[t] : 0u));
      const u32x4* wz = wq + wt * (size_t)(9 * dz);
#pragma unroll
      for (int r = 0; r < 9; r++) {
        unsigned idx[MT];
#pragma unroll
        for (int t = 0; t < MT; t++)
          idx[t] = tap_ok(t, r) ? bz[t] + (unsigned)((r % 3 - 1) * DIR * (int)kQ) +
                                      (unsigned)(r / 3 - 1) * XQ
                                : lane_q - kZeroFront / 16;
#pragma unroll
        for (int c = 0; c < CIN / 32; c++) {
          u32x4 av[NB], bv[MT];
#pragma unroll
          for (int n = 0; n < NB; n++) av[n] = wz[wt * (size_t)r + (size_t)n * 16 * kQ + 4 * c];
#pragma unroll
          for (int t = 0; t < MT; t++) bv[t] = xq[idx[t] + 4u * c];
#pragma unroll
          for (int n = 0; n < NB; n++)
#pragma unroll
            for (int t = 0; t < MT; t++) acc[n][t] = mfma32(av[n], bv[t], acc[n][t]);
        }
      }
    }
  }
  conv_store<NB, MT>(d, Cout, o, acc, v0, co0, m, kb);
}

// The same for 32 channels and more with the voxels' neighbourhoods staged in
// LDS: for each dz the 64 MT voxels of the workgroup and one row and one voxel
// to either side, as they lie in memory, then nine taps from there.  Read
// straight from memory the 27 taps take each voxel 27 times through L1, which
// does not hold the neighbourhoods of a CU's workgroups; so it comes in three
// times (and its edges).  At 51x91x181: 32->16 channels at 780 thousand
// voxels 104 -> 63 us, 64->32 at 101 thousand 101 -> 60 us, 128->64 at 13
// thousand 75 -> 55 us.
// A row's 16-byte words are stored exchanged by the row's number, so that the
// 16 rows of a read lie in different banks.
template <int CIN>
__device__ __forceinline__ int lds_word(int row, int w) {
  constexpr int Q = CIN / 8;
  return row * Q + (w ^ ((Q >= 16 ? row : Q == 8 ? row >> 1 : row >> 2) & (Q - 1)));
}

__host__ __device__ inline int conv_lds_rows(int MT, int X) { return 64 * MT + 2 * X + 2; }

template <int CIN, int NB, int MT, int DIR>
__global__ void __launch_bounds__(256)
    k_conv_lds(Dims d, int Cout, const uint16_t* __restrict__ x, const uint16_t* __restrict__ w,
               ConvOut o) {
  constexpr int Q = CIN / 8;
  extern __shared__ u32x4 sx[];  // conv_lds_rows rows and a row of zeros
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int m = lane & 15, kb = lane >> 4;
  const int per = (int)gridDim.x / 8;  // (as in k_conv)
  const int blk = (int)blockIdx.x < 8 * per
                      ? ((int)blockIdx.x & 7) * per + ((int)blockIdx.x >> 3)
                      : (int)blockIdx.x;
  const int vb = blk * (64 * MT), v0 = vb + wave * (16 * MT);
  const int co0 = blockIdx.y * (16 * NB);
  const int rows = conv_lds_rows(MT, d.X), XY = d.X * d.Y;
  if (tid < Q) sx[rows * Q + tid] = u32x4{0u, 0u, 0u, 0u};
  unsigned ok[MT];  // bit dx + 3 dy: that shift stays in the grid
#pragma unroll
  for (int t = 0; t < MT; t++) {
    const int v = v0 + t * 16 + m;
    ok[t] = 0;
    if (v < d.V) {
      int vx, vy, vz;
      coords(d, v, vx, vy, vz);
      constexpr bool fw = DIR > 0;
      const unsigned fx = (vx > 0 ? (fw ? 1u : 4u) : 0u) | 2u |
                          (vx < d.X - 1 ? (fw ? 4u : 1u) : 0u);
      ok[t] = (vy > 0 ? fx << (fw ? 0 : 6) : 0u) | fx << 3 |
              (vy < d.Y - 1 ? fx << (fw ? 6 : 0) : 0u);
    }
  }
  f32x4 acc[NB][MT];
#pragma unroll
  for (int n = 0; n < NB; n++)
#pragma unroll
    for (int t = 0; t < MT; t++) acc[n][t] = f32x4{0.f, 0.f, 0.f, 0.f};
  const u32x4* xq = (const u32x4*)x;
  const u32x4* wq = (const u32x4*)w + (size_t)(co0 + m) * Q + kb;
  const size_t wt = (size_t)Cout * Q;
#pragma unroll 1
  for (int dz = 0; dz < 3; dz++) {
    if (dz) __syncthreads();
    // rows vb - X - 1 + XY (dz - 1) on (mirrored: 1 - dz): where they leave the plane or the
    // grid in x or y no tap reads them; in z they are V-periodic (a grid of
    // few planes can leave the range even so)
    const int base = vb - d.X - 1 + XY * (dz - 1) * DIR;
    // six loads of a thread in flight at a time
    constexpr int kB = 6;
    for (int e0 = tid; e0 < rows * Q; e0 += 256 * kB) {
      u32x4 b[kB];
#pragma unroll
      for (int u = 0; u < kB; u++) {
        const int e = min(e0 + 256 * u, rows * Q - 1);
        int v = base + e / Q;
        v = v < 0 ? v + d.V : v;
        v = v >= d.V ? v - d.V : v;
        v = max(0, min(v, d.V - 1));
        b[u] = xq[(size_t)v * Q + e % Q];
      }
#pragma unroll
      for (int u = 0; u < kB; u++) {
        const int e = e0 + 256 * u;
        if (e < rows * Q) sx[lds_word<CIN>(e / Q, e % Q)] = b[u];
      }
    }
    __syncthreads();
    const u32x4* wz = wq + wt * (size_t)(9 * dz);
#pragma unroll
    for (int r = 0; r < 9; r++) {
      const int shift = d.X + 1 + ((r % 3 - 1) + (r / 3 - 1) * d.X) * DIR;
      int row[MT];
#pragma unroll
      for (int t = 0; t < MT; t++)
        row[t] = (ok[t] >> r) & 1u ? (wave * MT + t) * 16 + m + shift : rows;
#pragma unroll
      for (int c = 0; c < CIN / 32; c++) {
        u32x4 av[NB], bv[MT];
#pragma unroll
        for (int n = 0; n < NB; n++) av[n] = wz[wt * (size_t)r + (size_t)n * 16 * Q + 4 * c];
#pragma unroll
        for (int t = 0; t < MT; t++) bv[t] = sx[lds_word<CIN>(row[t], 4 * c + kb)];
#pragma unroll
        for (int n = 0; n < NB; n++)
#pragma unroll
          for (int t = 0; t < MT; t++) acc[n][t] = mfma32(av[n], bv[t], acc[n][t]);
      }
    }
  }
  conv_store<NB, MT>(d, Cout, o, acc, v0, co0, m, kb);
}

// dst[t][ci][co] = src[t][co][ci] for every convolution of the parameter
// buffer: the gradient of a convolution's input is the convolution of the
// output's gradient with these weights and mirrored shifts (dx[v][ci] = sum_t
// sum_co dy[nb(v,-t)][co] w[t][co][ci], added in that order).
__global__ void k_transpose_weights(ConvTable ct, const uint16_t* __restrict__ src,
                                    uint16_t* __restrict__ dst) {
  const ConvTable::Entry c = ct.e[blockIdx.y];
  const int e = blockIdx.x * 256 + threadIdx.x, cc = c.Cin * c.Cout;
  if (e >= 27 * cc) return;
  const int t = e / cc, r = e - t * cc, ci = r / c.Cout, co = r - ci * c.Cout;
  dst[c.w_off + e] = src[c.w_off + (size_t)t * cc + (size_t)co * c.Cin + ci];
}

// Partial weight gradients: part[chunk][t][co][ci] = sum over the chunk's
// voxels of dy[v][co] x[nb(v,t)][ci].  grid (chunks, (Cout/(16 COB)) *
// (Cin/(16 CIB))), block 256.
//
// K of this contraction is the voxels, which neither operand has innermost:
// 128 (or 96) voxels of dy and, for each of the nine (dy, dz) shifts, the 130 voxels
// of x that the three dx need are staged in LDS as they lie in memory, and the
// transposing LDS read (ds_read_b64_tr_b16: sixteen lanes read a 4 x 16 block
// by rows and receive it by columns) hands the matrix unit its operands.
// Wave w takes taps w, w + 4, ... and keeps their 16 x 16 results in
// registers over the whole chunk.  A tap outside the grid reads a row of
// zeros.
//
// What bounds it: memory latency of a step, then the LDS reads, 512 bytes for
// every four k of a tap, and the index arithmetic before each.  So the next
// step's values are asked for before the taps of this one.  The eight weight
// gradients of a backward pass at 51x91x181: 4183 us with two-byte loads from
// memory, 560 us staged step by step, 312 us so.
// voxels per step: 128, 96 where two workgroups would not fit a CU's LDS
constexpr int wgrad_step(int cib, int cob) { return cib == 2 && cob == 2 ? 96 : 128; }

typedef __attribute__((address_space(3))) bf16x4 lds_bf16x4;
__device__ __forceinline__ uint2 lds_read_tr(const uint16_t* p) {
  return __builtin_bit_cast(uint2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_bf16x4*)p));
}

template <int CIB, int COB>
__global__ void __launch_bounds__(256)
    k_conv_bwd_weight(Dims d, int Cin, int Cout, int chunk, const uint16_t* __restrict__ dy,
                      const uint16_t* __restrict__ x, float* __restrict__ part) {
  constexpr int XQ = 2 * CIB, YQ = 2 * COB;  // 16-byte words of a row
  constexpr int kWV = wgrad_step(CIB, COB), kWR = kWV + 2;  // rows of a segment
  __shared__ u32x4 sx[(9 * kWR + 1) * XQ];   // the last row is zero
  __shared__ u32x4 sy[kWV * YQ];
  __shared__ unsigned flag[kWV];  // bit dx + 3 dy: that shift stays in the grid
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int m = lane & 15, kb = lane >> 4;
  const int nci = Cin / (16 * CIB);
  const int co0 = ((int)blockIdx.y / nci) * (16 * COB), ci0 = ((int)blockIdx.y % nci) * (16 * CIB);
  const int vbeg = blockIdx.x * chunk, vend = min(d.V, vbeg + chunk);
  const int XY = d.X * d.Y;
  f32x4 acc[7][COB][CIB];
#pragma unroll
  for (int q = 0; q < 7; q++)
#pragma unroll
    for (int a = 0; a < COB; a++)
#pragma unroll
      for (int b = 0; b < CIB; b++) acc[q][a][b] = f32x4{0.f, 0.f, 0.f, 0.f};
  if (tid < XQ) sx[9 * kWR * XQ + tid] = u32x4{0u, 0u, 0u, 0u};
  const u32x4* xq = (const u32x4*)x + ci0 / 8;
  const u32x4* yq = (const u32x4*)dy + co0 / 8;
  // The next step's values, on their way to registers while this one's taps
  // are added.  Segment r = (dy+1) + 3 (dz+1): voxels v0 - 1 .. v0 + kWV
  // shifted by it.  Where the shift leaves the grid in y the row is some other
  // voxel's and not read; in z it is the periodic neighbour's (both are
  // V-periodic; a grid of few planes can leave the range even so)
  constexpr int NX = (9 * kWR * XQ + 255) / 256, NY = (kWV * YQ + 255) / 256;
  u32x4 bx[NX], by[NY];
  unsigned bf = 0;
  auto load = [&](int v0) {
#pragma unroll
    for (int u = 0; u < NX; u++) {
      const int e = min(tid + 256 * u, 9 * kWR * XQ - 1);
      const int r = e / (kWR * XQ), k = e - r * (kWR * XQ);
      int v = v0 - 1 + d.X * (r % 3 - 1) + XY * (r / 3 - 1) + k / XQ;
      v = v < 0 ? v + d.V : v;
      v = v >= d.V ? v - d.V : v;
      v = max(0, min(v, d.V - 1));
      bx[u] = xq[(size_t)v * (Cin / 8) + k % XQ];
    }
#pragma unroll
    for (int u = 0; u < NY; u++) {
      const int e = tid + 256 * u, v = v0 + e / YQ;
      by[u] = u32x4{0u, 0u, 0u, 0u};
      if (v < vend && e < kWV * YQ) by[u] = yq[(size_t)v * (Cout / 8) + e % YQ];
    }
    const int v = v0 + tid;
    bf = 0;
    if (v < vend) {
      int vx, vy, vz;
      coords(d, v, vx, vy, vz);
      const unsigned fx = (vx > 0 ? 1u : 0u) | 2u | (vx < d.X - 1 ? 4u : 0u);
      bf = (vy > 0 ? fx : 0u) | fx << 3 | (vy < d.Y - 1 ? fx << 6 : 0u);
    }
  };
  if (vbeg < vend) load(vbeg);
  for (int v0 = vbeg; v0 < vend; v0 += kWV) {
    __syncthreads();
#pragma unroll
    for (int u = 0; u < NX; u++)
      if (tid + 256 * u < 9 * kWR * XQ) sx[tid + 256 * u] = bx[u];
#pragma unroll
    for (int u = 0; u < NY; u++)
      if (tid + 256 * u < kWV * YQ) sy[tid + 256 * u] = by[u];
    if (tid < kWV) flag[tid] = bf;
    __syncthreads();
    if (v0 + kWV < vend) load(v0 + kWV);
    const uint16_t* lx = (const uint16_t*)sx;
    const uint16_t* ly = (const uint16_t*)sy;
    const int kr = 4 * kb + (m >> 2), col = (m & 3) * 4;  // this lane's row and part of it
#pragma unroll 1
    for (int b = 0; b < kWV / 32; b++) {
      const int k0 = 32 * b + kr, k1 = k0 + 16;
      const unsigned f0 = flag[k0], f1 = flag[k1];
      u32x4 a[COB];
#pragma unroll
      for (int q = 0; q < COB; q++) {
        const uint2 p0 = lds_read_tr(ly + k0 * (YQ * 8) + q * 16 + col);
        const uint2 p1 = lds_read_tr(ly + k1 * (YQ * 8) + q * 16 + col);
        a[q] = u32x4{p0.x, p0.y, p1.x, p1.y};
      }
#pragma unroll
      for (int q = 0; q < 7; q++) {
        const int t = 4 * q + wave;
        if (t < 27) {
          const int bit = t % 9, seg = t / 3;
          const int row = seg * kWR + t % 3;
          const int r0 = (f0 >> bit) & 1u ? row + k0 : 9 * kWR;
          const int r1 = (f1 >> bit) & 1u ? row + k1 : 9 * kWR;
#pragma unroll
          for (int c = 0; c < CIB; c++) {
            const uint2 p0 = lds_read_tr(lx + r0 * (XQ * 8) + c * 16 + col);
            const uint2 p1 = lds_read_tr(lx + r1 * (XQ * 8) + c * 16 + col);
            const u32x4 bb = {p0.x, p0.y, p1.x, p1.y};
#pragma unroll
            for (int o = 0; o < COB; o++) acc[q][o][c] = mfma32(a[o], bb, acc[q][o][c]);
          }
        }
      }
    }
  }
  // D[co = 4*kb+i][ci = m]
  float* out = part + (size_t)blockIdx.x * 27 * (size_t)Cout * Cin;
#pragma unroll
  for (int q = 0; q < 7; q++) {
    const int t = 4 * q + wave;
    if (t < 27)
#pragma unroll
      for (int o = 0; o < COB; o++)
#pragma unroll
        for (int c = 0; c < CIB; c++)
#pragma unroll
          for (int i = 0; i < 4; i++)
            out[((size_t)t * Cout + co0 + o * 16 + 4 * kb + i) * Cin + ci0 + c * 16 + m] =
                acc[q][o][c][i];
  }
}

// out[e] = sum over chunks (fixed order) of part[chunk][e]: 64 elements a
// block, 16 threads each (one would read the chunks one after the other: 38
// us for 381 of them).
__device__ __forceinline__ void reduce_chunks(int block, int nchunk, size_t n,
                                              const float* __restrict__ part,
                                              float* __restrict__ out, float (*sh)[64]) {
  const int l = threadIdx.x & 63, g = threadIdx.x >> 6;
  const size_t e = (size_t)block * 64 + l;
  float s = 0.f;
  if (e < n)
#pragma unroll 8
    for (int c = g; c < nchunk; c += 16) s += part[(size_t)c * n + e];
  sh[g][l] = s;
  __syncthreads();
  if (g == 0 && e < n) {
    float r = 0.f;
#pragma unroll
    for (int q = 0; q < 16; q++) r += sh[q][l];
    out[e] = r;
  }
}

__global__ void __launch_bounds__(1024)
    k_reduce_chunks(int nchunk, size_t n, const float* __restrict__ part,
                    float* __restrict__ out) {
  __shared__ float sh[16][64];
  reduce_chunks(blockIdx.x, nchunk, n, part, out, sh);
}

// ---------------------------------------------------------------------------
// 2x2x2 average pooling (children beyond the edge are skipped) and its
// backward; nearest upsampling and its backward (sum over children).
__device__ __forceinline__ int child_count(const Dims& f, int px, int py, int pz) {
  const int nx = min(2, f.X - 2 * px), ny = min(2, f.Y - 2 * py), nz = min(2, f.Z - 2 * pz);
  return nx * ny * nz;
}

// (one thread per voxel and 8 channels; 4 of the FP32 gradients)
__global__ void k_pool_fwd(Dims f, Dims c, int C, const uint16_t* __restrict__ x,
                           uint16_t* __restrict__ y) {
  const size_t e = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int Q = C / 8;
  if (e >= (size_t)c.V * Q) return;
  const int q = (int)(e % Q), v = (int)(e / Q);
  int px, py, pz;
  coords(c, v, px, py, pz);
  float s[8] = {};
  int n = 0;
  for (int dz = 0; dz < 2; dz++)
    for (int dy = 0; dy < 2; dy++)
      for (int dx = 0; dx < 2; dx++) {
        const int X = 2 * px + dx, Y = 2 * py + dy, Z = 2 * pz + dz;
        if (X < f.X && Y < f.Y && Z < f.Z) {
          const u32x4 w = ((const u32x4*)x)[((size_t)X + f.X * (Y + (size_t)f.Y * Z)) * Q + q];
#pragma unroll
          for (int i = 0; i < 4; i++) {
            s[2 * i] += lo2f(w[i]);
            s[2 * i + 1] += hi2f(w[i]);
          }
          n++;
        }
      }
  const float fn = (float)n;
  u32x4 o;
#pragma unroll
  for (int i = 0; i < 4; i++) o[i] = pack2(s[2 * i] / fn, s[2 * i + 1] / fn);
  ((u32x4*)y)[e] = o;
}

__global__ void k_up_fwd(Dims c, Dims f, int C, const uint16_t* __restrict__ x,
                         uint16_t* __restrict__ y) {
  const size_t e = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int Q = C / 8;
  if (e >= (size_t)f.V * Q) return;
  const int q = (int)(e % Q), v = (int)(e / Q);
  int X, Y, Z;
  coords(f, v, X, Y, Z);
  ((u32x4*)y)[e] =
      ((const u32x4*)x)[((size_t)(X / 2) + c.X * ((Y / 2) + (size_t)c.Y * (Z / 2))) * Q + q];
}

__global__ void k_up_bwd(Dims c, Dims f, int C, const float* __restrict__ dy,
                         float* __restrict__ dx) {
  const size_t e = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int Q = C / 4;
  if (e >= (size_t)c.V * Q) return;
  const int q = (int)(e % Q), v = (int)(e / Q);
  int px, py, pz;
  coords(c, v, px, py, pz);
  f32x4 s = {0.f, 0.f, 0.f, 0.f};
  for (int dz = 0; dz < 2; dz++)
    for (int dy_ = 0; dy_ < 2; dy_++)
      for (int dx_ = 0; dx_ < 2; dx_++) {
        const int X = 2 * px + dx_, Y = 2 * py + dy_, Z = 2 * pz + dz;
        if (X < f.X && Y < f.Y && Z < f.Z)
          s += ((const f32x4*)dy)[((size_t)X + f.X * (Y + (size_t)f.Y * Z)) * Q + q];
      }
  ((f32x4*)dx)[e] = s;
}

// What a convolution's backward pass starts from: the gradient of its output,
// g through the ReLU (post-activation y), g = ga (+ gp, the gradient of the
// average pooling that y feeds, spread over its children), as the BF16 operand
// of the two contractions, and the bias gradient's partial sums of the FP32
// values, bpart[block][C].  A thread keeps its 8 channels over all its voxels
// (C / 8 divides 256).
__global__ void __launch_bounds__(256)
    k_relu_bwd(Dims f, Dims c, int C, const uint16_t* __restrict__ y,
               const float* __restrict__ ga, const float* __restrict__ gp,
               uint16_t* __restrict__ dy, float* __restrict__ bpart) {
  __shared__ float sh[256][9];
  const int Q = C / 8, q = threadIdx.x % Q;
  float s[8] = {};
  const size_t n = (size_t)f.V * Q;
  for (size_t e = (size_t)blockIdx.x * 256 + threadIdx.x; e < n; e += (size_t)gridDim.x * 256) {
    f32x4 g0 = {0.f, 0.f, 0.f, 0.f}, g1 = g0;
    if (gp) {
      int X, Y, Z;
      coords(f, (int)(e / Q), X, Y, Z);
      const int px = X / 2, py = Y / 2, pz = Z / 2;
      const f32x4* p =
          (const f32x4*)(gp + ((size_t)px + c.X * (py + (size_t)c.Y * pz)) * C + 8 * q);
      const float k = (float)child_count(f, px, py, pz);
      g0 = p[0] / k;
      g1 = p[1] / k;
    }
    if (ga) {
      g0 += ((const f32x4*)ga)[2 * e];
      g1 += ((const f32x4*)ga)[2 * e + 1];
    }
    const u32x4 yv = ((const u32x4*)y)[e];
    float r[8];
#pragma unroll
    for (int i = 0; i < 8; i++) {
      const float a = i % 2 ? hi2f(yv[i / 2]) : lo2f(yv[i / 2]);
      r[i] = a > 0.f ? (i < 4 ? g0[i] : g1[i - 4]) : 0.f;
      s[i] += r[i];
    }
    ((u32x4*)dy)[e] = u32x4{pack2(r[0], r[1]), pack2(r[2], r[3]), pack2(r[4], r[5]),
                            pack2(r[6], r[7])};
  }
#pragma unroll
  for (int i = 0; i < 8; i++) sh[threadIdx.x][i] = s[i];
  __syncthreads();
  if ((int)threadIdx.x < C) {
    float t = 0.f;
    for (int r = threadIdx.x / 8; r < 256; r += Q) t += sh[r][threadIdx.x % 8];
    bpart[(size_t)blockIdx.x * C + threadIdx.x] = t;
  }
}

// sum of 256 values, one per thread, pairing those 128, 64, ... 1 apart; result
// in thread 0.  sh: 256 floats that no other sum since the last barrier used.
__device__ __forceinline__ float block_sum(float v, float* sh) {
  const int t = (int)threadIdx.x;
  sh[t] = v;
  __syncthreads();
  float s = 0.f;
  if (t < 64) {
    s = (sh[t] + sh[t + 128]) + (sh[t + 64] + sh[t + 192]);
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) s += __shfl_down(s, off);
  }
  return s;
}

// L = mean_v (out[v] - t[v])^2 (out FP32, the head's channel 0; its other 15
// channels have no gradient): part the loss's partial sums, one per 256
// consecutive voxels whatever the grid of blocks (k_loss_sums), bpart
// [block][16] those of the head's bias gradient, dy the gradient as BF16
// operand.  An FP64 target is divided by its scale here.
__global__ void __launch_bounds__(256)
    k_mse(int V, const float* __restrict__ out, const float* __restrict__ tgt,
          const double* __restrict__ tgt64, double tscale, uint16_t* __restrict__ dy,
          float* __restrict__ part, float* __restrict__ bpart) {
  __shared__ float sh[3][256];
  const int groups = (V + 255) / 256;
  float g = 0.f;
  int b = 0;
  for (int q = blockIdx.x; q < groups; q += gridDim.x, b ^= 1) {
    const int v = q * 256 + (int)threadIdx.x;
    float l = 0.f;
    if (v < V) {
      const float dlt = out[v] - (tgt64 ? (float)(tgt64[v] / tscale) : tgt[v]);
      const float gv = 2.f * dlt / (float)V;
      l = dlt * dlt;
      g += gv;
      u32x4* o = (u32x4*)(dy + (size_t)v * 16);
      o[0] = u32x4{(unsigned)f2bf(gv), 0u, 0u, 0u};
      o[1] = u32x4{0u, 0u, 0u, 0u};
    }
    const float ls = block_sum(l, sh[b]);
    if (threadIdx.x == 0) part[q] = ls;
  }
  const float gs = block_sum(g, sh[2]);
  if (threadIdx.x < 16) bpart[blockIdx.x * 16 + threadIdx.x] = threadIdx.x == 0 ? gs : 0.f;
}

// What follows k_mse.  Block 0: *loss = scale * (part[0] + part[1] + ... in this
// order).  The loss is this sum over its groups of 256 voxels, so its order
// belongs to the result (a tree over 1024 blocks' sums moved it by up to 2e-6
// of itself).  One lane adds, out of LDS, what all have loaded; the chain of
// additions bounds it: the 3050 groups of 51x91x181 take 141 us with one load
// after the other from memory, 15 us so.  Block 1: the head's bias gradient
// from its nb partial sums.
__global__ void __launch_bounds__(1024)
    k_loss_sums(int n, const float* __restrict__ part, float* __restrict__ loss, float scale,
                int nb, const float* __restrict__ bpart, float* __restrict__ gb) {
  constexpr int kC = 4096;
  __shared__ f32x4 sh[kC / 4];
  if (blockIdx.x == 1) {
    reduce_chunks(0, nb, 16, bpart, gb, (float(*)[64])sh);
    return;
  }
  float s = 0.f;
  for (int n0 = 0; n0 < n; n0 += kC) {
#pragma unroll
    for (int u = 0; u < kC; u += 1024) {
      const int i = n0 + u + (int)threadIdx.x;
      ((float*)sh)[u + threadIdx.x] = i < n ? part[i] : 0.f;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
      const int m = min(kC, n - n0), m4 = m / 4;
#pragma unroll 8
      for (int e = 0; e < m4; e++) {
        const f32x4 v = sh[e];
        s += v[0];
        s += v[1];
        s += v[2];
        s += v[3];
      }
      for (int e = 4 * m4; e < m; e++) s += ((const float*)sh)[e];
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) *loss = s * scale;
}

// Adam (bias-corrected) on FP32 weights; refreshes the BF16 copy when wb.
__global__ void k_adam(size_t n, float* __restrict__ w, const float* __restrict__ g,
                       float* __restrict__ m1, float* __restrict__ m2, float lr, float b1,
                       float b2, float eps, float c1, float c2, uint16_t* __restrict__ wb) {
  const size_t e = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= n) return;
  const float gg = g[e];
  const float a = b1 * m1[e] + (1.f - b1) * gg;
  const float b = b2 * m2[e] + (1.f - b2) * gg * gg;
  m1[e] = a;
  m2[e] = b;
  const float upd = lr * (a / c1) / (sqrtf(b / c2) + eps);
  const float wn = w[e] - upd;
  w[e] = wn;
  if (wb) wb[e] = f2bf(wn);
}

__global__ void k_to_bf16(size_t n, const float* __restrict__ x, uint16_t* __restrict__ y) {
  const size_t e = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (e < n) y[e] = f2bf(x[e]);
}

// Input features on the interior grid (a,b,c) from br0(nt,np) (Fortran
// order, interior at j+1,k+1) and a per-shell factor table:
//   ch0 = br0 * (r0/r)^2 / bscale,  ch1 = br0 / bscale,  ch2 = (r-r0)/(r1-r0)
__global__ void k_features(Dims d, int C, int nt, const double* __restrict__ br0,
                           const float* __restrict__ decay, const float* __restrict__ rpos,
                           float inv_bscale, int roll, int flip, uint16_t* __restrict__ x0) {
  const int v = blockIdx.x * blockDim.x + threadIdx.x;
  if (v >= d.V) return;
  int i, j, k;
  coords(d, v, i, j, k);
  // the sample seen rotated by `roll` interior phi points and, with flip,
  // reflected in theta (j -> Y-1-j); both 0 outside training
  const int js = flip ? d.Y - 1 - j : j;
  const int ks = k + roll < d.Z ? k + roll : k + roll - d.Z;
  const float b = (float)br0[(size_t)(js + 1) + (size_t)nt * (ks + 1)] * inv_bscale;
  u32x4* o = (u32x4*)(x0 + (size_t)v * C);
  o[0] = u32x4{pack2(b * decay[i], b), (unsigned)f2bf(rpos[i]), 0u, 0u};
  for (int c = 1; c < C / 8; c++) o[c] = u32x4{0u, 0u, 0u, 0u};
}

// Training target of a rotated/reflected sample: dst(i,j,k) = sign *
// src(i, flip ? Y-1-j : j, (k + roll) mod Z), the same map as k_features.
__global__ void k_gather_target(Dims d, int roll, int flip, float sign,
                                const float* __restrict__ src, float* __restrict__ dst) {
  const int v = blockIdx.x * blockDim.x + threadIdx.x;
  if (v >= d.V) return;
  int i, j, k;
  coords(d, v, i, j, k);
  const int js = flip ? d.Y - 1 - j : j;
  const int ks = k + roll < d.Z ? k + roll : k + roll - d.Z;
  dst[v] = sign * src[i + d.X * (js + d.Y * ks)];
}

// x (FP64, packed) = scale * out[v]
__global__ void k_head_to_x(int V, const float* __restrict__ out, double scale,
                            double* __restrict__ xo) {
  const int v = blockIdx.x * blockDim.x + threadIdx.x;
  if (v < V) xo[v] = scale * (double)out[v];
}

// Trilinear prolongation of a padded coarse field phi_c(nrc,ntc,npc) to the
// fine interior points: per-axis index/weight tables (fine interior -> lower
// coarse padded index and weight of the upper neighbour), phi periodic.
// One thread per point of a fine plane; its place in the plane by 32-bit
// arithmetic, the plane by the block (64-bit divisions of a flat index were
// most of the kernel: 128 us for 149x299x599 points, 98 us so).
__global__ void __launch_bounds__(256)
    k_prolong(int af, int bf, int cf, int nrc, int ntc, int npc,
                          const double* __restrict__ phic, const int* __restrict__ ir,
                          const double* __restrict__ wr, const int* __restrict__ it,
                          const double* __restrict__ wt, const int* __restrict__ ip,
                          const double* __restrict__ wp, double* __restrict__ xf) {
  const uint32_t q = blockIdx.x * 256u + threadIdx.x;
  if (q >= (uint32_t)af * (uint32_t)bf) return;
  const int j = (int)(q / (uint32_t)af), i = (int)(q - (uint32_t)j * (uint32_t)af);
  const double a1 = wr[i], b1 = wt[j];
  const size_t col = (size_t)ir[i] + (size_t)nrc * (size_t)it[j];
  const size_t plane = (size_t)nrc * ntc;
  for (int k = blockIdx.y; k < cf; k += gridDim.y) {
    const double c1 = wp[k];
    const double* p = phic + col + plane * (size_t)ip[k];
    double s = 0.0;
#pragma unroll
    for (int dk = 0; dk < 2; dk++)
#pragma unroll
      for (int dj = 0; dj < 2; dj++)
#pragma unroll
        for (int di = 0; di < 2; di++) {
          const double w = (di ? a1 : 1.0 - a1) * (dj ? b1 : 1.0 - b1) * (dk ? c1 : 1.0 - c1);
          s += w * p[(size_t)di + (size_t)nrc * dj + plane * dk];
        }
    xf[q + (size_t)af * bf * (size_t)k] = s;
  }
}

// D = A B for 16 x 16 matrices (A row-major MxK, B row-major KxN, BF16 bits; D
// FP32, row-major) as the convolutions and weight gradients form it: 16x16x32
// products, A's rows as they lie in memory, B through the transposing LDS read.
// Each half of the 32 k holds the product once, the other one zeros, so D is
// half their sum.
__global__ void __launch_bounds__(64)
    k_mfma_check(const uint16_t* __restrict__ A, const uint16_t* __restrict__ B,
                 float* __restrict__ D) {
  __shared__ u32x4 sb[32];
  const int l = threadIdx.x, m = l & 15, kb = l >> 4;
  if (l < 32) sb[l] = ((const u32x4*)B)[l];
  __syncthreads();
  const uint2 a = *(const uint2*)(A + m * 16 + 4 * kb);
  const uint2 b = lds_read_tr((const uint16_t*)sb + (4 * kb + (m >> 2)) * 16 + (m & 3) * 4);
  f32x4 acc = {0.f, 0.f, 0.f, 0.f};
  acc = mfma32(u32x4{a.x, a.y, 0u, 0u}, u32x4{b.x, b.y, 0u, 0u}, acc);
  acc = mfma32(u32x4{0u, 0u, a.x, a.y}, u32x4{0u, 0u, b.x, b.y}, acc);
#pragma unroll
  for (int i = 0; i < 4; i++) D[(4 * kb + i) * 16 + m] = 0.5f * acc[i];
}

// ---------------------------------------------------------------------------
// host launchers
static inline unsigned nblk(size_t n, int b) { return (unsigned)((n + b - 1) / b); }

template <int DIR, int CIN, int NB, int MT>
static void conv_launch(const Dims& d, int Cout, const uint16_t* x, const uint16_t* w,
                        const ConvOut& o, hipStream_t s) {
  const dim3 grid(nblk(d.V, 64 * MT), Cout / (16 * NB));
  if constexpr (CIN >= 32) {
    // three workgroups per CU, or the r axis is too long for whole rows
    const size_t lds = (size_t)(conv_lds_rows(MT, d.X) + 1) * CIN * 2;
    if (lds <= 52 * 1024) {
      k_conv_lds<CIN, NB, MT, DIR><<<grid, 256, lds, s>>>(d, Cout, x, w, o);
      return;
    }
  }
  k_conv<CIN, NB, MT, DIR><<<grid, 256, 0, s>>>(d, Cout, x, w, o);
}

template <int DIR, int CIN, int NB>
static void conv_mt(const Dims& d, int Cout, const uint16_t* x, const uint16_t* w,
                    const ConvOut& o, hipStream_t s) {
  // tiles per wave: as many as leave a few waves to every SIMD (1024 of them)
  if (d.V >= 200000)
    conv_launch<DIR, CIN, NB, 4>(d, Cout, x, w, o, s);
  else if (d.V >= 50000)
    conv_launch<DIR, CIN, NB, 2>(d, Cout, x, w, o, s);
  else
    conv_launch<DIR, CIN, NB, 1>(d, Cout, x, w, o, s);
}

template <int DIR, int CIN>
static void conv_nb(const Dims& d, int Cout, const uint16_t* x, const uint16_t* w,
                    const ConvOut& o, hipStream_t s) {
  if (Cout % 32 == 0 && d.V >= 10000)
    conv_mt<DIR, CIN, 2>(d, Cout, x, w, o, s);
  else
    conv_mt<DIR, CIN, 1>(d, Cout, x, w, o, s);
}

template <int DIR>
static void conv(const Dims3& d3, int Cin, int Cout, const uint16_t* x, const uint16_t* w,
                 const ConvOut& o, hipStream_t s) {
  const Dims d{d3.X, d3.Y, d3.Z, d3.X * d3.Y * d3.Z};
  if (Cin == 16)
    conv_nb<DIR, 16>(d, Cout, x, w, o, s);
  else if (Cin == 32)
    conv_nb<DIR, 32>(d, Cout, x, w, o, s);
  else if (Cin == 64)
    conv_nb<DIR, 64>(d, Cout, x, w, o, s);
  else
    conv_nb<DIR, 128>(d, Cout, x, w, o, s);
}

void conv_relu(const Dims3& d, int Cin, int Cout, const uint16_t* x, const uint16_t* w,
               const float* bias, uint16_t* y, const uint16_t* e, uint16_t* sum, hipStream_t s) {
  conv<1>(d, Cin, Cout, x, w, ConvOut{y, e, sum, nullptr, nullptr, bias, 1}, s);
}

void conv_head(const Dims3& d, int Cin, int Cout, const uint16_t* x, const uint16_t* w,
               const float* bias, float* y1, hipStream_t s) {
  conv<1>(d, Cin, Cout, x, w, ConvOut{nullptr, nullptr, nullptr, nullptr, y1, bias, 0}, s);
}

void transpose_weights(const ConvTable& ct, const uint16_t* w, uint16_t* wt, hipStream_t s) {
  size_t most = 0;
  for (int i = 0; i < ct.n; i++)
    most = std::max(most, (size_t)27 * ct.e[i].Cin * ct.e[i].Cout);
  k_transpose_weights<<<dim3(nblk(most, 256), ct.n), 256, 0, s>>>(ct, w, wt);
}

// Channel blocks of 16 per workgroup of the weight gradient (32 x 32 results
// per tap fill a wave's registers).
static int wgrad_block(int C) { return C % 32 == 0 ? 2 : 1; }

// Chunks of voxels of a weight gradient: workgroups for four per CU, of whole
// steps, and at most 32 MB of partial sums (they are written and read back).
int wgrad_chunks(const Dims3& d, int Cin, int Cout) {
  const long V = (long)d.V(), wv = wgrad_step(wgrad_block(Cin), wgrad_block(Cout));
  const long steps = (V + wv - 1) / wv;
  const long pairs = (long)(Cin / (16 * wgrad_block(Cin))) * (Cout / (16 * wgrad_block(Cout)));
  long n = std::min(steps, std::max(1L, 1024 / pairs));
  n = std::max(1L, std::min(n, (8L << 20) / (27L * Cin * Cout)));
  const long per = (steps + n - 1) / n;
  return (int)((steps + per - 1) / per);
}

void conv_bwd(const Dims3& d3, int Cin, int Cout, const uint16_t* dy, const uint16_t* x,
              const uint16_t* wt, float* dx, float* gw, float* part, hipStream_t s) {
  const Dims d{d3.X, d3.Y, d3.Z, d3.X * d3.Y * d3.Z};
  if (dx)
    conv<-1>(d3, Cout, Cin, dy, wt,
             ConvOut{nullptr, nullptr, nullptr, dx, nullptr, nullptr, 0}, s);
  const int nc = wgrad_chunks(d3, Cin, Cout);
  const int bi = wgrad_block(Cin), bo = wgrad_block(Cout), wv = wgrad_step(bi, bo);
  const int steps = (d.V + wv - 1) / wv, chunk = (steps + nc - 1) / nc * wv;
  const dim3 grid(nc, (Cin / (16 * bi)) * (Cout / (16 * bo)));
  if (bi == 1 && bo == 1)
    k_conv_bwd_weight<1, 1><<<grid, 256, 0, s>>>(d, Cin, Cout, chunk, dy, x, part);
  else if (bi == 1)
    k_conv_bwd_weight<1, 2><<<grid, 256, 0, s>>>(d, Cin, Cout, chunk, dy, x, part);
  else if (bo == 1)
    k_conv_bwd_weight<2, 1><<<grid, 256, 0, s>>>(d, Cin, Cout, chunk, dy, x, part);
  else
    k_conv_bwd_weight<2, 2><<<grid, 256, 0, s>>>(d, Cin, Cout, chunk, dy, x, part);
  const size_t nw = (size_t)27 * Cout * Cin;
  k_reduce_chunks<<<nblk(nw, 64), 1024, 0, s>>>(nc, nw, part, gw);
}

void pool_fwd(const Dims3& f3, const Dims3& c3, int C, const uint16_t* x, uint16_t* y,
              hipStream_t s) {
  Dims f{f3.X, f3.Y, f3.Z, f3.X * f3.Y * f3.Z}, c{c3.X, c3.Y, c3.Z, c3.X * c3.Y * c3.Z};
  k_pool_fwd<<<nblk((size_t)c.V * (C / 8), 256), 256, 0, s>>>(f, c, C, x, y);
}
void up_fwd(const Dims3& c3, const Dims3& f3, int C, const uint16_t* x, uint16_t* y,
            hipStream_t s) {
  Dims f{f3.X, f3.Y, f3.Z, f3.X * f3.Y * f3.Z}, c{c3.X, c3.Y, c3.Z, c3.X * c3.Y * c3.Z};
  k_up_fwd<<<nblk((size_t)f.V * (C / 8), 256), 256, 0, s>>>(c, f, C, x, y);
}
void up_bwd(const Dims3& c3, const Dims3& f3, int C, const float* dy, float* dx,
            hipStream_t s) {
  Dims f{f3.X, f3.Y, f3.Z, f3.X * f3.Y * f3.Z}, c{c3.X, c3.Y, c3.Z, c3.X * c3.Y * c3.Z};
  k_up_bwd<<<nblk((size_t)c.V * (C / 4), 256), 256, 0, s>>>(c, f, C, dy, dx);
}
// blocks of the kernels that leave partial sums (kSumBlocks at most)
static unsigned sum_blocks(size_t n) { return (unsigned)std::min<size_t>(nblk(n, 256), kSumBlocks); }

void relu_bwd(const Dims3& f3, const Dims3& c3, int C, const uint16_t* y, const float* ga,
              const float* gp, uint16_t* dy, float* bpart, float* gb, hipStream_t s) {
  const Dims f{f3.X, f3.Y, f3.Z, f3.X * f3.Y * f3.Z}, c{c3.X, c3.Y, c3.Z, c3.X * c3.Y * c3.Z};
  const unsigned nb = sum_blocks((size_t)f.V * (C / 8));
  k_relu_bwd<<<nb, 256, 0, s>>>(f, c, C, y, ga, gp, dy, bpart);
  k_reduce_chunks<<<nblk(C, 64), 1024, 0, s>>>((int)nb, (size_t)C, bpart, gb);
}
void mse(int V, const float* out, const float* tgt, const double* tgt64, double tscale,
         uint16_t* dy, float* part, float* bpart, float* loss, float* gb, hipStream_t s) {
  const unsigned nb = sum_blocks(V);
  k_mse<<<nb, 256, 0, s>>>(V, out, tgt, tgt64, tscale, dy, part, bpart);
  k_loss_sums<<<2, 1024, 0, s>>>((V + 255) / 256, part, loss, 1.0f / (float)V, (int)nb, bpart,
                                 gb);
}
void adam(size_t n, float* w, const float* g, float* m1, float* m2, float lr, float b1,
          float b2, float eps, int step, uint16_t* wb, hipStream_t s) {
  const float c1 = 1.f - powf(b1, (float)step), c2 = 1.f - powf(b2, (float)step);
  k_adam<<<nblk(n, 256), 256, 0, s>>>(n, w, g, m1, m2, lr, b1, b2, eps, c1, c2, wb);
}
void to_bf16(size_t n, const float* x, uint16_t* y, hipStream_t s) {
  k_to_bf16<<<nblk(n, 256), 256, 0, s>>>(n, x, y);
}
void features(const Dims3& d3, int C, int nt, const double* br0, const float* decay,
              const float* rpos, float inv_bscale, int roll, int flip, uint16_t* x0,
              hipStream_t s) {
  Dims d{d3.X, d3.Y, d3.Z, d3.X * d3.Y * d3.Z};
  k_features<<<nblk(d.V, 256), 256, 0, s>>>(d, C, nt, br0, decay, rpos, inv_bscale, roll, flip,
                                             x0);
}
void gather_target(const Dims3& d3, int roll, int flip, float sign, const float* src, float* dst,
                   hipStream_t s) {
  Dims d{d3.X, d3.Y, d3.Z, d3.X * d3.Y * d3.Z};
  k_gather_target<<<nblk(d.V, 256), 256, 0, s>>>(d, roll, flip, sign, src, dst);
}
void head_to_x(int V, const float* out, double scale, double* xo, hipStream_t s) {
  k_head_to_x<<<nblk(V, 256), 256, 0, s>>>(V, out, scale, xo);
}
void prolong(int af, int bf, int cf, int nrc, int ntc, int npc, const double* phic,
             const int* ir, const double* wr, const int* it, const double* wt, const int* ip,
             const double* wp, double* xf, hipStream_t s) {
  // four planes per thread, as long as that leaves enough blocks
  const unsigned gx = nblk((size_t)af * bf, 256);
  const unsigned gy = gx * (unsigned)cf >= 32768u ? (unsigned)(cf + 3) / 4 : (unsigned)cf;
  k_prolong<<<dim3(gx, std::min(gy, 65535u)), 256, 0, s>>>(af, bf, cf, nrc, ntc, npc, phic, ir, wr, it, wt, ip,
                                          wp, xf);
}
void mfma_check(const uint16_t* A, const uint16_t* B, float* D, hipStream_t s) {
  k_mfma_check<<<1, 64, 0, s>>>(A, B, D);
}

}  // namespace nn
}  // namespace p3d
