// Warm-start network: kernel launchers (p3d_nn_kernels.hip).
#pragma once
#include <hip/hip_runtime.h>
#include <stddef.h>
#include <stdint.h>

namespace p3d {
namespace nn {

struct Dims3 {
  int X, Y, Z;
  size_t V() const { return (size_t)X * Y * Z; }
};

// Zero bytes in front of every BF16 tensor that a convolution reads (one
// voxel's channels at most).
constexpr size_t kZeroFront = 256;

// y = relu(conv x + bias); with e also sum = y + e (the skip connection)
void conv_relu(const Dims3& d, int Cin, int Cout, const uint16_t* x, const uint16_t* w,
               const float* bias, uint16_t* y, const uint16_t* e, uint16_t* sum, hipStream_t s);
// y1[v] = channel 0 of conv x + bias (FP32)
void conv_head(const Dims3& d, int Cin, int Cout, const uint16_t* x, const uint16_t* w,
               const float* bias, float* y1, hipStream_t s);
// The convolutions of the parameter buffer.
struct ConvTable {
  struct Entry {
    int Cin, Cout;
    size_t w_off;
  } e[8];
  int n;
};
// wt: the BF16 weights for the gradients of the convolutions' inputs, placed
// as w
void transpose_weights(const ConvTable& ct, const uint16_t* w, uint16_t* wt, hipStream_t s);
// dx (FP32, may be null) and gw (27*Cout*Cin, FP32) from the BF16 gradient dy
// of the output (kZeroFront bytes before it); wt: transposed weights; part:
// scratch of wgrad_chunks*27*Cout*Cin floats
int wgrad_chunks(const Dims3& d, int Cin, int Cout);
void conv_bwd(const Dims3& d, int Cin, int Cout, const uint16_t* dy, const uint16_t* x,
              const uint16_t* wt, float* dx, float* gw, float* part, hipStream_t s);
void pool_fwd(const Dims3& f, const Dims3& c, int C, const uint16_t* x, uint16_t* y,
              hipStream_t s);
void up_fwd(const Dims3& c, const Dims3& f, int C, const uint16_t* x, uint16_t* y,
            hipStream_t s);
void up_bwd(const Dims3& c, const Dims3& f, int C, const float* dy, float* dx, hipStream_t s);
// Blocks, and so partial sums, of the two kernels below at most.
constexpr int kSumBlocks = 1024;
// dy (BF16) = (ga + pooling backward of gp) where y > 0; gb its sums by
// channel; ga or gp may be null; c: the pooled grid of f; bpart: kSumBlocks*C
void relu_bwd(const Dims3& f, const Dims3& c, int C, const uint16_t* y, const float* ga,
              const float* gp, uint16_t* dy, float* bpart, float* gb, hipStream_t s);
// loss = mean (out - t)^2, t = tgt or tgt64 / tscale, its BF16 gradient for the
// head's 16 channels and their bias gradient gb; part: one per 256 voxels,
// bpart: 16*kSumBlocks
void mse(int V, const float* out, const float* tgt, const double* tgt64, double tscale,
         uint16_t* dy, float* part, float* bpart, float* loss, float* gb, hipStream_t s);
void adam(size_t n, float* w, const float* g, float* m1, float* m2, float lr, float b1,
          float b2, float eps, int step, uint16_t* wb, hipStream_t s);
void to_bf16(size_t n, const float* x, uint16_t* y, hipStream_t s);
// roll/flip: the sample rotated by roll interior phi points and reflected in
// theta (training augmentation; 0, 0 otherwise)
void features(const Dims3& d, int C, int nt, const double* br0, const float* decay,
              const float* rpos, float inv_bscale, int roll, int flip, uint16_t* x0,
              hipStream_t s);
void gather_target(const Dims3& d, int roll, int flip, float sign, const float* src, float* dst,
                   hipStream_t s);
void head_to_x(int V, const float* out, double scale, double* xo, hipStream_t s);
void prolong(int af, int bf, int cf, int nrc, int ntc, int npc, const double* phic,
             const int* ir, const double* wr, const int* it, const double* wt, const int* ip,
             const double* wp, double* xf, hipStream_t s);
void mfma_check(const uint16_t* A, const uint16_t* B, float* D, hipStream_t s);

}  // namespace nn
}  // namespace p3d
