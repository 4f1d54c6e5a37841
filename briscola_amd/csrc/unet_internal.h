// Internal declarations of the learned preconditioner (3-D U-Net, BF16 on
// the gfx950 matrix cores).
#pragma once

#include <hip/hip_runtime.h>
#include <stdexcept>
#include <string>

struct bmg_unet;

namespace bmg {
namespace unet {

typedef __bf16 bf16;

struct UnetError : std::runtime_error
{
    using std::runtime_error::runtime_error;
};

struct Grid3 {
    int D, H, W;   // z, y, x extents; voxel m = (z*H + y)*W + x
};

// One convolution y = act(conv(x, w) + bias) on channel slices.
struct ConvArgs {
    Grid3 g;
    const bf16* x;    // input slice, row stride ldx, cin channels (cin % 8 == 0)
    int ldx;
    int cin;
    const bf16* w;    // [cout][kp], k = t*cin + c, zero beyond taps*cin
    int kp;           // taps*cin rounded up to 32
    int taps;         // 27 (3x3x3) or 1 (1x1x1)
    int cout;         // a multiple of 16 up to 192
    const float* bias;  // cout values or null
    int relu;
    bf16* y;          // output slice, row stride ldy
    int ldy;
};

// One convolution of the inference pass (with bias and ReLU): the first c0
// input channels from a tensor of half the extents through nearest-neighbour
// upsampling, the others from x; also the 2x2x2 averages of the output
// (pool set) or, instead of it, the output projection (head set).
struct TileConvArgs {
    Grid3 g;
    const bf16* up;    // coarse tensor (extents g/2), c0 channels; or null
    int ldu, c0;
    const bf16* x;     // fine tensor, the remaining channels
    int ldx;
    int cin;
    const bf16* w;     // [cout][kp], k = t*cin + c
    int kp, cout;
    const float* bias;
    bf16* y;
    int ldy;
    bf16* pool;        // POOL: coarse output, row stride ldp
    int ldp;
    const float* head; // HEAD: 16 weights and the bias
    float* out;
};

// dw[n][k] += sum_m dz[m][n] * x[tap_k(m)][c_k] (FP32 accumulation).
struct WgradArgs {
    Grid3 g;
    const bf16* x;
    int ldx;
    int cin;
    const bf16* dz;
    int lddz;
    int cout;
    int taps;
    int kp;
    float* dw;
    int chunk = 0;    // voxels per workgroup of the general kernel
};

inline int round32(int k) { return (k + 31)/32*32; }

void conv_fwd(const ConvArgs& a, hipStream_t s);
// nt, mt: tiles of 16 output channels and rows of a wavefront (0: by size).
void conv_rows(const TileConvArgs& a, hipStream_t s, int nt = 0, int mt = 0);
// The first convolution (2 real input channels, BF16 of f and c; w as E0's
// [16][kp]) with bias and ReLU, and its averages.
void conv_first(const Grid3& g, const float* f, const float* c, const bf16* w,
                int kp, const float* bias, bf16* y, int ldy, bf16* pool,
                int ldp, hipStream_t s);
// Floats of workspace the tiled weight gradient of these arguments needs (0:
// the general kernel takes them, without workspace).
size_t wgrad_workspace(const WgradArgs& a);
// dbias (tiled kernel only): cout column sums of dz, added at the end of dw's
// cout*kp weights.
void conv_wgrad(const WgradArgs& a, float* workspace, float* dbias,
                hipStream_t s);
// weights of the data gradient: wt[c][t'*cout + n] = w[n][(26-t')*cin + c]
void flip_weights(const bf16* w, int cin, int cout, int kp, int taps, bf16* wt,
                  int kpt, hipStream_t s);
void pool(const bf16* x, int ldx, Grid3 fine, int C, bf16* y, int ldy,
          hipStream_t s);
// dx = (dx + dy/8 of the parent) where y > 0 (C, strides and bases multiples
// of 8 channels, likewise up_relu_bwd)
void pool_relu_bwd(const bf16* dy, int lddy, Grid3 fine, int C, const bf16* y,
                   int ldy, bf16* dx, int lddx, hipStream_t s);
void up(const bf16* x, int ldx, Grid3 fine, int C, bf16* y, int ldy,
        hipStream_t s);
// dx = the sum of the eight children's dy where y > 0
void up_relu_bwd(const bf16* dy, int lddy, Grid3 fine, int C, const bf16* y,
                 int ldy, bf16* dx, int lddx, hipStream_t s);
// w[0..15] weights, w[16] bias
void head_fwd(const bf16* x, int ldx, int M, const float* w, float* out,
              hipStream_t s);
int head_bwd(const bf16* x, int ldx, int M, const float* w, const float* gout,
             bf16* dx, int lddx, float* partial, hipStream_t s);
int mse(const float* p, const float* t, int M, const float* shift, float* g,
        float* partial, hipStream_t s);
int diff_sum(const float* a, const float* b, int M, float* partial,
             hipStream_t s);
void col_sum(const float* in, int rows, int cols, float scale, float* out,
             hipStream_t s);
// The BF16 copies of a layer's weights: parameters [off, off + cout*kp).
struct WeightView {
    int off, cin, cout, kp, kpt;
    bf16* w;
    bf16* wt;    // flipped, for the data gradient; null: none
};
struct WeightViews {
    enum { LAYERS = 7 };
    WeightView l[LAYERS];
};
void adam(const WeightViews& views, float* w, float* m, float* v,
          const float* g, int n, float lr, float b1, float b2, float eps,
          int step, hipStream_t s);
void refresh_weights(const WeightViews& views, const float* w, int n,
                     hipStream_t s);
void pack_input(const float* f, const float* lam, int M, bf16* x,
                hipStream_t s);

// Solver-facing calls on a network (bmg_unet of bmg_unet.h): allocate the
// activations of a grid (not allowed during graph capture), and run the
// forward pass on a given stream (capturable once prepared).  net_prepare
// returns the buffers' generation: a capture made at another one refers to
// freed memory.
long net_prepare(struct ::bmg_unet* net, int D, int H, int W);
void net_forward(struct ::bmg_unet* net, int D, int H, int W, const float* f,
                 const float* c, float* out, hipStream_t s);

}  // namespace unet
}  // namespace bmg
