// hf_cnn.h -- structures and launchers of the learned coarse-grid correction
// (a 5-layer 3x3 CNN on BF16 MFMA with FP32 accumulation).
//
// Activations are NHWC BF16 images with a one-pixel zero border:
// [(ny+2)][(nx+2)][C], C = 8 (the 4 conserved variables, zero padded) or 32.
// The border is zeroed once at allocation and never written, so every 3x3
// tap reads in bounds and "same" zero padding needs no branches.
//
// A convolution is an implicit GEMM per 16-pixel row segment:
//   out[o][p] = sum_k W^T[o][k] * patch[k][p],  k = (tap, input channel),
// run as v_mfma_f32_16x16x32_bf16 with the weights as the A operand (rows =
// output channels, preloaded in registers in the order the lanes consume
// them) and the input patch as the B operand (one 16-byte load of 8
// channels per lane).  The weight gradient is the same product with the
// pixels as the reduction dimension, staged through LDS in channel-major
// order.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace hfn {

enum { NET_OUT_PLANES = 0, NET_APPLY = 1 };

// The forward pass.
struct NetArgs {
    const uint16_t* x;        // packed input, NHWC BF16, padded, 8 channels
    const uint16_t* w[5];     // A operands of each layer [MT][S][64 lanes][8]
    const float* bias[5];
    int32_t nx, ny, rows;     // interior size; rows per workgroup (set by launch_net)
    uint16_t* act[4];         // hidden activations, NHWC BF16, padded (null: not stored)
    float* outf;              // NET_OUT_PLANES: dense planes [4][ny][nx]
    float* U;                 // NET_APPLY: state planes (interior origin), corrected in place
    int64_t plane;            // elements per plane of U
    int32_t pitch;            // row pitch of U
    float gamma;              // ideal-gas gamma for the pressure check
    float scale[4];           // correction = scale * network output
    float max_output;         // fall back where |output| > max_output (<= 0: no bound)
    const uint8_t* shock;     // per-cell shock flag [ny][nx] (null: none)
    uint32_t* fallback;       // cells left at the plain state
};

// The data gradient of one layer.
struct ConvArgs {
    const uint16_t* in;       // gradient at the layer's output, NHWC BF16, padded, CIN channels
    const uint16_t* wa;       // A operands [2][S][64 lanes][8]
    int32_t nx, ny, rows;     // interior size; rows per wave
    uint16_t* out;            // NHWC BF16, padded, 32 channels
    const uint16_t* mask;     // activation whose positive entries pass the gradient
};

// One layer's weight-gradient partials and where their sum goes.
struct ReduceLayer {
    const float* part;
    float* grads;
    int32_t nparts, ci, co, ci_r, co_r, first;   // first: set by launch_reduce_grad
};
constexpr int MAX_LAYERS = 5;

// The weight gradients of all layers.
struct WgradLayer {
    const uint16_t* a;      // layer input activation, NHWC padded, ci channels
    const uint16_t* gz;     // gradient at the layer's pre-activation, NHWC padded, co channels
    float* part;            // [workgroups][9*ci*co + co] partial sums
    int32_t ci, co;         // storage channels: (8, 32), (32, 32) or (32, 8)
};
struct WgradArgs {
    WgradLayer layer[MAX_LAYERS];
    int32_t nlayers, nx, ny;
    int32_t rows, nwg;      // rows and workgroups per layer, set by launch_wgrad
};

struct ReduceArgs {
    ReduceLayer layer[MAX_LAYERS];
    int32_t nlayers;
    int32_t nloss;
    const float* lossp;     // [nloss] partial sums of the loss
    float loss_scale;
    float* loss;            // their sum times loss_scale
};

// Input normalisation + optional shock sensor.  U: planes of the conserved
// variables with the interior origin at U, element (v, y, x) at
// U[v*plane + y*pitch + x].
struct PackArgs {
    const float* U;
    int64_t plane;
    int32_t pitch, nx, ny;
    float mean[4], iscale[4];
    uint16_t* X;            // NHWC BF16, padded, 8 channels
    uint8_t* shock;         // null: no sensor
    float gamma, theta;
};

struct LossArgs {
    const float* Y;         // network output, dense planes [4][ny][nx]
    const float* Uc;        // plain coarse state, dense planes
    const float* T;         // target state (restricted fine solution), dense planes
    float inv_scale[4];     // target residual = (T - Uc) * inv_scale
    float gscale;           // d loss / d y = gscale * 2 (y - t)
    int32_t nx, ny;
    uint16_t* G;            // NHWC BF16, padded, 8 channels
    float* part;            // [blocks] partial sums of squared errors
};

// Launchers (hf_cnn.hip).  cin/cout are storage channel counts (8 or 32).
hipError_t launch_net(NetArgs a, int mode, hipStream_t s);
hipError_t launch_conv_bwd(int cin, const ConvArgs& a, hipStream_t s);
hipError_t launch_wgrad(WgradArgs a, hipStream_t s);
int wgrad_workgroups(int nx, int ny);   // per layer
hipError_t launch_pack(const PackArgs& a, hipStream_t s);
hipError_t launch_loss(const LossArgs& a, int* nblocks, hipStream_t s);
hipError_t launch_reduce_grad(ReduceArgs a, hipStream_t s);
hipError_t launch_adam(float* w, const float* g, float* m, float* v, int n, float lr, float b1, float b2, float eps,
                       float c1, float c2, hipStream_t s);
// Packs the FP32 layer weights W[9][ci_r][co_r] into the A-operand order of
// a convolution with cin -> cout storage channels; transposed = 1 packs the
// data-gradient convolution (taps flipped, channels swapped).
hipError_t launch_pack_weights(int cin, int cout, const float* W, int ci_r, int co_r, int transposed, uint16_t* wa,
                               hipStream_t s);
int packed_weight_elems(int cin, int cout);
hipError_t launch_state_copy(const float* src, int64_t splane, int spitch, float* dst, int64_t dplane, int dpitch,
                             int nx, int ny, hipStream_t s);
hipError_t launch_restrict2(const float* U, int64_t plane, int pitch, int nxc, int nyc, float* dst, hipStream_t s);

}  // namespace hfn
