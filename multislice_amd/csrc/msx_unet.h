// msx_unet.h -- internal interface of the surrogate network's GPU kernels.
#pragma once
#include <hip/hip_runtime.h>

namespace msx {
namespace unet {

enum ConvMode { kFwd = 0, kBwdData = 1, kBwdWeight = 2 };

// One convolution layer, stride 1, zero padding KS/2, NCHW FP32 tensors.
//  kFwd      : out[n, out_c0 + co] (+)= relu?(conv(x, w) + bias)
//  kBwdData  : out[n, out_c0 + ci] (+)= conv^T(G, w)
//  kBwdWeight: out[co, ci, tap]    +=  sum_{n,p} G[n, co, p] x[n, ci, p + off(tap)]
// G = g masked by (y > 0) when relu is set (y = the layer's forward output).
struct ConvArgs {
    const float* x;     // [N, Cin, H, W]   (kFwd, kBwdWeight)
    const float* w;     // [Cout, Cin, KS*KS]
    const float* bias;  // [Cout] or null   (kFwd)
    const float* g;     // [N, Cout, H, W]  (kBwdData, kBwdWeight)
    const float* y;     // [N, Cout, H, W]  ReLU mask source (backward with relu)
    float* out;
    int N, Cin, Cout, H, W;
    int relu;
    int out_c, out_c0;  // channel count and offset of the destination tensor
    int accumulate;
    // kBwdWeight split over several slices of its reduction: per-slice
    // partial weight gradients [splits][Cout][Cin * KS * KS], summed in a
    // fixed order into out (conv_wgrad_scratch floats; unused otherwise)
    float* partial;
    float* db;  // kBwdWeight: bias gradient [Cout], or null
    // kFwd, kBwdData of 3x3 layers: the layer's weights packed for that mode
    // (launch_pack_conv3), or null: the general kernel
    const __bf16* pack;
    // kFwd with pack: further copies of the output, each optional: its 2x2
    // average [N, Cout, H/2, W/2] (H, W even), itself as channels skip_c0 ..
    // of a tensor with skip_c channels, and its nearest x2 upsampling as the
    // first channels of a [N, up_c, 2H, 2W] tensor
    float *pool, *skip, *up;
    int skip_c, skip_c0, up_c;
    // kFwd without pack: out = mean over res_c channels of res [N, res_c, H, W]
    // + the convolution (one output channel), or null
    const float* res;
    int res_c;
};

// Packing of 3x3 weights into conv3's fragment order, several layers (and
// modes) per launch.  M output rows and C reduction channels: (Cout, Cin) for
// kFwd, (Cin, Cout) for kBwdData; offsets in elements from w and out.
constexpr int kMaxPack = 48;
struct PackLayer {
    int mode, M, C;
    long long w_off, out_off;
};
struct PackArgs {
    const float* w;
    __bf16* out;
    PackLayer layer[kMaxPack];
};
size_t conv3_pack_size(int M, int C);  // elements of one layer's packed weights
bool conv3_fits(const ConvArgs& a);    // image small enough for the packed kernel
hipError_t launch_pack_conv3(const PackArgs& a, int layers, hipStream_t s);

hipError_t launch_conv(int mode, int ks, const ConvArgs& a, hipStream_t s);  // kFwd, kBwdData

// kBwdWeight of several layers at once: the products, one launch for all 3x3
// layers that wgrad3 takes and one for each other, then one launch that adds
// their slices and forms the bias gradients.
constexpr int kMaxWgrad = 24;
struct WgradLayer {
    ConvArgs a;
    int ks;
};
// floats of ConvArgs::partial that a layer needs (0: none)
size_t conv_wgrad_scratch(int ks, const ConvArgs& a);
hipError_t launch_wgrad(const WgradLayer* layers, int n, hipStream_t s);  // n <= kMaxWgrad
hipError_t launch_avgpool_fwd(const float* x, float* y, long long nc, int H, int W, hipStream_t s);
hipError_t launch_avgpool_bwd(const float* gy, float* gx, long long nc, int H, int W, hipStream_t s);
hipError_t launch_upsample_fwd(const float* x, float* y, int N, int C, int H, int W, int Ct, int c0, hipStream_t s);
hipError_t launch_cat_bwd(const float* g, float* gup, int C1, float* gskip, int C2, int N, int H, int W,
                          hipStream_t s);
hipError_t launch_copy_channels(const float* src, int Cs, int s0, float* dst, int Cd, int d0, int N, int C, int HW,
                                hipStream_t s);
// y[n][p] = (1/C) sum_c x[n][c][p] (FP32, channels in order)
hipError_t launch_channel_mean(const float* x, float* y, int N, int C, long long HW, hipStream_t s);
hipError_t launch_residual_loss(const float* in, const float* z, const float* t, float* g, long long n, float scale,
                                double* partial, int nblocks, hipStream_t s);
// zeros in a and b (b 16-byte aligned, nb a multiple of 4)
hipError_t launch_clear(float* a, long long na, float* b, long long nb, hipStream_t s);
hipError_t launch_adam(float* w, const float* gw, float* m, float* v, long long n, float lr, float b1, float b2,
                       float eps, float c1, float c2, hipStream_t s);

}  // namespace unet
}  // namespace msx
