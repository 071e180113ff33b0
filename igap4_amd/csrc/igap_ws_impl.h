// igap_ws_impl.h -- internal state and launchers of the warm-start network.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace igap {
namespace ws {

constexpr int NL = 4;                  // convolution layers
constexpr int CH = 16;                 // channels between layers (and padded in/out)
constexpr int LAYER_W = 27 * CH * CH;  // weights of one layer
constexpr int LAYER_P = LAYER_W + CH;  // weights + bias
constexpr int CHUNK = 512;             // voxels per weight-gradient partial
// Weight-gradient partials of all layers together up to this size, so that one
// launch reduces them; beyond, one layer's at a time, each reduced before the
// next layer overwrites it: 7 GB in place of 28 on the largest grid a net accepts.
// Neither is faster (training step, upload included: 176^3, 1.18 GB of partials,
// 17.8 to 17.9 ms layer by layer, 18.0 to 18.5 all at once), so the line is where
// the memory begins to count, 0.4% of the device.
constexpr int64_t PART_ALL_BYTES = (int64_t)1 << 30;
constexpr float ADAM_B1 = 0.9f, ADAM_B2 = 0.999f, ADAM_EPS = 1e-8f;

struct Net {
    int nx = 0, ny = 0, nz = 0, cin = 0, cout = 0;
    int dil[NL] = {1, 1, 1, 1};
    int nchunk = 0;
    int part_layers = NL;               // layers whose weight-gradient partials are held at once: NL or 1
    int64_t step = 0;                   // Adam step count
    float *P = nullptr, *G = nullptr, *M = nullptr, *S = nullptr;   // FP32 params, grads, moments
    uint16_t *Wb = nullptr, *WTb = nullptr;                          // BF16 weight copies
    uint16_t *a[NL] = {};               // layer inputs (a[0] = packed input)
    uint16_t *dz[NL] = {};              // gradients w.r.t. each layer's pre-activation output
    float *y = nullptr, *tg = nullptr, *x = nullptr;
    float *part = nullptr, *bpart = nullptr, *lpart = nullptr;
    float *hG = nullptr;                // pinned host memory: gradients, then the loss sum (8-byte aligned)
    double *hloss = nullptr;
};

hipError_t conv_forward(const Net &n, int layer, const uint16_t *ain, uint16_t *aout, float *yout, hipStream_t s);
// the last layer, its loss partials and the gradient of its output in one launch
hipError_t conv_loss(const Net &n, const uint16_t *ain, const float *tg, uint16_t *dz, hipStream_t s);
// weight and bias partials of a layer and, with dzprev, its input gradient
hipError_t layer_back(const Net &n, int layer, const uint16_t *ain, const uint16_t *dz, uint16_t *dzprev, hipStream_t s);
// G of every layer and the sum of squared errors, after all layers; or, where the
// partials of one layer are held at a time, that layer's G (and with layer 0 the
// sum), after its layer_back.  hG (pinned) may be null
hipError_t grad_reduce(const Net &n, int layer, float *hG, double *hloss, hipStream_t s);
hipError_t pack_input(const Net &n, const float *x, uint16_t *a, hipStream_t s);
hipError_t pack_weights(const Net &n, hipStream_t s);
hipError_t adam(const Net &n, float lr, float c1, float c2, hipStream_t s);
hipError_t selftest_bf16(float *out, hipStream_t s);

}  // namespace ws
}  // namespace igap
