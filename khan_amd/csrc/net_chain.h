// Launch interface of net_chain.hip: float32 networks of any depth, all layers of a pass in one launch, for inference.
#pragma once
#include <hip/hip_runtime.h>
#include <stddef.h>
#include <stdint.h>

#include "net_layers.h"

namespace khan {

constexpr int kChainWidth = 256;         // widest hidden layer
constexpr int kChainPiece = 128;         // the feature width is a multiple of this

// A network of `hidden` CELU layers widths[0] -> ... -> widths[hidden] and the output layer to one value, for the four types
struct NetChain {
    const float *x[4];                           // [n_t, widths[0]]
    const float *w[kNetMaxLayers][4];            // [widths[l], widths[l + 1]]
    const float *b[kNetMaxLayers][4];
    int n[4], hidden, widths[kNetMaxLayers + 1];
    unsigned absolute;                           // a bit per layer: exp(z) - 1 in its CELU as it is (NetLayer)
    float alpha;
    bool want_rows;                              // row gradients will be asked for
};

bool net_chain_fits(const int* widths, int hidden);
// Workspace: the weights split and packed, and with want_rows the activations.
size_t net_chain_workspace(const NetChain& net);
// packs the weights into the workspace, then the values
hipError_t launch_net_chain_values(const NetChain& net, void* workspace, float* const value[4], hipStream_t stream);
// from the workspace that launch_net_chain_values left (of the same net): scale_r d value_r / d x_r (scale null: ones), added to what
// grad holds with `accumulate`
hipError_t launch_net_chain_rows(const NetChain& net, const void* workspace, const float* const scale[4], float* const grad[4], bool accumulate,
                                 hipStream_t stream);

}  // namespace khan
