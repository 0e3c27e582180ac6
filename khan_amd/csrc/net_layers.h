// Launch interface of net_layers.hip: the per-type networks layer by layer, forward, gradient, second order and weight
// gradients (the mathematics and its names are described there).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace khan {

constexpr int kNetMaxLayers = 12;        // products of a network, the output layer included

// What a product's epilogue makes of y = in . W (+ bias):
enum NetKind {
    kNetCelu = 0,        // celu(y)
    kNetSlope = 1,       // y celu'(act)
    kNetRows = 2,        // y scale[row] (scale null: 1), added to out with `accumulate`
    kNetTangent = 3,     // y' = y scale[row]: out = y' celu'(act), out2 = act < 0 ? y' d / alpha : 0
    kNetSecond = 4,      // y celu'(act) + scale[row] t
};

template <typename T>
struct NetLayer {
    const T *in[4], *w[4], *bias[4];
    const T *act[4], *d[4], *t[4], *scale[4];
    T *out[4], *out2[4];
    int n[4];                       // rows per type
    int k, n_out;
    int kind, accumulate;
    bool absolute;                  // kNetCelu: an error of 2^-24 alpha is small enough, that of small activations may be larger
    T alpha, inv_alpha;
    int tile_end[4], col_tiles;     // filled by the launcher
};

// the output layer: value = act . w + bias and out = w celu'(act) (either null); or `second`: out = scale[row] t
template <typename T>
struct NetTop {
    const T *act[4], *w[4], *bias[4], *t[4], *scale[4];
    T *value[4], *out[4];
    int n[4];
    int k, second;
    T inv_alpha;
    int row_end[4];                 // filled by the launcher
};

// Gradients of all weights and biases, written to `out`: for every layer the four types' [k, n_out], then for every layer
// the four types' biases.  left[l] (l >= 1) and right[l] are [rows of all types, width] arrays, type t from row row0[t] on;
// layer 0's left operand are the four arrays x.  `first` has a bit for every layer with left^T right, `second` for every
// layer with left2^T right2 (added to it).  A null right: ones.  scale_first, scale_second: the rows of the right operands
// are multiplied by scale.
template <typename T>
struct NetGrads {
    const T *x[4], *x2[4];
    const T *left[kNetMaxLayers], *right[kNetMaxLayers], *left2[kNetMaxLayers], *right2[kNetMaxLayers];
    const T* scale[4];
    bool scale_first, scale_second;
    unsigned first, second;
    int n[4];
    int64_t row0[4];
    int layers;
    int k[kNetMaxLayers + 1];       // widths: layer l is [k[l], k[l + 1]]
    T* out;
    // filled by the launcher: rows per workgroup, the workgroups' numbering by layer and type and where their partial sums
    // begin; the layers whose operands may be read 16 bytes at a time, and those on split products (with their own rows per
    // workgroup)
    int per, per_split, job_end[4 * kNetMaxLayers];
    int64_t job_base[4 * kNetMaxLayers];
    unsigned whole, split;
};

template <typename T> hipError_t launch_net_layer(NetLayer<T> a, bool trans, hipStream_t stream);
template <typename T> hipError_t launch_net_top(NetTop<T> a, hipStream_t stream);
template <typename T> size_t net_grads_workspace(NetGrads<T> a);          // bytes; from n, layers and k
template <typename T> hipError_t launch_net_grads(NetGrads<T> a, void* workspace, hipStream_t stream);

}  // namespace khan
