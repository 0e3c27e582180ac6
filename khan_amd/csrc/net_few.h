// Launch interface of net_few.hip: the default networks in float64 on few rows in one launch.
#pragma once
#include <hip/hip_runtime.h>

namespace khan {

constexpr int kFewRows = 16;         // rows per workgroup
constexpr int kFewLayers = 4;        // products of a network, the output layer included

struct NetFew {
    const double *x[4], *w[kFewLayers][4], *b[kFewLayers][4];
    double *value[4], *grad[4];      // grad null: values only
    int n[4];
    double alpha, inv_alpha;
    int tile_end[4];                 // filled by the launcher
};

bool net_few_fits(const int* widths, int layers);
hipError_t launch_net_few(NetFew a, hipStream_t stream);

}  // namespace khan
