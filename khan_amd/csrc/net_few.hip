// The reference's default networks, 384-128-128-64-1 with CELU (khan/model/nn.py:38-68; sizes:
// khan/inference/energy_server.py:121), in float64 on few rows: values and row gradients in one launch.  Layer by layer
// (net_layers.hip, whose names these are) a request for one molecule's energy and gradient is seven launches of 4 to 12 us, each of
// which waits for a chain of loads and leaves the GPU empty: here a workgroup of sixteen wavefronts takes sixteen rows of one
// type through the whole network and back, its activations in LDS (the last layer's in registers).
//
// A product of the sixteen rows with 128 (or 64) columns: a wavefront has 32 columns and a quarter (an eighth) of the summed
// index, on v_mfma_f64_16x16x4_f64 with operands as in layer_kernel: the rows' from LDS, the weights' 16 bytes at a time from
// memory, four steps (eight loads) ahead, those of a product's first four steps before the sums of the product before it are
// added up.  The shares' sums meet in LDS and are added up in order.  The widths are constants of the code: with widths read at
// run time the index arithmetic between the products took as long as they did (with gradients 54 us, 27 now; seven launches
// were 28 us of kernels and as many of gaps).  With gradients three workgroups form the same values and a third of the 384
// gradient columns each, while that many find a compute unit of their own (launch_net_few).
#include "khan_internal.h"
#include "net_few.h"

namespace khan {

namespace {

typedef double v2d __attribute__((ext_vector_type(2)));
typedef double v4d __attribute__((ext_vector_type(4)));

constexpr int kThreads = 1024, kWaves = 16, kAhead = 4;
constexpr int kPad = 2;                       // doubles between rows: sixteen rows' pieces fall into different banks
constexpr int kIn = 384, kN1 = 128, kN2 = 128, kN3 = 64;

struct __align__(16) FewLds {
    double x[kFewRows][kIn + kPad];           // the rows; then the gradients, layer by layer
    double part[8 * kFewRows * (64 + kPad)];  // [share][row][column] of a product (four shares of 128 columns need no more)
    double a1[kFewRows][kN1 + kPad], a2[kFewRows][kN2 + kPad];
};
static_assert(4 * (128 + kPad) <= 8 * (64 + kPad), "the sums of four shares of 128 columns");
static_assert(sizeof(FewLds) <= 160 * 1024, "one workgroup per compute unit");

struct Lane {
    int l16, grp, wave;
};

// in . W for W [K, N] as stored or, kTrans, in . W^T for N columns of it (W [columns, K] as stored)
template <int K, int N, bool kTrans>
struct Product {
    static constexpr int kTiles = N / 32, kShares = kWaves / kTiles, kSteps = K / (8 * kShares), kLd = N + kPad;
    static_assert(N % 32 == 0 && kWaves % kTiles == 0 && K % (8 * kShares) == 0, "every wavefront has whole steps");
    static constexpr int kGroup = kSteps < kAhead ? kSteps : kAhead;
    static_assert(kSteps % kGroup == 0, "whole groups of steps");

    static __device__ __forceinline__ void fetch(const double* __restrict__ w, const Lane& L, int first, v2d (&b)[2 * kAhead])
    {
        const int tile = L.wave % kTiles, share = L.wave / kTiles;
        const int kk = (share * kSteps + first) * 8 + L.grp * 2, col = 32 * tile + 2 * L.l16;
        const double* at = kTrans ? w + col * K + kk : w + kk * N + col;
#pragma unroll
        for (int s = 0; s < kGroup; ++s)
#pragma unroll
            for (int e = 0; e < 2; ++e) b[2 * s + e] = *reinterpret_cast<const v2d*>(kTrans ? at + e * K + 8 * s : at + (8 * s + e) * N);
    }
    // in: [16][ld] in LDS; b: the first group's weights; ends with a barrier behind which the sums are complete
    static __device__ __forceinline__ void multiply(FewLds& S, const double* __restrict__ w, const Lane& L, const double* in, int ld, v2d (&b)[2 * kAhead])
    {
        const int tile = L.wave % kTiles, share = L.wave / kTiles;
        v4d acc[2] = {v4d(0.0), v4d(0.0)};
        const double* a_at = in + L.l16 * ld + share * kSteps * 8 + L.grp * 2;
#pragma unroll
        for (int first = 0; first < kSteps; first += kGroup) {
            v2d now[2 * kGroup];
#pragma unroll
            for (int i = 0; i < 2 * kGroup; ++i) now[i] = b[i];
            if (first + kGroup < kSteps) fetch(w, L, first + kGroup, b);
#pragma unroll
            for (int s = 0; s < kGroup; ++s) {
                const v2d a = *reinterpret_cast<const v2d*>(a_at + 8 * (first + s));
#pragma unroll
                for (int e = 0; e < 2; ++e)
#pragma unroll
                    for (int j = 0; j < 2; ++j)
                        acc[j] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[e], kTrans ? now[2 * s + j][e] : now[2 * s + e][j], acc[j], 0, 0, 0);
            }
        }
        double* out = S.part + share * kFewRows * kLd + 32 * tile + 2 * L.l16;
#pragma unroll
        for (int v = 0; v < 4; ++v) *reinterpret_cast<v2d*>(out + (L.grp + 4 * v) * kLd) = v2d{acc[0][v], acc[1][v]};
        __syncthreads();
    }
    // the results: thread i forms those of column i % N, rows i / N, i / N + 1024 / N, ...
    template <typename Use>
    static __device__ __forceinline__ void results(const FewLds& S, Use use)
    {
        const int c = threadIdx.x % N, r0 = threadIdx.x / N;
#pragma unroll
        for (int r = r0; r < kFewRows; r += kThreads / N) {
            const double* at = S.part + r * kLd + c;
            double sum = at[0];
#pragma unroll
            for (int s = 1; s < kShares; ++s) sum += at[s * kFewRows * kLd];
            use(r, c, sum);
        }
    }
};
typedef Product<kIn, kN1, false> First;
typedef Product<kN1, kN2, false> Second;
typedef Product<kN2, kN3, false> Third;
typedef Product<kN3, kN2, true> BackThird;
typedef Product<kN2, kN1, true> BackSecond;
typedef Product<kN1, 128, true> BackFirst;

__device__ __forceinline__ double few_slope(double a, double inv_alpha) { return a >= 0.0 ? 1.0 : fma(a, inv_alpha, 1.0); }

__global__ __launch_bounds__(kThreads) void net_few_kernel(const NetFew a, int log_parts)
{
    __shared__ FewLds S;
    const int tid = threadIdx.x, lane = tid & 63;
    const Lane L = {lane & 15, lane >> 4, __builtin_amdgcn_readfirstlane(tid >> 6)};
    // (log_parts: three workgroups out of each four take a third of the gradients' columns)
    const int part = log_parts ? static_cast<int>(blockIdx.x & 3u) : 0, tile = static_cast<int>(blockIdx.x) >> log_parts;
    if (part == 3) return;
    const int t = (tile >= a.tile_end[0]) + (tile >= a.tile_end[1]) + (tile >= a.tile_end[2]);
    const int row0 = (tile - (t == 0 ? 0 : a.tile_end[t - 1])) * kFewRows, n = a.n[t];
    const double* const w1 = a.w[0][t];
    const double* const w2 = a.w[1][t];
    const double* const w3 = a.w[2][t];
    const double* const w4 = a.w[3][t];
    double* const grad = a.grad[t];

    v2d b[2 * kAhead];
    First::fetch(w1, L, 0, b);
    // the rows (past the end: the last one again, never stored)
    constexpr int kPieces = kIn / 2;
#pragma unroll
    for (int i = 0; i < kFewRows * kPieces / kThreads; ++i) {
        const int at = tid + i * kThreads, r = at / kPieces, c = at % kPieces;
        *reinterpret_cast<v2d*>(&S.x[r][2 * c]) = *reinterpret_cast<const v2d*>(a.x[t] + static_cast<size_t>(min(row0 + r, n - 1)) * kIn + 2 * c);
    }
    const double bias1 = a.b[0][t][tid % kN1], bias2 = a.b[1][t][tid % kN2], bias3 = a.b[2][t][tid % kN3], top = w4[lane];
    auto celu = [&](double z) { return z >= 0.0 ? z : a.alpha * expm1(z * a.inv_alpha); };
    __syncthreads();
    // ---- forward
    First::multiply(S, w1, L, &S.x[0][0], kIn + kPad, b);
    Second::fetch(w2, L, 0, b);
    First::results(S, [&](int r, int c, double z) { S.a1[r][c] = celu(z + bias1); });
    __syncthreads();
    Second::multiply(S, w2, L, &S.a1[0][0], kN1 + kPad, b);
    Third::fetch(w3, L, 0, b);
    Second::results(S, [&](int r, int c, double z) { S.a2[r][c] = celu(z + bias2); });
    __syncthreads();
    Third::multiply(S, w3, L, &S.a2[0][0], kN2 + kPad, b);
    if (grad) BackThird::fetch(w3, L, 0, b);
    // a wavefront has one row of the 64 last activations (and the gradient by them): the output layer is a sum over its lanes
    static_assert(kN3 == 64, "a lane per activation");
    double* const g = &S.x[0][0];
    Third::results(S, [&](int r, int c, double z) {
        const double act = celu(z + bias3);
        double sum = act * top;
#pragma unroll
        for (int d = 32; d >= 1; d >>= 1) sum += __shfl_xor(sum, d, 64);
        if (c == 0 && part == 0 && row0 + r < n) a.value[t][row0 + r] = sum + *a.b[3][t];
        g[r * (kN3 + kPad) + c] = top * few_slope(act, a.inv_alpha);
    });
    if (!grad) return;
    __syncthreads();
    // ---- the way back: d_l = (d_{l+1} W^T) celu'
    BackThird::multiply(S, w3, L, g, kN3 + kPad, b);
    BackSecond::fetch(w2, L, 0, b);
    BackThird::results(S, [&](int r, int c, double d) { g[r * (kN2 + kPad) + c] = d * few_slope(S.a2[r][c], a.inv_alpha); });
    __syncthreads();
    BackSecond::multiply(S, w2, L, g, kN2 + kPad, b);
    BackFirst::fetch(w1 + part * 128 * kN1, L, 0, b);
    BackSecond::results(S, [&](int r, int c, double d) { g[r * (kN1 + kPad) + c] = d * few_slope(S.a1[r][c], a.inv_alpha); });
    __syncthreads();
    // ---- and to the rows, 128 columns at a time
    const int last = log_parts ? part : kIn / 128 - 1;
    for (int ct = part; ct <= last; ++ct) {
        BackFirst::multiply(S, w1 + ct * 128 * kN1, L, g, kN1 + kPad, b);
        if (ct < last) BackFirst::fetch(w1 + (ct + 1) * 128 * kN1, L, 0, b);
        BackFirst::results(S, [&](int r, int c, double d) {
            if (row0 + r < n) grad[static_cast<size_t>(row0 + r) * kIn + ct * 128 + c] = d;
        });
        __syncthreads();                                       // the sums have been read
    }
}

}  // namespace

bool net_few_fits(const int* k, int layers)
{
    return layers == 4 && k[0] == kIn && k[1] == kN1 && k[2] == kN2 && k[3] == kN3 && k[4] == 1;
}

hipError_t launch_net_few(NetFew a, hipStream_t stream)
{
    int tiles = 0;
    bool grad = false;
    for (int t = 0; t < 4; ++t) {
        a.tile_end[t] = tiles += (a.n[t] + kFewRows - 1) / kFewRows;
        grad = grad || a.grad[t];
    }
    if (tiles == 0) return hipSuccess;
    const int log_parts = grad && tiles * 3 <= kCUs ? 2 : 0;
    net_few_kernel<<<dim3(static_cast<unsigned>(tiles) << log_parts), dim3(kThreads), 0, stream>>>(a, log_parts);
    return hipGetLastError();
}

}  // namespace khan
