// The per-type atomic networks of any widths with CELU (khan/model/nn.py:38-68, activations.py:63-65), float32 and float64,
// layer by layer: the products of the forward pass, of the gradient, of a loss on the gradient (second order), and of the
// weights' gradients, for the four atom types in one launch each.
//
// With z_l = a_{l-1} W_l + b_l, a_l = celu(z_l), value = a_L w + b (L hidden layers, a_0 = the feature row x):
//     d_l    = d value / d z_l,  d_L = w celu'(z_L),  d_{l-1} = (d_l W_l^T) celu'(z_{l-1}),  d value / d x = d_1 W_1^T
//     tangent along x' :  z'_l = a'_{l-1} W_l,  a'_l = celu'(z_l) z'_l
//     q_l    = d phi / d z_l of phi = sum_r s_r (tangent of value_r), whose gradient a loss on d value / d x needs:
//              q_L = s t_L,  q_{l-1} = (q_l W_l^T) celu'(z_{l-1}) + s t_{l-1},  t_l = celu''(z_l) z'_l (d value / d a_l)
//     dW_l   = a_{l-1}^T q_l + a'_{l-1}^T (s d_l),   db_l = sum of q_l over the rows
// and for phi = sum_r s_r value_r, plain training, dW_l = a_{l-1}^T (s d_l).  celu' and celu'' come from the activation: 1
// and 0 for a >= 0, a / alpha + 1 and that over alpha below; t_l = z'_l d_l / alpha for a_l < 0.  What a product needs of
// these is formed in its epilogue, so that every operand of the next one is read as it lies in memory.
//
// These replace library products (rocBLAS, one per type, with elementwise passes between them) in training, in force
// training, for networks the one-launch kernel (dense_fused.hip) is not made for or may not take (float64, charge networks): a
// step on 1,024 organic molecules was 95 launches, one with a loss on forces 430, an energy request 330.  Measured with what
// goes with it (no graph in inference, csrc/torch_autograd.cpp), us a pass, library products -> here: a request for an energy
// and a gradient in float64 4,000 -> 210; training, float32 default networks, 1,024 / 16,384 / 65,536 organic molecules
// 1,840 -> 480, 4,870 -> 1,120, 16,200 -> 3,630, deep networks on 1,024 / 16,384 6,450 -> 910, 12,700 -> 5,410; in float64
// 1,024 / 16,384 3,550 -> 490, 39,300 -> 2,540; with a loss on forces, float32 1,024 / 16,384 6,470 -> 830, 17,500 -> 3,280,
// float64 7,520 -> 970, 80,000 -> 7,760.  No size was found where library products are faster, so there is no line to draw.
//
// The products run on the matrix instructions of the operands' own precision, v_mfma_f32_16x16x4_f32 and
// v_mfma_f64_16x16x4_f64, with nothing staged through LDS: a lane's piece of either operand is 16 contiguous bytes of a
// row in memory, loaded straight into registers, because the k of a step and the columns of a tile may be dealt to
// the lanes in any order as long as both operands agree.  A step multiplies 4 kVec k (kVec = values per 16 bytes: 4 or 2),
// the lanes of group g = lane / 16 holding k = g kVec .. g kVec + kVec - 1, and the columns of a tile are
// kVec (lane % 16) + j, so that weights as they are stored are read 16 bytes along their columns and outputs are stored 16
// bytes at a time.  Per step a wavefront of the 32-row form loads six kilobytes for 32 matrix instructions (1,024
// cycles): the matrix pipe binds, at the float32 rate (52,000 rows of the eleven-layer network: 74 TFLOP/s of 153).  Float32
// products with enough rows to fill the GPU run on the bfloat16 instructions instead (layer_split_kernel).
#include <algorithm>
#include <type_traits>

#include "khan_internal.h"
#include "net_celu.h"
#include "net_layers.h"
#include "split_bf16.h"

namespace khan {

namespace {

template <typename T> struct MatrixOp;
template <> struct MatrixOp<float> {
    typedef float acc __attribute__((ext_vector_type(4)));
    static constexpr int kVec = 4;
    static __device__ __forceinline__ acc mul(float a, float b, acc c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }
    static __device__ __forceinline__ int row(int lane, int v) { return 4 * (lane >> 4) + v; }      // of result element v
    static __device__ __forceinline__ float celu(float z, float alpha, float inv) { return celu_exact(z, alpha, inv); }
    static __device__ __forceinline__ float celu_abs(float z, float alpha, float inv) { return celu_absolute(z, alpha, inv); }
};
template <> struct MatrixOp<double> {
    typedef double acc __attribute__((ext_vector_type(4)));
    static constexpr int kVec = 2;
    static __device__ __forceinline__ acc mul(double a, double b, acc c) { return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0); }
    static __device__ __forceinline__ int row(int lane, int v) { return (lane >> 4) + 4 * v; }
    static __device__ __forceinline__ double celu(double z, double alpha, double inv) { return z >= 0. ? z : alpha * expm1(z * inv); }
    static __device__ __forceinline__ double celu_abs(double z, double alpha, double inv) { return celu(z, alpha, inv); }
};
template <typename T, int W = MatrixOp<T>::kVec> using Vec = T __attribute__((ext_vector_type(W)));

template <typename T>
__device__ __forceinline__ T slope(T a, T inv_alpha) { return a >= T(0) ? T(1) : fma(a, inv_alpha, T(1)); }

// W values of a row from column c on; kWhole: aligned to their size and inside the row; otherwise one by one, zeros past `end`
template <bool kWhole, typename T, int W = MatrixOp<T>::kVec>
__device__ __forceinline__ Vec<T, W> load(const T* __restrict__ row, int c, int end)
{
    if constexpr (kWhole) {
        return *reinterpret_cast<const Vec<T, W>*>(row + c);
    } else {
        Vec<T, W> v;
#pragma unroll
        for (int e = 0; e < W; ++e) v[e] = c + e < end ? row[min(c + e, end - 1)] : T(0);
        return v;
    }
}

// W sums of each of R rows (r, may lie past the end: not stored) from column `cols` on -> the outputs of the product's kind
// (NetKind); n: rows, N: width.  What the rows need from memory is loaded for all of them before the first is stored: a
// load behind a store waits for that store, and row by row the sixteen round trips of a wavefront's tile were longer than its
// products (gradient of 47,000 rows through 256 x 256: 48 -> 40 us).
template <bool kWhole, int W, int R, typename T>
__device__ __forceinline__ void finish(const NetLayer<T>& a, int t, const int (&r)[R], int n, int cols, int N, Vec<T, W> (&y)[R])
{
    size_t at[R];
#pragma unroll
    for (int i = 0; i < R; ++i) at[i] = static_cast<size_t>(min(r[i], n - 1)) * N;
    auto put = [&](T* out, const Vec<T, W> (&v)[R]) {
#pragma unroll
        for (int i = 0; i < R; ++i) {
            if (r[i] >= n) continue;
            if constexpr (kWhole) {
                *reinterpret_cast<Vec<T, W>*>(out + at[i] + cols) = v[i];
            } else {
#pragma unroll
                for (int e = 0; e < W; ++e)
                    if (cols + e < N) out[at[i] + cols + e] = v[i][e];
            }
        }
    };
    auto get = [&](Vec<T, W> (&v)[R], const T* from) {
#pragma unroll
        for (int i = 0; i < R; ++i) v[i] = load<kWhole, T, W>(from + at[i], cols, N);
    };
    T s[R];
    if (a.kind >= kNetRows) {
#pragma unroll
        for (int i = 0; i < R; ++i) s[i] = T(1);
        if (a.scale[t]) {
#pragma unroll
            for (int i = 0; i < R; ++i) s[i] = a.scale[t][min(r[i], n - 1)];
        }
    }
    if (a.kind == kNetCelu) {
        if (a.absolute) {
#pragma unroll
            for (int i = 0; i < R; ++i)
#pragma unroll
                for (int j = 0; j < W; ++j) y[i][j] = MatrixOp<T>::celu_abs(y[i][j], a.alpha, a.inv_alpha);
        } else {
#pragma unroll
            for (int i = 0; i < R; ++i)
#pragma unroll
                for (int j = 0; j < W; ++j) y[i][j] = MatrixOp<T>::celu(y[i][j], a.alpha, a.inv_alpha);
        }
    } else if (a.kind == kNetRows) {
#pragma unroll
        for (int i = 0; i < R; ++i) y[i] *= s[i];
        if (a.accumulate) {
            Vec<T, W> before[R];
            get(before, a.out[t]);          // (a row past the end reads the last one, whose new value it does not use)
#pragma unroll
            for (int i = 0; i < R; ++i) y[i] += before[i];
        }
    } else {
        Vec<T, W> h[R];
        get(h, a.act[t]);
        if (a.kind == kNetTangent) {
            Vec<T, W> d[R];
            get(d, a.d[t]);
#pragma unroll
            for (int i = 0; i < R; ++i)
#pragma unroll
                for (int j = 0; j < W; ++j) {
                    const T zd = y[i][j] * s[i];
                    d[i][j] = h[i][j] >= T(0) ? T(0) : zd * d[i][j] * a.inv_alpha;
                    y[i][j] = zd * slope(h[i][j], a.inv_alpha);
                }
            put(a.out2[t], d);
        } else {
#pragma unroll
            for (int i = 0; i < R; ++i)
#pragma unroll
                for (int j = 0; j < W; ++j) y[i][j] *= slope(h[i][j], a.inv_alpha);
            if (a.kind == kNetSecond) {
                get(h, a.t[t]);
#pragma unroll
                for (int i = 0; i < R; ++i)
#pragma unroll
                    for (int j = 0; j < W; ++j) y[i][j] = fma(s[i], h[i][j], y[i][j]);
            }
        }
    }
    put(a.out[t], y);
}

// One product for the four types, out = epilogue(in . W) with W [k, n_out] as stored, or (kTrans) in . W^T with W [n_out, k]
// as stored.  A wavefront forms 16 kMI rows x 16 kVec columns.  kSplit: the four wavefronts of a workgroup take every
// fourth step of one tile and their sums meet in LDS (few rows: the latency of a tile is what the launch lasts);
// otherwise a tile each, the column tiles of a row tile side by side, so that they share its rows in cache.
// kWhole: widths are multiples of kVec and every pointer is 16-byte aligned.
template <typename T, int kMI, bool kTrans, bool kSplit, bool kWhole>
__global__ __launch_bounds__(256) void layer_kernel(const NetLayer<T> a, int total)
{
    typedef MatrixOp<T> Op;
    typedef typename Op::acc acc_t;
    constexpr int V = Op::kVec, kStep = 4 * V;
    __shared__ T part[kSplit ? 3 : 1][kSplit ? kMI * V * 4 : 1][64];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int l16 = lane & 15, grp = lane >> 4;
    const int tile = kSplit ? static_cast<int>(blockIdx.x) : static_cast<int>(blockIdx.x) * 4 + wave;
    if (!kSplit && tile >= total) return;
    const int t = (tile >= a.tile_end[0]) + (tile >= a.tile_end[1]) + (tile >= a.tile_end[2]);
    const int rel = tile - (t == 0 ? 0 : a.tile_end[t - 1]);
    const int rt = rel / a.col_tiles, ct = rel - rt * a.col_tiles;
    const int n = a.n[t], K = a.k, N = a.n_out;
    const int row0 = rt * 16 * kMI, col0 = ct * 16 * V;
    const T* __restrict__ in = a.in[t];
    const T* __restrict__ w = a.w[t];

    const T* rows[kMI];                       // this lane's rows (past the end: the last one again, never stored)
#pragma unroll
    for (int i = 0; i < kMI; ++i) rows[i] = in + static_cast<size_t>(min(row0 + i * 16 + l16, n - 1)) * K;
    const int cols = col0 + V * l16;          // this lane's columns cols .. cols + V - 1
    const int wcol = kWhole ? min(cols, N - V) : cols;       // (past the end: others again, never stored)

    Vec<T> av[kMI], bv[V];
    auto fetch = [&](int c) {
        const int k = c * kStep + grp * V;
        // k past the end: zeros from the rows are enough, but the loads have to stay inside the arrays
        const bool live = k < K;
        const int kk = kWhole ? min(k, K - V) : k;
#pragma unroll
        for (int i = 0; i < kMI; ++i) {
            av[i] = load<kWhole>(rows[i], kk, K);
            if (kWhole && !live) av[i] = Vec<T>(T(0));
        }
        if constexpr (!kTrans) {
#pragma unroll
            for (int e = 0; e < V; ++e) {
                if constexpr (kWhole) bv[e] = load<true>(w + static_cast<size_t>(kk + e) * N, wcol, N);
                else bv[e] = load<false>(w + static_cast<size_t>(min(kk + e, K - 1)) * N, wcol, N);
            }
        } else {
#pragma unroll
            for (int j = 0; j < V; ++j) bv[j] = load<kWhole>(w + static_cast<size_t>(min(wcol + j, N - 1)) * K, kk, K);
        }
    };
    acc_t acc[kMI][V];
#pragma unroll
    for (int i = 0; i < kMI; ++i)
#pragma unroll
        for (int j = 0; j < V; ++j) acc[i][j] = acc_t(T(0));
    const int steps = (K + kStep - 1) / kStep;
    const int first = kSplit ? wave : 0, stride = kSplit ? 4 : 1;
    if (first < steps) fetch(first);
#pragma unroll 2
    for (int c = first; c < steps; c += stride) {
        Vec<T> x[kMI], y[V];
#pragma unroll
        for (int i = 0; i < kMI; ++i) x[i] = av[i];
#pragma unroll
        for (int j = 0; j < V; ++j) y[j] = bv[j];
        if (c + stride < steps) fetch(c + stride);           // in flight while this step is multiplied
#pragma unroll
        for (int e = 0; e < V; ++e)
#pragma unroll
            for (int i = 0; i < kMI; ++i)
#pragma unroll
                for (int j = 0; j < V; ++j) acc[i][j] = Op::mul(x[i][e], kTrans ? y[j][e] : y[e][j], acc[i][j]);
    }
    if constexpr (kSplit) {
        if (wave > 0) {
#pragma unroll
            for (int i = 0; i < kMI; ++i)
#pragma unroll
                for (int j = 0; j < V; ++j)
#pragma unroll
                    for (int v = 0; v < 4; ++v) part[wave - 1][(i * V + j) * 4 + v][lane] = acc[i][j][v];
        }
        __syncthreads();
        if (wave > 0) return;
#pragma unroll
        for (int i = 0; i < kMI; ++i)
#pragma unroll
            for (int j = 0; j < V; ++j)
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    const int q = (i * V + j) * 4 + v;
                    acc[i][j][v] = (acc[i][j][v] + part[0][q][lane]) + (part[1][q][lane] + part[2][q][lane]);
                }
    }

    // ---- epilogue: row row0 + 16 i + row(v), columns cols .. cols + V - 1
    if (cols >= N) return;
    Vec<T> bias = Vec<T>(T(0));
    if (a.bias[t]) bias = load<kWhole>(a.bias[t], cols, N);
#pragma unroll
    for (int i = 0; i < kMI; ++i) {
        int r[4];
        Vec<T> y[4];
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            r[v] = row0 + i * 16 + Op::row(lane, v);
#pragma unroll
            for (int j = 0; j < V; ++j) y[v][j] = acc[i][j][v] + bias[j];
        }
        finish<kWhole, V, 4>(a, t, r, n, cols, N, y);
    }
}

// The same product in float32 for many rows and wide layers, on the bfloat16 matrix instructions: every operand is split
// into three bfloat16 values and the six largest of the nine partial products are accumulated in float32 (the split and
// what it leaves out: dense_first.hip; infinite operands give NaN there as here).
// A workgroup forms 128 rows x 32 kNB columns in chunks of 32 k.  A wavefront has 32 rows: its lanes load and split the
// rows' values themselves, in registers, once per workgroup; the weights go through LDS, split by the workgroup for its
// four wavefronts, a thread a block of 4 k x kNB columns.  LDS holds [plane][8 k][column] pieces of 16 bytes, column
// kNB c + j of the tile at place 32 j + c: reads and writes run along consecutive places, or (writes of transposed weights)
// over the four 8 k, two places apart in the banks: no bank conflicts; and a lane's kNB matrix blocks are neighbouring
// columns, stored and loaded together.  The next chunk's loads are in flight during a chunk's products, its weights go into
// the other of two buffers: one barrier per chunk.
// Per chunk a wavefront issues 48 matrix instructions (1,536 cycles; kNB = 4) and 250 vector ones (1,000), most of them
// splitting, and the two hide each other only in part: 172 TFLOP/s where the float32 instructions gave 70 (96,000 rows
// 256 -> 256: 139 -> 73 us; 48,000 rows 73 -> 38; transposed 78 -> 40).
// kApart (64 columns): the five small partial products have accumulators of their own.  The large sum is then rounded once in
// 16 k instead of six times, and a layer's distance from float64 is 0.4 of the float32 library product's, where without it
// it can lie above (values of 384-192-100-8-1 networks on 47,000 rows: library 2.17e-7, without 2.40e-7, with 2.12e-7).  It
// costs nothing with 64 columns (12,000 rows 384 -> 128: 17.9 -> 17.8 us); with 128 there are no registers for it at three
// workgroups per compute unit (two: deep networks on 47,000 rows 1,790 -> 1,950 us).
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f4v __attribute__((ext_vector_type(4)));
constexpr int kWideRows = 128;

template <int kNB, bool kTrans, bool kApart>
__global__ __launch_bounds__(256, 3) void layer_split_kernel(const NetLayer<float> a, int row_tiles)
{
    typedef Vec<float, kNB> vec;
    constexpr int kCols = 32 * kNB;
    __shared__ u4v S[2][3][4][kCols + 2];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int l32 = lane & 31, half = lane >> 5;
    // the column tiles of a row tile run side by side on one XCD (workgroup w is on XCD w % 8), whose L2 they share
    const int xcd = blockIdx.x & 7, q = blockIdx.x >> 3;
    const int ct = q % a.col_tiles, tile = q / a.col_tiles * 8 + xcd;
    if (tile >= row_tiles) return;
    const int t = (tile >= a.tile_end[0]) + (tile >= a.tile_end[1]) + (tile >= a.tile_end[2]);
    const int rt = tile - (t == 0 ? 0 : a.tile_end[t - 1]);
    const int n = a.n[t], K = a.k, N = a.n_out;
    const int row0 = rt * kWideRows + wave * 32;
    const float* __restrict__ row = a.in[t] + static_cast<size_t>(min(row0 + l32, n - 1)) * K;
    const float* __restrict__ w = a.w[t];
    // this thread's weights: columns kNB wc .. of the tile (past the end: others again, never stored), k 4 wk .. + 3;
    // neighbouring lanes along the weights' rows in memory
    const int wc = kTrans ? threadIdx.x >> 3 : threadIdx.x & 31, wk = kTrans ? threadIdx.x & 7 : threadIdx.x >> 5;
    const int wcol = min(ct * kCols + kNB * wc, N - kNB);
    const float* __restrict__ wsrc = kTrans ? w + static_cast<size_t>(wcol) * K + 4 * wk : w + static_cast<size_t>(4 * wk) * N + wcol;
    const size_t wnext = kTrans ? K : N, wstep = kTrans ? 32 : static_cast<size_t>(32) * N;

    f4v av[4];
    typename std::conditional<kTrans, f4v, vec>::type wv[kTrans ? kNB : 4];
    auto fetch = [&](int c) {
#pragma unroll
        for (int i = 0; i < (kTrans ? kNB : 4); ++i) wv[i] = *reinterpret_cast<const decltype(wv[0] + wv[0])*>(wsrc + c * wstep + i * wnext);
#pragma unroll
        for (int i = 0; i < 4; ++i) av[i] = *reinterpret_cast<const f4v*>(row + c * 32 + (i >> 1) * 16 + half * 8 + (i & 1) * 4);
    };
    auto stage = [&](int buffer) {
#pragma unroll
        for (int j = 0; j < kNB; ++j) {
            unsigned lo[3], hi[3];
            if constexpr (kTrans) {
                split_pair(wv[j][0], wv[j][1], lo[0], lo[1], lo[2]);
                split_pair(wv[j][2], wv[j][3], hi[0], hi[1], hi[2]);
            } else {
                split_pair(wv[0][j], wv[1][j], lo[0], lo[1], lo[2]);
                split_pair(wv[2][j], wv[3][j], hi[0], hi[1], hi[2]);
            }
#pragma unroll
            for (int p = 0; p < 3; ++p)
                reinterpret_cast<u2v*>(&S[buffer][p][wk >> 1][32 * j + wc])[wk & 1] = u2v{lo[p], hi[p]};
        }
    };
    f32x16 acc[kNB], apart[kApart ? kNB : 1];
    auto& small = [&]() -> f32x16(&)[kNB] {
        if constexpr (kApart) return apart;
        else return acc;
    }();
#pragma unroll
    for (int j = 0; j < kNB; ++j) acc[j] = small[j] = f32x16(0.f);
    const int chunks = K / 32;
    fetch(0);
    stage(0);
    for (int c = 0; c < chunks; ++c) {
        f4v x[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) x[i] = av[i];
        __syncthreads();              // chunk c is in its buffer, and the reads of the other one are done
        if (c + 1 < chunks) fetch(c + 1);
#pragma unroll
        for (int s = 0; s < 2; ++s) {
            u4v xs[3];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                unsigned p[3];
                const f4v v = x[2 * s + (e >> 1)];
                split_pair(v[2 * (e & 1)], v[2 * (e & 1) + 1], p[0], p[1], p[2]);
                xs[0][e] = p[0], xs[1][e] = p[1], xs[2][e] = p[2];
            }
            auto mul = [&](f32x16 (&to)[kNB], int i, int p) {
#pragma unroll
                for (int j = 0; j < kNB; ++j)
                    to[j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, xs[i]),
                                                                    __builtin_bit_cast(bf16x8, S[c & 1][p][2 * s + half][32 * j + l32]), to[j], 0, 0, 0);
            };
            mul(small, 0, 2);
            mul(small, 1, 1);
            mul(small, 0, 1);
            mul(small, 2, 0);
            mul(small, 1, 0);
            mul(acc, 0, 0);
        }
        if (c + 1 < chunks) stage((c + 1) & 1);
    }
    if constexpr (kApart) {
#pragma unroll
        for (int j = 0; j < kNB; ++j) acc[j] += small[j];
    }
    // element v of a block: row 8 (v / 4) + 4 half + v % 4, column kNB l32 + (the block's number)
    const int cols = ct * kCols + kNB * l32;
    if (cols >= N) return;
    vec bias = vec(0.f);
    if (a.bias[t]) bias = load<true, float, kNB>(a.bias[t], cols, N);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        int r[4];
        vec y[4];
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            r[v] = row0 + 8 * i + 4 * half + v;
            y[v] = bias;
#pragma unroll
            for (int j = 0; j < kNB; ++j) y[v][j] += acc[j][4 * i + v];
        }
        finish<true, kNB, 4>(a, t, r, n, cols, N, y);
    }
}

// The output layer, 16 lanes per row: value = a . w + b and d = w celu'(a), whichever is asked for; or (second) q = s t.
// Sixteen lanes a row, kVec values each at a time, all of a row's loads together (one value at a time, each step's behind the
// last one's stores and the addresses of the rows' types from memory: 36,000 rows of 64 10.4 us where it is 6.5 now).
template <typename T, bool kWhole>
__global__ __launch_bounds__(256) void top_kernel(const NetTop<T> a, int total)
{
    constexpr int V = MatrixOp<T>::kVec, kSteps = 4;
    const int row = static_cast<int>(blockIdx.x) * 16 + static_cast<int>(threadIdx.x >> 4), sub = threadIdx.x & 15;
    if (row >= total) return;
    const int t = (row >= a.row_end[0]) + (row >= a.row_end[1]) + (row >= a.row_end[2]);
    const int r = row - (t == 0 ? 0 : t == 1 ? a.row_end[0] : t == 2 ? a.row_end[1] : a.row_end[2]);
    const size_t base = static_cast<size_t>(r) * a.k;
    const auto of = [&](auto* const (&p)[4]) { return t == 0 ? p[0] : t == 1 ? p[1] : t == 2 ? p[2] : p[3]; };
    T* const out = of(a.out);
    const auto put = [&](int c, const Vec<T>& v) {
        if constexpr (kWhole) {
            *reinterpret_cast<Vec<T>*>(out + base + c) = v;
        } else {
#pragma unroll
            for (int e = 0; e < V; ++e)
                if (c + e < a.k) out[base + c + e] = v[e];
        }
    };
    if (a.second) {
        const T* const scale = of(a.scale);
        const T s = scale ? scale[r] : T(1);
        for (int c = sub * V; c < a.k; c += 16 * V) put(c, load<kWhole, T>(of(a.t) + base, c, a.k) * s);
        return;
    }
    const T *const act = of(a.act) + base, *const weight = of(a.w);
    T sum = T(0);
    for (int c0 = sub * V; c0 < a.k; c0 += kSteps * 16 * V) {
        Vec<T> h[kSteps], w[kSteps];
#pragma unroll
        for (int u = 0; u < kSteps; ++u) {
            if (c0 - sub * V + u * 16 * V >= a.k) break;                 // (the same for all)
            const int c = min(c0 + u * 16 * V, a.k - 1) / V * V;         // (past the end: the last values again, not used)
            h[u] = load<kWhole, T>(act, c, a.k);
            w[u] = load<kWhole, T>(weight, c, a.k);
        }
#pragma unroll
        for (int u = 0; u < kSteps; ++u) {
            const int c = c0 + u * 16 * V;
            if (c >= a.k) break;
#pragma unroll
            for (int e = 0; e < V; ++e) sum = fma(h[u][e], w[u][e], sum);
            if (out) {
#pragma unroll
                for (int e = 0; e < V; ++e) h[u][e] = w[u][e] * slope(h[u][e], a.inv_alpha);
                put(c, h[u]);
            }
        }
    }
    T* const value = of(a.value);
    if (value) {
#pragma unroll
        for (int d = 8; d >= 1; d >>= 1) sum += __shfl_xor(sum, d, 64);
        const T* const bias = of(a.bias);
        if (sub == 0) value[r] = sum + (bias ? *bias : T(0));
    }
}

// ---- gradients of the weights: dW [k, n_out] = sum over rows of left[r, :]^T right[r, :] (+ left2^T right2), db = sum of right
// A workgroup forms a tile of 16 kVec x 16 kVec (64 x 64, or 32 x 32 in float64) over `per` rows, its wavefronts four rows in
// sixteen each; a lane's 16 bytes of a row are kVec of the tile's rows (left) or columns (right), the four groups of lanes
// hold four rows: one load of each operand per kVec^2 matrix instructions.  The wavefronts' sums meet in LDS, the
// workgroups' in memory, where grad_sum_kernel adds them up in a fixed order: no atomics, the same bits every time.
// The column sums (the biases' gradients, factors of random sign that cancel) are formed by the first row of tiles alone and
// carry their rounding errors along: added up plainly, 64 rows to a lane, they were 2e-7 off where a library sum is 4e-8 off
// (124 -> 126 us a launch at 35,000 rows).
// In float32 this form is left for layers narrower than 64, for few rows and for operands that are not aligned
// (weight_grad_split_tile takes the others): 61 TFLOP/s of the instructions' 153 at 35,000 rows of 384-128-128-64-1 (85 us).
// The compiler's overlap of the unrolled loop's loads with the products beats four row groups loaded ahead by hand (104 us).
// sum += x, its rounding error added to `lost` (Knuth's two-sum)
template <typename V>
__device__ __forceinline__ void add_exactly(V& sum, V& lost, V x)
{
    const V s = sum + x, b = s - sum;
    lost += (sum - (s - b)) + (x - b);
    sum = s;
}
template <typename T>
__device__ __forceinline__ T with_lost(T sum, T lost) { return isfinite(sum) ? sum + lost : sum; }      // (lost is NaN beside an infinite sum)

template <typename T>
struct GradLds {
    static constexpr int kVec = MatrixOp<T>::kVec;
    T part[2][kVec * kVec * 4][64];
    T bias[4][16 * kVec];
};
template <typename T, bool kWhole>
__device__ __forceinline__ void weight_grad_tile(const NetGrads<T>& a, T* __restrict__ partial, GradLds<T>& S, int job, int rel)
{
    typedef MatrixOp<T> Op;
    typedef typename Op::acc acc_t;
    constexpr int V = Op::kVec, kSide = 16 * V;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int l16 = lane & 15, grp = lane >> 4;
    const int layer = job >> 2, t = job & 3;
    const int K = a.k[layer], N = a.k[layer + 1], n = a.n[t];
    const int tiles_n = (N + kSide - 1) / kSide, tiles = (K + kSide - 1) / kSide * tiles_n;
    const int split = rel / tiles, tile = rel - split * tiles;
    const int i0 = tile / tiles_n * kSide, j0 = tile % tiles_n * kSide;
    const int r0 = split * a.per, r1 = min(n, r0 + a.per);
    acc_t acc[V][V];
#pragma unroll
    for (int i = 0; i < V; ++i)
#pragma unroll
        for (int j = 0; j < V; ++j) acc[i][j] = acc_t(T(0));
    Vec<T> bias = Vec<T>(T(0)), bias_lost = Vec<T>(T(0));
    const int ci = i0 + V * l16, cj = j0 + V * l16;
    const int li = kWhole ? min(ci, K - V) : ci, lj = kWhole ? min(cj, N - V) : cj;
#pragma unroll 1
    for (int pair = 0; pair < 2; ++pair) {
        if (!(((pair == 0 ? a.first : a.second) >> layer) & 1u)) continue;
        const T* left = pair == 0 ? a.left[layer] : a.left2[layer];
        const T* right = pair == 0 ? a.right[layer] : a.right2[layer];
        if (layer == 0) left = pair == 0 ? a.x[t] : a.x2[t];
        else left += static_cast<size_t>(a.row0[t]) * K;
        const bool ones = right == nullptr;
        if (!ones) right += static_cast<size_t>(a.row0[t]) * N;
        const T* scale = (pair == 0 ? a.scale_first : a.scale_second) ? a.scale[t] : nullptr;
#pragma unroll 4
        for (int r = r0 + wave * 4 + grp; r < r0 + a.per; r += 16) {
            const bool live = r < r1;
            const size_t at = static_cast<size_t>(live ? r : r1 - 1);
            Vec<T> x = load<kWhole>(left + at * K, li, K);
            Vec<T> y = ones ? Vec<T>(T(1)) : load<kWhole>(right + at * N, lj, N);
            const T s = scale ? scale[at] : T(1);
#pragma unroll
            for (int e = 0; e < V; ++e) {
                x[e] = live ? x[e] : T(0);
                y[e] = live ? y[e] * s : T(0);
            }
            if (pair == 0 && i0 == 0) add_exactly(bias, bias_lost, y);
#pragma unroll
            for (int i = 0; i < V; ++i)
#pragma unroll
                for (int j = 0; j < V; ++j) acc[i][j] = Op::mul(x[i], y[j], acc[i][j]);
        }
    }
    // the four wavefronts' sums: 2 and 3 into LDS, 0 and 1 take them, 1 into LDS, 0 takes it
    auto give = [&](int slot) {
#pragma unroll
        for (int i = 0; i < V; ++i)
#pragma unroll
            for (int j = 0; j < V; ++j)
#pragma unroll
                for (int v = 0; v < 4; ++v) S.part[slot][(i * V + j) * 4 + v][lane] = acc[i][j][v];
    };
    auto take = [&](int slot) {
#pragma unroll
        for (int i = 0; i < V; ++i)
#pragma unroll
            for (int j = 0; j < V; ++j)
#pragma unroll
                for (int v = 0; v < 4; ++v) acc[i][j][v] += S.part[slot][(i * V + j) * 4 + v][lane];
    };
#pragma unroll
    for (int e = 0; e < V; ++e) {
        T b = with_lost(bias[e], bias_lost[e]);
        b += __shfl_xor(b, 16, 64);
        b += __shfl_xor(b, 32, 64);
        if (grp == 0) S.bias[wave][V * l16 + e] = b;
    }
    if (wave >= 2) give(wave - 2);
    __syncthreads();
    if (wave < 2) take(wave);
    __syncthreads();
    if (wave == 1) give(0);
    __syncthreads();
    if (wave != 0) return;
    take(0);
    // tile element (i, j): row kVec row(v) + i of the tile, column kVec l16 + j
    T* __restrict__ out = partial + a.job_base[job] + static_cast<size_t>(rel) * (kSide * kSide + kSide);
#pragma unroll
    for (int i = 0; i < V; ++i)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            Vec<T> y;
#pragma unroll
            for (int j = 0; j < V; ++j) y[j] = acc[i][j][v];
            *reinterpret_cast<Vec<T>*>(out + (V * Op::row(lane, v) + i) * kSide + V * l16) = y;
        }
    if (lane < kSide) out[kSide * kSide + lane] = (S.bias[0][lane] + S.bias[1][lane]) + (S.bias[2][lane] + S.bias[3][lane]);
}

// The same in float32 on the bfloat16 matrix instructions (the split of layer_split_kernel), for layers of at least 64 x 64.
// A workgroup forms 128 of the left operand's columns x 128 (kWide) or 64 of the right's over `per_split` rows, 32 rows at a
// time.  The rows are what is summed over, so that a matrix instruction's operand is eight rows of one column, which lie a row
// apart in memory: a thread loads two neighbouring columns of eight rows (a wavefront 512 contiguous bytes of each row), splits
// them and writes them to LDS as [part][eight rows][column] pieces of 16 bytes, column 2 c + j at place 64 j + c, so that
// writes and reads run along consecutive places.  A wavefront multiplies 64 x 64 (32 x 64) from there.  The five small partial
// products have accumulators of their own, so that the large sum is rounded once in 32 rows: the distance from float64 is half
// of the float32 instructions' (35,000 rows: 2.85e-7 -> 1.39e-7; with one set of accumulators 3.06e-7).  The next rows'
// loads are in flight during the products; two workgroups share a compute unit and fill each other's barriers.
// Gradients of 384-128-128-64-1 on 35,000 rows, this launch alone: one pair of operands 85 -> 49 us (105 TFLOP/s), both 160 ->
// 81 (128); 12,132 rows 41 -> 27.  With grad_sum_kernel 92 -> 58, 167 -> 90 and 49 -> 35.  What is left of one pair is products (14 us), splitting and the loads of 144 MB (30 us) one after the other.  No faster: two
// chunks in flight instead of one (with the small products added to the large ones chunk by chunk, for its registers),
// splitting by v_dot2_f32_bf16 (seven instructions instead of eleven).
// Both operands are split 2^24 times their size (the bias sums are formed before): a value's third part has its exponent 24
// below the value's, and of values below 2^-110 it would lose bits at the end of bfloat16's exponents (2^-115: gradients 1e-6
// off, 2^-125: 1e-3), as they are when a loss is scaled down that far.  The sums are scaled back exactly.
// An element that is not finite (infinite, NaN or overflowing operands: the split makes NaN of infinities; sums from 2^80 on)
// has the workgroup form its tile again by float32 multiply-adds whose roundings are carried along (2,048 rows added up plainly
// are further off than the matrix instructions' sums), so that infinities and NaN come out as they do there.
constexpr int kGradLeft = 128, kGradChunk = 32;
constexpr float kGradLift = 0x1p24f;
struct SplitGradLds {
    u4v left[3][4][kGradLeft], right[3][4][128];
};
__device__ __forceinline__ int grad_place(int column) { return 64 * (column & 1) + (column >> 1); }
__device__ __forceinline__ int grad_column(int place) { return 2 * (place & 63) + (place >> 6); }

template <bool kWide>
__device__ __forceinline__ void weight_grad_split_tile(const NetGrads<float>& a, float* __restrict__ partial, SplitGradLds& S, int job, int rel)
{
    constexpr int kCols = kWide ? 128 : 64, kRC = kCols / 64;       // right columns of the tile, and per thread
    constexpr int kLB = kWide ? 4 : 2, kRB = 4;                     // a wavefront's blocks of 16 left and right columns
    typedef Vec<float, kRC> rvec;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int l16 = lane & 15, grp = lane >> 4;
    const int lb0 = kWide ? 4 * (wave >> 1) : 2 * wave, rb0 = kWide ? 4 * (wave & 1) : 0;
    const int layer = job >> 2, t = job & 3;
    const int K = a.k[layer], N = a.k[layer + 1], n = a.n[t];
    const int tiles_n = (N + kCols - 1) / kCols, tiles = (K + kGradLeft - 1) / kGradLeft * tiles_n;
    const int share = rel / tiles, tile = rel - share * tiles;
    const int i0 = tile / tiles_n * kGradLeft, j0 = tile % tiles_n * kCols;
    const int r0 = share * a.per_split, r1 = min(n, r0 + a.per_split);
    const int chunks = (r1 - r0 + kGradChunk - 1) / kGradChunk;
    // this thread's columns (past the end: the last ones again, whose sums are never read)
    const int li = min(i0 + 2 * lane, K - 2), lj = min(j0 + kRC * lane, N - kRC);

    struct Operands {
        const float *left, *right, *scale;
    };
    auto operands = [&](int pair) -> Operands {
        const float* left = pair == 0 ? a.left[layer] : a.left2[layer];
        const float* right = pair == 0 ? a.right[layer] : a.right2[layer];
        left = layer == 0 ? (pair == 0 ? a.x[t] : a.x2[t]) : left + static_cast<size_t>(a.row0[t]) * K;
        return {left, right + static_cast<size_t>(a.row0[t]) * N, (pair == 0 ? a.scale_first : a.scale_second) ? a.scale[t] : nullptr};
    };
    auto live_pair = [&](int pair) { return (((pair == 0 ? a.first : a.second) >> layer) & 1u) != 0; };
    f4v acc[kRB][kLB], small[kRB][kLB];
#pragma unroll
    for (int i = 0; i < kRB; ++i)
#pragma unroll
        for (int j = 0; j < kLB; ++j) acc[i][j] = small[i][j] = f4v(0.f);
    rvec bias = rvec(0.f), bias_lost = rvec(0.f);
    f2v x[8];
    rvec y[8];
#pragma unroll 1
    for (int pair = 0; pair < 2; ++pair) {
        if (!live_pair(pair)) continue;
        const Operands op = operands(pair);
        auto fetch = [&](int c) {
            const int r = r0 + c * kGradChunk + 8 * wave;
            if (r + 8 <= r1) {
                const float* left = op.left + static_cast<size_t>(r) * K;
                const float* right = op.right + static_cast<size_t>(r) * N;
#pragma unroll
                for (int i = 0; i < 8; ++i) {
                    x[i] = *reinterpret_cast<const f2v*>(left + li);
                    y[i] = *reinterpret_cast<const rvec*>(right + lj);
                    left += K;
                    right += N;
                }
            } else {
#pragma unroll
                for (int i = 0; i < 8; ++i) {
                    const size_t at = static_cast<size_t>(min(r + i, r1 - 1));
                    x[i] = *reinterpret_cast<const f2v*>(op.left + at * K + li);
                    y[i] = *reinterpret_cast<const rvec*>(op.right + at * N + lj);
                }
            }
        };
        fetch(0);
#pragma unroll 1
        for (int c = 0; c < chunks; ++c) {
            const int r = r0 + c * kGradChunk + 8 * wave;
            if (r + 8 <= r1) {
                if (op.scale) {
#pragma unroll
                    for (int i = 0; i < 8; ++i) y[i] *= op.scale[r + i];
                }
            } else {
#pragma unroll
                for (int i = 0; i < 8; ++i) {
                    const float s = op.scale ? op.scale[min(r + i, r1 - 1)] : 1.0f;
                    y[i] = r + i < r1 ? y[i] * s : rvec(0.f);
                    if (r + i >= r1) x[i] = f2v(0.f);
                }
            }
            if (pair == 0 && i0 == 0) {
#pragma unroll
                for (int i = 0; i < 8; ++i) add_exactly(bias, bias_lost, y[i]);
            }
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                x[i] *= kGradLift;
                y[i] *= kGradLift;
            }
            __syncthreads();                   // the planes' previous contents have been read
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                u4v p[3];
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    unsigned q[3];
                    split_pair(x[2 * e][j], x[2 * e + 1][j], q[0], q[1], q[2]);
                    p[0][e] = q[0], p[1][e] = q[1], p[2][e] = q[2];
                }
#pragma unroll
                for (int q = 0; q < 3; ++q) S.left[q][wave][64 * j + lane] = p[q];
            }
#pragma unroll
            for (int j = 0; j < kRC; ++j) {
                u4v p[3];
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    unsigned q[3];
                    split_pair(y[2 * e][j], y[2 * e + 1][j], q[0], q[1], q[2]);
                    p[0][e] = q[0], p[1][e] = q[1], p[2][e] = q[2];
                }
#pragma unroll
                for (int q = 0; q < 3; ++q) S.right[q][wave][64 * j + lane] = p[q];
            }
            __syncthreads();
            if (c + 1 < chunks) fetch(c + 1);  // in flight while this chunk is multiplied
            bf16x8 lv[3][kLB];
#pragma unroll
            for (int q = 0; q < 3; ++q)
#pragma unroll
                for (int j = 0; j < kLB; ++j) lv[q][j] = __builtin_bit_cast(bf16x8, S.left[q][grp][16 * (lb0 + j) + l16]);
#pragma unroll
            for (int q = 2; q >= 0; --q) {
                bf16x8 rv[kRB];
#pragma unroll
                for (int i = 0; i < kRB; ++i) rv[i] = __builtin_bit_cast(bf16x8, S.right[q][grp][16 * (rb0 + i) + l16]);
#pragma unroll
                for (int p = 2 - q; p >= 0; --p)
#pragma unroll
                    for (int i = 0; i < kRB; ++i)
#pragma unroll
                        for (int j = 0; j < kLB; ++j) {
                            f4v& to = p + q == 0 ? acc[i][j] : small[i][j];
                            to = __builtin_amdgcn_mfma_f32_16x16x32_bf16(rv[i], lv[p][j], to, 0, 0, 0);
                        }
            }
        }
    }
    // element v of a block: right place 16 (rb0 + i) + 4 grp + v, left place 16 (lb0 + j) + l16
    bool bad = false;
#pragma unroll
    for (int i = 0; i < kRB; ++i)
#pragma unroll
        for (int j = 0; j < kLB; ++j) {
            acc[i][j] += small[i][j];
#pragma unroll
            for (int v = 0; v < 4; ++v) bad = bad || !isfinite(acc[i][j][v]);
        }
    const bool again = __syncthreads_or(bad);
#pragma unroll
    for (int i = 0; i < kRB; ++i)
#pragma unroll
        for (int j = 0; j < kLB; ++j) acc[i][j] *= 1.0f / (kGradLift * kGradLift);
    if (again) {
        // (a block of 16 right columns at a time: the roundings of all of them do not fit in the registers)
#pragma unroll
        for (int i = 0; i < kRB; ++i) {
            f4v lost[kLB];
#pragma unroll
            for (int j = 0; j < kLB; ++j) acc[i][j] = lost[j] = f4v(0.f);
#pragma unroll 1
            for (int pair = 0; pair < 2; ++pair) {
                if (!live_pair(pair)) continue;
                const Operands op = operands(pair);
#pragma unroll 1
                for (int r = r0; r < r1; ++r) {
                    const float s = op.scale ? op.scale[r] : 1.0f;
                    float lv[kLB];
#pragma unroll
                    for (int j = 0; j < kLB; ++j)
                        lv[j] = op.left[static_cast<size_t>(r) * K + min(i0 + grad_column(16 * (lb0 + j) + l16), K - 1)];
#pragma unroll
                    for (int v = 0; v < 4; ++v) {
                        const int place = 16 * (rb0 + i) + 4 * grp + v, column = j0 + (kWide ? grad_column(place) : place);
                        const float rv = op.right[static_cast<size_t>(r) * N + min(column, N - 1)] * s;
#pragma unroll
                        for (int j = 0; j < kLB; ++j) {
                            const float sum = acc[i][j][v], s1 = fmaf(lv[j], rv, sum), b = s1 - sum;
                            lost[j][v] += fmaf(lv[j], rv, -b) + (sum - (s1 - b));
                            acc[i][j][v] = s1;
                        }
                    }
                }
            }
#pragma unroll
            for (int j = 0; j < kLB; ++j)
#pragma unroll
                for (int v = 0; v < 4; ++v) acc[i][j][v] = with_lost(acc[i][j][v], lost[j][v]);
        }
    }
    // partial sums: [left place][right place], then the right columns' own sums by place
    float* __restrict__ out = partial + a.job_base[job] + static_cast<size_t>(rel) * (kGradLeft * kCols + kCols);
#pragma unroll
    for (int j = 0; j < kLB; ++j)
#pragma unroll
        for (int i = 0; i < kRB; ++i)
            *reinterpret_cast<f4v*>(out + (16 * (lb0 + j) + l16) * kCols + 16 * (rb0 + i) + 4 * grp) = acc[i][j];
    if (i0 != 0) return;
    float* const sums = reinterpret_cast<float*>(S.left);       // (the last reads of the planes lie before the barrier above)
#pragma unroll
    for (int j = 0; j < kRC; ++j) sums[wave * 128 + 64 * j + lane] = with_lost(bias[j], bias_lost[j]);
    __syncthreads();
    if (threadIdx.x < kCols) {
        const float* b = sums + threadIdx.x;
        out[kGradLeft * kCols + threadIdx.x] = (b[0] + b[128]) + (b[256] + b[384]);
    }
}

// kSplit: some of the layers are on split products.  A form of its own: with them in one kernel the others' workgroups, 152
// registers and 33.8 KB of LDS, had 255 and 49.4 KB and were two on a compute unit instead of three (3,500 rows 17.7 -> 22.2 us).
template <typename T, bool kSplit>
__global__ __launch_bounds__(256, kSplit || sizeof(T) == 8 ? 2 : 1) void weight_grad_kernel(const NetGrads<T> a, T* __restrict__ partial)
{
    int job = 0;
    while (static_cast<int>(blockIdx.x) >= a.job_end[job]) ++job;                 // (layer, type)
    const int rel = static_cast<int>(blockIdx.x) - (job == 0 ? 0 : a.job_end[job - 1]);
    if constexpr (kSplit) {
        __shared__ union {
            GradLds<float> plain;
            SplitGradLds split;
        } S;
        if ((a.split >> (job >> 2)) & 1u) {
            if (a.k[(job >> 2) + 1] > 64) weight_grad_split_tile<true>(a, partial, S.split, job, rel);
            else weight_grad_split_tile<false>(a, partial, S.split, job, rel);
        } else if ((a.whole >> (job >> 2)) & 1u) {
            weight_grad_tile<T, true>(a, partial, S.plain, job, rel);
        } else {
            weight_grad_tile<T, false>(a, partial, S.plain, job, rel);
        }
    } else {
        __shared__ GradLds<T> S;
        if ((a.whole >> (job >> 2)) & 1u) weight_grad_tile<T, true>(a, partial, S, job, rel);
        else weight_grad_tile<T, false>(a, partial, S, job, rel);
    }
}

// The workgroups' partial tiles and bias sums -> the gradients: 64 runs of 16 bytes of one tile to a wavefront, or (kQuarters) to a
// workgroup, whose wavefronts take a quarter of the shares each; the quarters are added in order.
template <typename T, bool kQuarters>
__global__ __launch_bounds__(256) void grad_sum_kernel(const NetGrads<T> a, const T* __restrict__ partial)
{
    constexpr int V = MatrixOp<T>::kVec, kSide = 16 * V, kRun = 64 * V;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    int64_t out = 0;                       // where the layer's weights begin
    int block = static_cast<int>(blockIdx.x), layer = 0, rows, cols, tiles_n, tiles, runs;
    if constexpr (!kQuarters) block = 4 * block + wave;
    bool split;
    for (;; ++layer) {
        if (!kQuarters && layer == a.layers) return;
        split = (a.split >> layer) & 1u;
        rows = split ? kGradLeft : kSide;
        cols = split ? (a.k[layer + 1] > 64 ? 128 : 64) : kSide;
        tiles_n = (a.k[layer + 1] + cols - 1) / cols;
        tiles = (a.k[layer] + rows - 1) / rows * tiles_n;
        runs = (rows * cols + cols + kRun - 1) / kRun;
        if (block < 4 * tiles * runs) break;
        block -= 4 * tiles * runs;
        out += 4 * static_cast<int64_t>(a.k[layer]) * a.k[layer + 1];
    }
    const int t = block / (tiles * runs), tile = block / runs - t * tiles, at = (block % runs * 64 + lane) * V;
    const int K = a.k[layer], N = a.k[layer + 1], size = rows * cols + cols;
    const int per = split ? a.per_split : a.per, shares = (a.n[t] + per - 1) / per;
    const T* p = partial + a.job_base[layer * 4 + t] + static_cast<size_t>(tile) * size + min(at, size - V);
    const size_t stride = static_cast<size_t>(tiles) * size;
    Vec<T> sum = Vec<T>(T(0)), lost = Vec<T>(T(0));
    const int first = kQuarters ? wave * shares >> 2 : 0, last = kQuarters ? (wave + 1) * shares >> 2 : shares;
    constexpr int U = kQuarters ? 8 : 4;       // loads in flight together
    int s = first;
    for (; s + U <= last; s += U) {
        Vec<T> v[U];
#pragma unroll
        for (int u = 0; u < U; ++u) v[u] = *reinterpret_cast<const Vec<T>*>(p + (s + u) * stride);
#pragma unroll
        for (int u = 0; u < U; ++u) add_exactly(sum, lost, v[u]);
    }
    if (s < last) {
        Vec<T> v[U - 1];
#pragma unroll
        for (int u = 0; u < U - 1; ++u) v[u] = *reinterpret_cast<const Vec<T>*>(p + min(s + u, last - 1) * stride);
#pragma unroll
        for (int u = 0; u < U - 1; ++u)
            if (s + u < last) add_exactly(sum, lost, v[u]);
    }
    if constexpr (kQuarters) {
        __shared__ Vec<T> quarter[4][2][64];
        quarter[wave][0][lane] = sum;
        quarter[wave][1][lane] = lost;
        __syncthreads();
        if (wave > 0) return;
#pragma unroll
        for (int w = 1; w < 4; ++w) {
            add_exactly(sum, lost, quarter[w][0][lane]);
            lost += quarter[w][1][lane];
        }
    }
    if (at >= size) return;
    const bool is_bias = at >= rows * cols;
    if (is_bias && tile >= tiles_n) return;                    // the first row of tiles holds the bias sums
    int row = tile / tiles_n * rows;
    if (!is_bias) row += split ? grad_column(at / cols) : at / cols;
    if (is_bias) {
        // behind all weights, layer by layer
        for (int l = layer; l < a.layers; ++l) out += 4 * static_cast<int64_t>(a.k[l]) * a.k[l + 1];
        for (int l = 0; l < layer; ++l) out += 4 * a.k[l + 1];
    }
    if (row >= K) return;
    T* const to = a.out + out + (is_bias ? static_cast<int64_t>(t) : static_cast<int64_t>(t) * K + row) * N;
    const int place = at % cols, column0 = tile % tiles_n * cols;
    Vec<T> value;
#pragma unroll
    for (int e = 0; e < V; ++e) value[e] = with_lost(sum[e], lost[e]);
    const bool apart = split && cols == 128;                   // (columns two apart)
    if (!apart && column0 + place + V <= N && (reinterpret_cast<uintptr_t>(to + column0 + place) & 15u) == 0) {
        *reinterpret_cast<Vec<T>*>(to + column0 + place) = value;
        return;
    }
#pragma unroll
    for (int e = 0; e < V; ++e) {
        const int column = column0 + (apart ? grad_column(place + e) : place + e);
        if (column < N) to[column] = value[e];
    }
}

template <typename T>
bool aligned(const T* const (&p)[4], const int (&n)[4])
{
    for (int t = 0; t < 4; ++t)
        if (n[t] > 0 && (reinterpret_cast<uintptr_t>(p[t]) & 15u)) return false;
    return true;
}

template <typename T, int kMI, bool kSplit>
void launch_layer_kernel(NetLayer<T>& a, bool trans, bool whole, hipStream_t stream)
{
    constexpr int V = MatrixOp<T>::kVec;
    a.col_tiles = (a.n_out + 16 * V - 1) / (16 * V);
    int total = 0;
    for (int t = 0; t < 4; ++t) a.tile_end[t] = total += (a.n[t] + 16 * kMI - 1) / (16 * kMI) * a.col_tiles;
    const dim3 grid(static_cast<unsigned>(kSplit ? total : (total + 3) / 4));
    if (trans) {
        if (whole) layer_kernel<T, kMI, true, kSplit, true><<<grid, dim3(256), 0, stream>>>(a, total);
        else layer_kernel<T, kMI, true, kSplit, false><<<grid, dim3(256), 0, stream>>>(a, total);
    } else {
        if (whole) layer_kernel<T, kMI, false, kSplit, true><<<grid, dim3(256), 0, stream>>>(a, total);
        else layer_kernel<T, kMI, false, kSplit, false><<<grid, dim3(256), 0, stream>>>(a, total);
    }
}

template <int kNB, bool kApart>
void launch_split(NetLayer<float>& a, bool trans, hipStream_t stream)
{
    a.col_tiles = (a.n_out + 32 * kNB - 1) / (32 * kNB);
    int total = 0;
    for (int t = 0; t < 4; ++t) a.tile_end[t] = total += (a.n[t] + kWideRows - 1) / kWideRows;
    const dim3 grid(static_cast<unsigned>((total + 7) / 8 * 8 * a.col_tiles));
    if (trans) layer_split_kernel<kNB, true, kApart><<<grid, dim3(256), 0, stream>>>(a, total);
    else layer_split_kernel<kNB, false, kApart><<<grid, dim3(256), 0, stream>>>(a, total);
}

}  // namespace

template <typename T>
hipError_t launch_net_layer(NetLayer<T> a, bool trans, hipStream_t stream)
{
    constexpr int V = MatrixOp<T>::kVec;
    const int64_t rows = static_cast<int64_t>(a.n[0]) + a.n[1] + a.n[2] + a.n[3];
    if (rows == 0) return hipSuccess;
    bool whole = a.k % V == 0 && a.n_out % V == 0 && aligned<T>(a.in, a.n) && aligned<T>(a.w, a.n);
    for (int t = 0; t < 4 && whole; ++t)
        if (a.n[t] > 0)
            whole = ((reinterpret_cast<uintptr_t>(a.bias[t]) | reinterpret_cast<uintptr_t>(a.act[t]) | reinterpret_cast<uintptr_t>(a.d[t]) |
                      reinterpret_cast<uintptr_t>(a.t[t]) | reinterpret_cast<uintptr_t>(a.out[t]) | reinterpret_cast<uintptr_t>(a.out2[t])) & 15u) == 0;
    if constexpr (std::is_same<T, float>::value) {
        // Split products from half a workgroup of 128 x 64 per compute unit on (us, float32 instructions -> split): 3,000 rows
        // 256 -> 256 9.2 -> 12.1 (96 tiles), 128 -> 384 transposed 12.6 -> 9.0 (144); 12,000 rows 384 -> 128 22.9 -> 16.8
        // (188), 128 -> 64 5.9 -> 8.5 (94).  128 columns instead of 64 from two such workgroups per compute unit on:
        // 48,000 rows 256 -> 256 43.9 -> 38.4 (750 tiles), 384 -> 128 35.3 -> 34.4 (375), 12,000 rows 23.7 -> 23.4 (188).
        // Output widths that are multiples of 64 are those that dense_first.hip's split products take, with sums rounded as
        // often as here; others are measured against float32 sums, which kApart stays below.
        const int64_t row_tiles = (rows + kWideRows - 1) / kWideRows;
        if (whole && a.k % 32 == 0 && a.n_out >= 64 && row_tiles * ((a.n_out + 63) / 64) >= 128) {
            if (a.n_out % 64) launch_split<2, true>(a, trans, stream);
            else if (row_tiles * ((a.n_out + 127) / 128) >= 512) launch_split<4, false>(a, trans, stream);
            else launch_split<2, false>(a, trans, stream);
            return hipGetLastError();
        }
    }
    // 32 rows per wavefront where that fills the GPU (1,024 SIMDs) with wavefronts of their own, 16 below, and a workgroup
    // per tile where even those are few
    const int64_t col_tiles = (a.n_out + 16 * V - 1) / (16 * V);
    if (rows / 32 * col_tiles >= 1024) launch_layer_kernel<T, 2, false>(a, trans, whole, stream);
    else if (rows / 16 * col_tiles >= 1024 || a.k < 8 * V) launch_layer_kernel<T, 1, false>(a, trans, whole, stream);
    else launch_layer_kernel<T, 1, true>(a, trans, whole, stream);
    return hipGetLastError();
}

template <typename T>
hipError_t launch_net_top(NetTop<T> a, hipStream_t stream)
{
    int total = 0;
    for (int t = 0; t < 4; ++t) a.row_end[t] = total += a.n[t];
    if (total == 0) return hipSuccess;
    bool whole = a.k % MatrixOp<T>::kVec == 0;
    for (int t = 0; t < 4; ++t)
        if (a.n[t] > 0)
            whole = whole && ((reinterpret_cast<uintptr_t>(a.act[t]) | reinterpret_cast<uintptr_t>(a.w[t]) | reinterpret_cast<uintptr_t>(a.t[t]) |
                               reinterpret_cast<uintptr_t>(a.out[t])) & 15u) == 0;
    const auto kernel = whole ? top_kernel<T, true> : top_kernel<T, false>;
    kernel<<<dim3((total + 15u) / 16u), dim3(256), 0, stream>>>(a, total);
    return hipGetLastError();
}

// rows per workgroup, the workgroups' numbering, and the bytes of partial sums; `split`: layers of at least 64 x 64 on split
// products
template <typename T>
static int64_t plan_grads(NetGrads<T>& a, bool split)
{
    constexpr int kSide = 16 * MatrixOp<T>::kVec;
    a.split = 0;
    int64_t tiles = 0, split_tiles = 0, rows = 0;
    for (int t = 0; t < 4; ++t) rows += a.n[t];
    auto tiles_of = [&](int l) -> int64_t {
        const int height = (a.split >> l) & 1u ? kGradLeft : kSide, width = (a.split >> l) & 1u ? (a.k[l + 1] > 64 ? 128 : 64) : kSide;
        return static_cast<int64_t>((a.k[l] + height - 1) / height) * ((a.k[l + 1] + width - 1) / width);
    };
    for (int l = 0; l < a.layers; ++l) {
        if (split && a.k[l] >= 64 && a.k[l + 1] >= 64) a.split |= 1u << l;
        ((a.split >> l) & 1u ? split_tiles : tiles) += tiles_of(l);
    }
    // Few rows are faster on the float32 instructions, whose tiles are smaller, as long as their workgroups, three to a compute
    // unit, are all resident (us with the summation, float32 -> split): 384-128-128-64-1, 5 tiles: 2,000 rows 21 -> 23, 2,500 (798
    // workgroups) 26 -> 24, 4,000 (in larger shares 630) 23 -> 25, 5,000 31 -> 25, 24,000 75 -> 44, with both pairs of
    // operands 125 -> 66; 384-256-1, 6 tiles: 3,000 rows 23 -> 24, 3,500 31 -> 25, 6,000 33 -> 28; 384-64-1, 3 tiles: 4,000
    // rows 17 -> 17, 8,000 24 -> 19; eleven layers, 33 tiles: 300 rows 33 -> 31, 2,000 59 -> 40, 48,000 780 -> 378.
    if (a.split && rows * split_tiles < 24000) {
        NetGrads<T> plain = a;
        const int64_t bytes = plan_grads(plain, false);
        if (plain.job_end[4 * a.layers - 1] <= 3 * kCUs) {
            a = plain;
            return bytes;
        }
    }
    auto blocks_of = [&](int64_t per, int64_t per_row) {
        int64_t shares = 0;
        for (int t = 0; t < 4; ++t) shares += (a.n[t] + per - 1) / per;
        return shares * per_row;
    };
    // about two workgroups per compute unit and wave: short shares where rows are few, and never fewer than 64 rows
    int64_t per = 64;
    while (per < 4096 && rows / per * tiles > 1024) per *= 2;
    // beside split products as many rows as theirs, whose workgroups take as long: all workgroups at once, two per compute unit, or
    // as few such rounds as shares of up to 2,048 rows make (520 workgroups on 512 places took 56 us where 505 take 50).  Where the
    // next larger shares would fit for the narrow layers' sake alone, those alone take them (35,000 rows of 384-128-128-64-1, 516
    // workgroups of 416 rows, 510 with the narrow ones of 448: one pair 50.6 -> 49 us, both 83 -> 81).
    int64_t share = per;
    if (split_tiles) {
        per = share = 4 * kGradChunk;
        for (int64_t rounds = 1; blocks_of(share, split_tiles) + blocks_of(per, tiles) > 512 * rounds;) {
            if (per == share && share < 64 * kGradChunk) per += kGradChunk;
            else if (share < 64 * kGradChunk) share = per;
            else per = share = 4 * kGradChunk, ++rounds;
        }
    }
    a.per = static_cast<int>(per);
    a.per_split = static_cast<int>(share);
    int64_t end = 0, base = 0;
    for (int l = 0; l < a.layers; ++l) {
        const bool is_split = (a.split >> l) & 1u;
        const int64_t size = is_split ? (kGradLeft + 1) * (a.k[l + 1] > 64 ? 128 : 64) : kSide * kSide + kSide;
        const int64_t rows_each = is_split ? share : per;
        for (int t = 0; t < 4; ++t) {
            const int64_t blocks = (a.n[t] + rows_each - 1) / rows_each * tiles_of(l);
            a.job_base[l * 4 + t] = base;
            base += blocks * size;
            a.job_end[l * 4 + t] = static_cast<int>(end += blocks);
        }
    }
    return base * static_cast<int64_t>(sizeof(T));
}

// (which of the two plans a launch takes depends on its operands' alignment too, which may not be known yet)
template <typename T>
size_t net_grads_workspace(NetGrads<T> a)
{
    const int64_t plain = plan_grads(a, false), split = std::is_same<T, float>::value ? plan_grads(a, true) : 0;
    return static_cast<size_t>(std::max(plain, split)) + 16;
}

template <typename T>
hipError_t launch_net_grads(NetGrads<T> a, void* workspace, hipStream_t stream)
{
    constexpr int V = MatrixOp<T>::kVec;
    a.whole = 0;
    bool split = std::is_same<T, float>::value;
    for (int l = 0; l < a.layers; ++l) {
        // (operands that a layer does not have are null, which is aligned)
        const uintptr_t bits = reinterpret_cast<uintptr_t>(a.right[l]) | reinterpret_cast<uintptr_t>(a.right2[l]) |
                               reinterpret_cast<uintptr_t>(a.left[l]) | reinterpret_cast<uintptr_t>(a.left2[l]);
        const bool whole = a.k[l] % V == 0 && a.k[l + 1] % V == 0 && (bits & 15u) == 0 && (l > 0 || (aligned<T>(a.x, a.n) && aligned<T>(a.x2, a.n)));
        if (whole) a.whole |= 1u << l;
        const bool ones = ((a.first >> l & 1u) && !a.right[l]) || ((a.second >> l & 1u) && !a.right2[l]);
        if (a.k[l] >= 64 && a.k[l + 1] >= 64 && (!whole || ones)) split = false;
    }
    plan_grads(a, split);
    const int blocks = a.job_end[a.layers * 4 - 1];
    if (blocks > 0) {
        auto kernel = weight_grad_kernel<T, false>;
        if constexpr (std::is_same<T, float>::value) {
            if (a.split) kernel = weight_grad_kernel<T, true>;
        }
        kernel<<<dim3(static_cast<unsigned>(blocks)), dim3(256), 0, stream>>>(a, static_cast<T*>(workspace));
    }
    int64_t sums = 0;
    for (int l = 0; l < a.layers; ++l) {
        const int rows = a.split >> l & 1u ? kGradLeft : 16 * V, cols = a.split >> l & 1u ? (a.k[l + 1] > 64 ? 128 : 64) : 16 * V;
        sums += 4ll * ((a.k[l] + rows - 1) / rows) * ((a.k[l + 1] + cols - 1) / cols) * ((rows * cols + cols + 64 * V - 1) / (64 * V));
    }
    // A workgroup's four wavefronts to each run where there are few runs for the shares (us of gradients and sums, a wavefront to
    // each run -> four): 384-128-128-64-1 (1,300 times 64 runs), 8 shares 15.4 -> 16.7, 17 shares 20.3 -> 20.4, 85 shares
    // 69.7 -> 67.9; 384-64-1 (480), 10 shares 13.2 -> 12.8; eleven layers (9,600 to 11,600), 3 to 13 shares 31 -> 50, 61 -> 80, 372 -> 387.
    int most = 0;
    for (int t = 0; t < 4; ++t) most = std::max(most, a.n[t]);
    if ((static_cast<int64_t>(most) + a.per_split - 1) / a.per_split * 50 > sums)
        grad_sum_kernel<T, true><<<dim3(static_cast<unsigned>(sums)), dim3(256), 0, stream>>>(a, static_cast<const T*>(workspace));
    else
        grad_sum_kernel<T, false><<<dim3(static_cast<unsigned>((sums + 3) / 4)), dim3(256), 0, stream>>>(a, static_cast<const T*>(workspace));
    return hipGetLastError();
}

template hipError_t launch_net_layer<float>(NetLayer<float>, bool, hipStream_t);
template hipError_t launch_net_layer<double>(NetLayer<double>, bool, hipStream_t);
template hipError_t launch_net_top<float>(NetTop<float>, hipStream_t);
template hipError_t launch_net_top<double>(NetTop<double>, hipStream_t);
template size_t net_grads_workspace<float>(NetGrads<float>);
template size_t net_grads_workspace<double>(NetGrads<double>);
template hipError_t launch_net_grads<float>(NetGrads<float>, void*, hipStream_t);
template hipError_t launch_net_grads<double>(NetGrads<double>, void*, hipStream_t);

}  // namespace khan
