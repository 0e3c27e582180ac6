// Inference of float32 networks with CELU of up to twelve layers (khan/model/nn.py:38-68, khan/inference/energy_server.py:121-123), for
// the four atom types: all layers of the forward pass in one launch, and all layers of the way back to the feature rows in another.
// With the names of net_layers.hip, a_l = celu(a_{l-1} W_l + b_l), value = a_L w + b; d_L = w celu'(a_L), d_{l-1} = (d_l W_l^T)
// celu'(a_{l-1}), row gradient = s d_1 W_1^T.
//
// The products are made of half-precision ones (split_half.h, dense_fused.hip): every operand as the sum of two half-precision values,
// three of the four partial products accumulated in float32, the two small ones in an accumulator of their own.  Half precision has
// no room for float32's exponents, so a row's operand is scaled by the power of two that brings its largest value to 2^14, and so is each
// column of the weights: what is within 2^-28 of its row's (column's) largest value keeps all its bits, what is smaller an error of
// 2^-52 of that value.  The three-way bfloat16 split needs six products: deep networks with charges on 4,001 organic molecules
// 1,527 us so and 1,266 like this, deep ones alone on 100 molecules 182 and 164, default ones with charges on 16,384 1,264 and 1,226.
// Relative errors against float64 of energies and gradients of the first of these, layer by layer on the bfloat16 split
// 4.5e-7 and 1.28e-6, in one launch on it 2.8e-7 and 8.2e-7, like this 2.9e-7 and 9.2e-7 (of default networks with charges on 3,000:
// 4.0e-7 and 8.3e-7, 3.3e-7 and 6.9e-7, 3.3e-7 and 7.4e-7; boxes with deep ones 9.9e-7 and 10.5e-7, 7.2e-7 and 7.4e-7, 5.3e-7 and 8.2e-7).
//
// Layer by layer, the tiles of a launch run side by side, first all waiting for their rows, then
// all multiplying, then all storing.  Here a workgroup takes 64 (or
// 32) rows through all layers: the rows of the next product are split once, by the lanes that have just formed them, into two planes
// in LDS (66 KB for 64 rows of 256), and the weights, split and packed beforehand by a launch of their own, go from memory straight to
// registers, 4 KB or 8 KB of a wavefront's ahead, across the ends of the layers.  A wavefront takes 64 columns of all 64 rows, or 32 (of 32
// rows where the layer is so narrow that its columns would leave wavefronts idle), so that no two of a workgroup load the same
// weights.  Four wavefronts with 64 columns each instead of eight with 32 leave room for a second workgroup on the compute unit, which
// multiplies while the first forms activations: deep networks on 2,700 molecules 490 -> 418 us.  Of 512 such tiles' 155 us
// forward the matrix instructions are 41, the vector ones 35, and 31 go into storing the activations; reading the rows of the next
// chunk from LDS ahead of a chunk's products, and three vector instructions less in CELU, changed nothing.
// The weights are the matrix instruction's first operand and the rows its second: a lane has one row and, with the columns packed in a
// suitable order, twice eight neighbouring columns of it, which go to the planes 16 bytes at a time.  The activations that the
// way back needs go to memory in the order in which the lanes hold them, a kilobyte at a time, and come back the same way.
// Widths are padded to multiples of 64 with weights and biases of zero.
#include <algorithm>
#include <climits>
#include <type_traits>

#include "khan_internal.h"
#include "net_chain.h"
#include "net_celu.h"
#include "split_half.h"

namespace khan {

namespace {

typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f4v __attribute__((ext_vector_type(4)));

constexpr int kParts = 2;                    // half-precision values that an operand is split into
constexpr int kChunkBytes = kParts * 1024;   // packed weights of 16 k x 32 columns: [part][lane][8 k]
constexpr int kWaitLoads = 0x0f70;           // s_waitcnt vmcnt(0)

struct ChainProduct {
    int64_t at;                  // packed weights of type 0: [type][32 columns][16 k]
    int blocks, chunks;          // 32 columns, 16 k; multiples of 2 and 4
    int back_at;                 // column_back of the columns of type 0, an exponent's byte each: [type][column]
};
struct ChainArgs {
    const float* x[4];
    int n[4], tile_end[4];
    const char* packed;
    const float* fixed;          // per type: the hidden layers' biases one after the other, the output layer's weights, its bias
    const unsigned char* backs;
    ChainProduct p[kNetMaxLayers];       // the pass's products in its order
    float* act[kNetMaxLayers];           // activations of the hidden layers, or null: [tile][32 columns][32 rows][half a column block][lane][8]
    int act_blocks[kNetMaxLayers];       // their padded widths / 32
    int fixed_at[kNetMaxLayers + 2], fixed_size;
    int hidden, k0;
    unsigned absolute;
    float alpha, inv_alpha;
    float* value[4];
    const float* scale[4];
    float* grad[4];
    bool accumulate;
};

// 8 (v / 4) + 4 half + v % 4 is the matrix row of a lane's element v; the column of the weights that stands there, so that a lane has
// the columns 16 (v / 8) + 8 half + v % 8
__device__ __forceinline__ int column_of(int matrix_row)
{
    const int q = matrix_row >> 3, half = (matrix_row >> 2) & 1;
    return 16 * (q >> 1) + 8 * half + 4 * (q & 1) + (matrix_row & 3);
}

// The power of two that brings a row's or a column's largest value (its bits: never negative) to between 2^14 and 2^15, as it
// is multiplied by: rows, at most 2^111; columns, at least 2^-112 (from 2^128 (1 - 2^-11) on a weight becomes infinite, and NaN)
__device__ __forceinline__ float row_scale(unsigned largest) { return __uint_as_float((268u - max(largest >> 23, 30u)) << 23); }
__device__ __forceinline__ float column_scale(unsigned largest) { return __uint_as_float((268u - min(max(largest >> 23, 15u), 253u)) << 23); }
// what brings a sum of their products back is the product of the two inverses, a factor of 2^15 moved from the row's to the column's
// so that neither the factors nor the sum between them leave float32's range before row and product do
__device__ __forceinline__ float row_back(unsigned largest) { return __uint_as_float((max(largest >> 23, 30u) - 29u) << 23); }
__device__ __forceinline__ float column_back(unsigned largest) { return __uint_as_float((min(max(largest >> 23, 15u), 253u) + 1u) << 23); }

// a workgroup of kWaves wavefronts takes 32 kRB rows, and 32 kCB columns to a wavefront where a layer has as many
template <int kWaves, int kRB, int kCB>
struct ChainLds {
    static constexpr int kRows = 32 * kRB, kBlocks = kWaves * kCB;
    u4v planes[kParts][4 * kBlocks][kRows + 1];  // [part][8 columns][row]
    // the rows' largest values, as they come from products 0, 1, 2, 0, ...: of the operand in the planes, of the one that is being made,
    // and zeros for the one after
    unsigned largest[3][kRows];
    float sums[kBlocks][kRows];
    float fixed[kNetMaxLayers * 32 * kBlocks + 4];       // the type's biases and output layer
};

struct Lane {
    int lane, wave, l32, half;
};
// Chunks of weights on their way, of kCB column blocks `stride` bytes apart (0 where one block is all that is taken: the second load
// is of the same).
template <int kCB>
struct Ring {
    static constexpr int kDepth = kCB == 2 ? 2 : 4;      // (the same bytes; four chunks of two blocks do not fit the registers)
    u4v part[kDepth][kCB][kParts];
    __device__ __forceinline__ void load(int u, const char* chunk, int stride, unsigned lane16)
    {
#pragma unroll
        for (int c = 0; c < kCB; ++c)
#pragma unroll
            for (int m = 0; m < kParts; ++m) part[u][c][m] = *reinterpret_cast<const u4v*>(chunk + c * stride + m * 1024 + lane16);
    }
};
struct Source {
    const char* at;
    int stride;
};
template <int kCB>
__device__ __forceinline__ void start(Ring<kCB>& ring, const Source& from, unsigned lane16)
{
#pragma unroll
    for (int u = 0; u < Ring<kCB>::kDepth; ++u) ring.load(u, from.at + u * kChunkBytes, from.stride, lane16);
}

// Which part of a product a wavefront forms: CB blocks of 32 columns (from column block `cb`) of RB blocks of 32 rows (from block rb0).
struct Share {
    int cb, rb0;
    bool active;
};
// the layer's columns are so few that two wavefronts share them, a block of rows each
template <int kWaves, int kRB>
__device__ __forceinline__ bool by_rows(int blocks) { return kRB == 2 && 2 * blocks <= kWaves; }
// so many that a wavefront takes two blocks of them (the padded widths have an even number)
template <int kWaves, int kCB>
__device__ __forceinline__ bool by_pairs(int blocks) { return kCB == 2 && blocks > kWaves; }
template <int kWaves, int kRB, int kCB>
__device__ __forceinline__ Share share_of(int wave, int blocks)
{
    if (by_rows<kWaves, kRB>(blocks)) {
        const int rb0 = wave / blocks;
        return {wave - rb0 * blocks, min(rb0, kRB - 1), rb0 < kRB};
    }
    if (by_pairs<kWaves, kCB>(blocks)) return {min(2 * wave, blocks - 2), 0, 2 * wave < blocks};
    return {min(wave, blocks - 1), 0, wave < blocks};
}

// acc + 2^-11 low += the planes' columns from 8 first8 on (16 `chunks` of them) times the weights from `weights` on, whose first chunks
// are in the ring; `next`: the weights that come after these
template <int RB, int CB, class Lds, int kCB>
__device__ __forceinline__ void multiply(const Lds& S, const Lane& P, int first8, int rb0, int chunks, const Source& weights, const Source& next,
                                         Ring<kCB>& ring, f32x16 (&acc)[CB][RB], f32x16 (&low)[CB][RB])
{
    constexpr int kDepth = Ring<kCB>::kDepth;
    const unsigned lane16 = P.lane * 16;
    const auto group = [&](int c0) __attribute__((always_inline)) {
        const bool more = c0 + kDepth < chunks;
        const char* const ahead = more ? weights.at + (c0 + kDepth) * kChunkBytes : next.at;
        const int stride = more ? weights.stride : next.stride;
#pragma unroll
        for (int u = 0; u < kDepth; ++u) {
            h8v x[RB][kParts], w[CB][kParts];
#pragma unroll
            for (int j = 0; j < RB; ++j)
#pragma unroll
                for (int m = 0; m < kParts; ++m) x[j][m] = __builtin_bit_cast(h8v, S.planes[m][first8 + 2 * (c0 + u) + P.half][32 * (rb0 + j) + P.l32]);
#pragma unroll
            for (int c = 0; c < CB; ++c)
#pragma unroll
                for (int m = 0; m < kParts; ++m) w[c][m] = __builtin_bit_cast(h8v, ring.part[u][c][m]);
            const auto mul = [&](f32x16 (&to)[CB][RB], int xi, int wi) {
#pragma unroll
                for (int c = 0; c < CB; ++c)
#pragma unroll
                    for (int j = 0; j < RB; ++j) to[c][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(w[c][wi], x[j][xi], to[c][j], 0, 0, 0);
            };
            mul(low, 1, 0);
            mul(acc, 0, 0);
            mul(low, 0, 1);
            ring.load(u, ahead + u * kChunkBytes, stride, lane16);
            // the loads stay behind the chunk's products (vector, scalar and LDS instructions may pass): the compiler would gather
            // them behind the last one
            __builtin_amdgcn_sched_barrier(0x386);
        }
    };
    // (the first chunks apart: they have come, and wait for nothing that was asked for or stored after them)
    group(0);
#pragma unroll 1
    for (int c = kDepth; c < chunks; c += kDepth) group(c);
}

// the largest of a lane's values of a layer, to those of their rows
template <int RB, class Lds>
__device__ __forceinline__ void note_largest(Lds& S, const Lane& P, int product, int rb0, const f32x16 (&y)[RB])
{
#pragma unroll
    for (int j = 0; j < RB; ++j) {
        float m[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int v = 0; v < 16; ++v) m[v & 3] = fmaxf(m[v & 3], fabsf(y[j][v]));
        atomicMax(&S.largest[product % 3][32 * (rb0 + j) + P.l32], __float_as_uint(fmaxf(fmaxf(m[0], m[1]), fmaxf(m[2], m[3]))));
    }
}
// a lane's values of a layer -> the planes, scaled and split
template <int RB, class Lds>
__device__ __forceinline__ void to_planes(Lds& S, const Lane& P, int product, int cb, int rb0, const f32x16 (&y)[RB])
{
#pragma unroll
    for (int j = 0; j < RB; ++j) {
        const float scale = row_scale(S.largest[product % 3][32 * (rb0 + j) + P.l32]);
#pragma unroll
        for (int g = 0; g < 2; ++g) {
            u4v p[kParts];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                unsigned q[kParts];
                split_pair(y[j][8 * g + 2 * e] * scale, y[j][8 * g + 2 * e + 1] * scale, q[0], q[1]);
                p[0][e] = q[0], p[1][e] = q[1];
            }
#pragma unroll
            for (int m = 0; m < kParts; ++m) S.planes[m][4 * cb + 2 * g + P.half][32 * (rb0 + j) + P.l32] = p[m];
        }
    }
}

template <int RB>
struct Blocks {
    f32x16 v[RB];
};
// a lane's sixteen values of a block in the activations' order in memory
__device__ __forceinline__ void load_block(const float* block, const Lane& P, f32x16& v)
{
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const f4v f = *reinterpret_cast<const f4v*>(block + (q >> 1) * 512 + P.lane * 8 + (q & 1) * 4);
#pragma unroll
        for (int e = 0; e < 4; ++e) v[4 * q + e] = f[e];
    }
}
__device__ __forceinline__ void store_block(float* block, const Lane& P, const f32x16& v)
{
#pragma unroll
    for (int q = 0; q < 4; ++q)
        *reinterpret_cast<f4v*>(block + (q >> 1) * 512 + P.lane * 8 + (q & 1) * 4) = f4v{v[4 * q], v[4 * q + 1], v[4 * q + 2], v[4 * q + 3]};
}
// a lane's sixteen columns of a vector over the layer's columns
__device__ __forceinline__ f32x16 of_columns(const float* from, const Lane& P, int cb)
{
    f32x16 v;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const f4v f = *reinterpret_cast<const f4v*>(from + 32 * cb + 16 * (q >> 1) + 8 * P.half + 4 * (q & 1));
#pragma unroll
        for (int e = 0; e < 4; ++e) v[4 * q + e] = f[e];
    }
    return v;
}
// column_back of a lane's sixteen columns
struct Backs {
    u2v q[2];
    __device__ __forceinline__ void load(const unsigned char* from, const Lane& P, int cb)
    {
#pragma unroll
        for (int g = 0; g < 2; ++g) q[g] = *reinterpret_cast<const u2v*>(from + 32 * cb + 16 * g + 8 * P.half);
    }
    __device__ __forceinline__ float operator[](int v) const { return __uint_as_float(((q[v >> 3][(v >> 2) & 1] >> (8 * (v & 3))) & 0xffu) << 23); }
};
__device__ __forceinline__ float slope_of(float a, float inv_alpha) { return a >= 0.f ? 1.f : fmaf(a, inv_alpha, 1.f); }

// wavefronts per SIMD: two workgroups of four wavefronts with 64 rows on a compute unit (82 KB each for 256 columns, all there is), and
// with 32 rows two of eight and four of four
constexpr int chain_waves(int rb) { return rb == 2 ? 2 : 4; }

template <int kWaves, int kRB, int kCB, bool kBack>
__global__ __launch_bounds__(64 * kWaves) __attribute__((amdgpu_waves_per_eu(chain_waves(kRB), chain_waves(kRB))))
void chain_kernel(const ChainArgs a)
{
    typedef ChainLds<kWaves, kRB, kCB> Lds;
    constexpr int kRows = Lds::kRows, kBlocks = Lds::kBlocks, kThreads = 64 * kWaves;
    __shared__ Lds S;
    float* const fixed = S.fixed;
    const int tid = threadIdx.x;
    const Lane P = {tid & 63, __builtin_amdgcn_readfirstlane(tid >> 6), tid & 31, (tid >> 5) & 1};
    const unsigned lane16 = P.lane * 16;
    const int tile = static_cast<int>(blockIdx.x);
    const int t = (tile >= a.tile_end[0]) + (tile >= a.tile_end[1]) + (tile >= a.tile_end[2]);
    const int row0 = (tile - (t == 0 ? 0 : a.tile_end[t - 1])) * kRows, n = a.n[t], H = a.hidden, k0 = a.k0;
    const float alpha = a.alpha, inv_alpha = a.inv_alpha;
    // a wavefront's weights of the column blocks of a product from cb0 on
    const auto source_of = [&](const ChainProduct& p, int cb0) __attribute__((always_inline)) {
        const int blocks = min(p.blocks - cb0, kBlocks), size = p.chunks * kChunkBytes;
        const int cb = cb0 + share_of<kWaves, kRB, kCB>(P.wave, blocks).cb;
        return Source{a.packed + p.at + (static_cast<int64_t>(t) * p.blocks + cb) * size, by_pairs<kWaves, kCB>(blocks) ? size : 0};
    };
    const auto act_at = [&](int h, int cb, int rb) __attribute__((always_inline)) -> float* {
        return a.act[h] + (static_cast<size_t>(tile) * a.act_blocks[h] + cb) * kRB * 1024 + rb * 1024;
    };
    Ring<kCB> ring;
    start(ring, source_of(a.p[0], 0), lane16);
    for (int i = tid; i < 3 * kRows; i += kThreads) S.largest[0][i] = 0u;
    for (int i = tid; i < a.fixed_size; i += kThreads) fixed[i] = a.fixed[static_cast<size_t>(t) * a.fixed_size + i];

    // product l, column blocks from `cb0` on, in one of the shares; `operands(multiply)` may call it more than once.  `finish` has the
    // sums but for the columns' factors.
    const auto run = [&](auto rb_count, auto cb_count, int l, int cb0, auto&& before, auto&& operands, auto&& finish) __attribute__((always_inline)) {
        constexpr int RB = decltype(rb_count)::value, CB = decltype(cb_count)::value;
        const ChainProduct& p = a.p[l];
        const int blocks = min(p.blocks - cb0, kBlocks);
        const Share s = share_of<kWaves, kRB, kCB>(P.wave, blocks);
        const Source weights = source_of(p, cb0);
        Source next = weights;
        if (cb0 + kBlocks < p.blocks) next = source_of(p, cb0 + kBlocks);
        else if (l + 1 < H) next = source_of(a.p[l + 1], 0);
        f32x16 acc[CB][RB], low[CB][RB];
#pragma unroll
        for (int c = 0; c < CB; ++c)
#pragma unroll
            for (int j = 0; j < RB; ++j) acc[c][j] = low[c][j] = f32x16(0.f);
        Backs back[CB];
#pragma unroll
        for (int c = 0; c < CB; ++c) back[c].load(a.backs + p.back_at + 32 * (t * p.blocks + cb0), P, s.cb + c);
        auto met = before(rb_count, s);
        operands(p, s, [&](int first8, int first, int chunks) __attribute__((always_inline)) {
            if (s.active) {
                const Source from = {weights.at + first * kChunkBytes, weights.stride};
                const Source then = first + chunks < p.chunks ? Source{from.at + chunks * kChunkBytes, weights.stride} : next;
                multiply<RB, CB>(S, P, first8, s.rb0, chunks, from, then, ring, acc, low);
            }
        });
        if (!s.active) start(ring, next, lane16);
#pragma unroll
        for (int j = 0; j < RB; ++j) {
            const float rows_back = row_back(S.largest[l % 3][32 * (s.rb0 + j) + P.l32]);
#pragma unroll
            for (int c = 0; c < CB; ++c)
#pragma unroll
                for (int v = 0; v < 16; ++v) acc[c][j][v] = fmaf(low[c][j][v], kResidualBack, acc[c][j][v]) * rows_back;
        }
        finish(s, cb0, acc, back, met);
    };
    const auto run_any = [&](int l, int cb0, auto&& before, auto&& operands, auto&& finish) __attribute__((always_inline)) {
        const int blocks = min(a.p[l].blocks - cb0, kBlocks);
        if constexpr (kCB == 2) {
            if (by_pairs<kWaves, kCB>(blocks)) return run(std::integral_constant<int, kRB>(), std::integral_constant<int, 2>(), l, cb0, before, operands, finish);
        }
        if constexpr (kRB == 2) {
            if (by_rows<kWaves, kRB>(blocks)) return run(std::integral_constant<int, 1>(), std::integral_constant<int, 1>(), l, cb0, before, operands, finish);
        }
        run(std::integral_constant<int, kRB>(), std::integral_constant<int, 1>(), l, cb0, before, operands, finish);
    };
    // (product's place was last read as that of the operand of product - 3, which every wavefront is through with)
    const auto clear_largest = [&](int product) {
        if (tid < kRows) S.largest[product % 3][tid] = 0u;
    };
    const auto nothing = [](auto, const Share&) { return 0; };
    const auto from_planes = [&](const ChainProduct& p, const Share&, auto&& mul) { mul(0, 0, p.chunks); };

    if constexpr (!kBack) {
        // ---- layer 1: the feature rows through the planes piece by piece (the compute unit's other workgroups have the time it takes)
        constexpr int kPiece = 32 * kWaves, kUnits = kRows * kPiece / 8 / kThreads;       // 8 columns of a row
        const auto place = [&](int i, int& row, int& k8) {
            const int unit = tid + i * kThreads, rest = unit >> 3;
            row = rest % kRows;
            k8 = (unit & 7) + 8 * (rest / kRows);
        };
        const auto fetch = [&](int i, int piece, f4v (&x)[2]) __attribute__((always_inline)) {
            int row, k8;
            place(i, row, k8);
            const int column = min(piece * kPiece + 8 * k8, k0 - 8);           // (past the end: others again, not read)
            const float* const from = a.x[t] + static_cast<size_t>(min(row0 + row, n - 1)) * k0 + column;
            x[0] = *reinterpret_cast<const f4v*>(from);
            x[1] = *reinterpret_cast<const f4v*>(from + 4);
        };
        const auto stage = [&](int i, const f4v (&x)[2]) {
            int row, k8;
            place(i, row, k8);
            const float scale = row_scale(S.largest[0][row]);
            u4v p[kParts];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                unsigned q[kParts];
                split_pair(x[e >> 1][2 * (e & 1)] * scale, x[e >> 1][2 * (e & 1) + 1] * scale, q[0], q[1]);
                p[0][e] = q[0], p[1][e] = q[1];
            }
#pragma unroll
            for (int m = 0; m < kParts; ++m) S.planes[m][k8][row] = p[m];
        };
        // the rows' largest values before anything of them is split: a reading more, of which the second finds the lines in the L2
        __syncthreads();
#pragma unroll 3
        for (int piece = 0; piece < (k0 + kPiece - 1) / kPiece; ++piece)
#pragma unroll
            for (int i = 0; i < kUnits; ++i) {
                f4v x[2];
                int row, k8;
                place(i, row, k8);
                fetch(i, piece, x);
                float m = 0.f;
#pragma unroll
                for (int e = 0; e < 8; ++e) m = fmaxf(m, fabsf(x[e >> 2][e & 3]));
                atomicMax(&S.largest[0][row], __float_as_uint(m));
            }
        __syncthreads();
        const auto through_pieces = [&](const ChainProduct&, const Share&, auto&& mul) __attribute__((always_inline)) {
#pragma unroll 1
            for (int piece = 0; piece * kPiece < k0; ++piece) {
                if (piece > 0) __syncthreads();         // the planes have been read
#pragma unroll
                for (int i = 0; i < kUnits; ++i) {
                    f4v x[2];
                    fetch(i, piece, x);
                    stage(i, x);
                }
                __syncthreads();
                mul(0, piece * (kPiece / 16), min(kPiece, k0 - piece * kPiece) / 16);
            }
        };
        const auto layer = [&](int l, auto&& operands) __attribute__((always_inline)) {
            run_any(l, 0, nothing, operands, [&](const Share& s, int, auto& y, const auto& back, int) __attribute__((always_inline)) {
                constexpr int CB = std::extent<std::remove_reference_t<decltype(y)>, 0>::value, RB = std::extent<std::remove_reference_t<decltype(y)>, 1>::value;
                if (s.active) {
                    const bool absolute = (a.absolute >> l) & 1u;
#pragma unroll
                    for (int c = 0; c < CB; ++c) {
                        const f32x16 bias = of_columns(fixed + a.fixed_at[l], P, s.cb + c);
#pragma unroll
                        for (int j = 0; j < RB; ++j) {
                            if (absolute) {
#pragma unroll
                                for (int v = 0; v < 16; ++v) y[c][j][v] = celu_absolute(fmaf(y[c][j][v], back[c][v], bias[v]), alpha, inv_alpha);
                            } else {
#pragma unroll
                                for (int v = 0; v < 16; ++v) y[c][j][v] = celu_exact(fmaf(y[c][j][v], back[c][v], bias[v]), alpha, inv_alpha);
                            }
                        }
                        if (l + 1 < H) note_largest<RB>(S, P, l + 1, s.rb0, y[c]);
                    }
                }
                clear_largest(l + 2);
                __syncthreads();           // the planes have been read, the rows' largest values are there
                if (s.active) {
                    if (l + 1 < H) {
#pragma unroll
                        for (int c = 0; c < CB; ++c) to_planes<RB>(S, P, l + 1, s.cb + c, s.rb0, y[c]);
                    } else {
#pragma unroll
                        for (int c = 0; c < CB; ++c) {
                            const f32x16 w = of_columns(fixed + a.fixed_at[H], P, s.cb + c);
#pragma unroll
                            for (int j = 0; j < RB; ++j) {
                                float part[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
                                for (int v = 0; v < 16; ++v) part[v & 3] = fmaf(y[c][j][v], w[v], part[v & 3]);
                                float sum = (part[0] + part[1]) + (part[2] + part[3]);
                                sum += __shfl_xor(sum, 32, 64);
                                if (P.half == 0) S.sums[s.cb + c][32 * (s.rb0 + j) + P.l32] = sum;
                            }
                        }
                    }
                    if (a.act[l]) {
                        // loads and stores are waited for in the order they were issued: the next layer's first weights have to be
                        // there before the stores go out, which then have those chunks' time
                        __builtin_amdgcn_s_waitcnt(kWaitLoads);
#pragma unroll
                        for (int c = 0; c < CB; ++c)
#pragma unroll
                            for (int j = 0; j < RB; ++j) store_block(act_at(l, s.cb + c, s.rb0 + j), P, y[c][j]);
                    }
                }
                __syncthreads();
            });
        };
        layer(0, through_pieces);
#pragma unroll 1
        for (int l = 1; l < H; ++l) layer(l, from_planes);
        if (tid < kRows && row0 + tid < n) {
            float sum = 0.f;
            for (int cb = 0; cb < a.act_blocks[H - 1]; ++cb) sum += S.sums[cb][tid];
            a.value[t][row0 + tid] = sum + fixed[a.fixed_at[H + 1]];
        }
    } else {
        // ---- d_L = w celu'(a_L)
        __syncthreads();
        f32x16 d[kRB * kCB][1];
#pragma unroll
        for (int i = 0; i < kRB * kCB; ++i) {
            const int u = P.wave + i * kWaves, cb = u / kRB, rb = u - cb * kRB;
            if (cb >= a.act_blocks[H - 1]) break;
            load_block(act_at(H - 1, cb, rb), P, d[i][0]);
            const f32x16 w = of_columns(fixed + a.fixed_at[H], P, cb);
#pragma unroll
            for (int v = 0; v < 16; ++v) d[i][0][v] = w[v] * slope_of(d[i][0][v], inv_alpha);
            note_largest<1>(S, P, 0, rb, d[i]);
        }
        __syncthreads();
#pragma unroll
        for (int i = 0; i < kRB * kCB; ++i) {
            const int u = P.wave + i * kWaves, cb = u / kRB, rb = u - cb * kRB;
            if (cb >= a.act_blocks[H - 1]) break;
            to_planes<1>(S, P, 0, cb, rb, d[i]);
        }
        __syncthreads();
        // ---- d_{L-1} .. d_1
#pragma unroll 1
        for (int l = 0; l + 1 < H; ++l) {
            const int h = H - 2 - l;               // the hidden layer whose activations are met
            // (of a second column block they are asked for when the first one's are met: there are no registers for them before)
            const auto activations = [&](auto rb_count, const Share& s) {
                constexpr int RB = decltype(rb_count)::value;
                Blocks<RB> act;
#pragma unroll
                for (int j = 0; j < RB; ++j) load_block(act_at(h, s.cb, s.rb0 + j), P, act.v[j]);
                return act;
            };
            run_any(l, 0, activations, from_planes, [&](const Share& s, int, auto& y, const auto& back, auto& act) {
                constexpr int CB = std::extent<std::remove_reference_t<decltype(y)>, 0>::value, RB = std::extent<std::remove_reference_t<decltype(y)>, 1>::value;
                const auto meet = [&](int c, const Blocks<RB>& with) {
#pragma unroll
                    for (int j = 0; j < RB; ++j)
#pragma unroll
                        for (int v = 0; v < 16; ++v) y[c][j][v] = y[c][j][v] * back[c][v] * slope_of(with.v[j][v], inv_alpha);
                };
                if constexpr (CB == 2) {
                    Blocks<RB> second;
#pragma unroll
                    for (int j = 0; j < RB; ++j) load_block(act_at(h, s.cb + 1, s.rb0 + j), P, second.v[j]);
                    meet(0, act);
                    meet(1, second);
                } else {
                    meet(0, act);
                }
                if (s.active)
#pragma unroll
                    for (int c = 0; c < CB; ++c) note_largest<RB>(S, P, l + 1, s.rb0, y[c]);
                clear_largest(l + 2);
                __syncthreads();           // the planes have been read, the rows' largest values are there
                if (s.active)
#pragma unroll
                    for (int c = 0; c < CB; ++c) to_planes<RB>(S, P, l + 1, s.cb + c, s.rb0, y[c]);
                __syncthreads();
            });
        }
        // ---- the rows
#pragma unroll 1
        for (int cb0 = 0; cb0 < a.p[H - 1].blocks; cb0 += kBlocks) {
            run_any(H - 1, cb0, nothing, from_planes, [&](const Share& s, int cb0, auto& y, const auto& back, int) {
                constexpr int CB = std::extent<std::remove_reference_t<decltype(y)>, 0>::value, RB = std::extent<std::remove_reference_t<decltype(y)>, 1>::value;
                if (!s.active) return;
#pragma unroll
                for (int j = 0; j < RB; ++j) {
                    const int r = row0 + 32 * (s.rb0 + j) + P.l32;
                    const float scale = a.scale[t] ? a.scale[t][min(r, n - 1)] : 1.f;
#pragma unroll
                    for (int c = 0; c < CB; ++c) {
                        float* const out = a.grad[t] + static_cast<size_t>(min(r, n - 1)) * k0 + 32 * (cb0 + s.cb + c) + 8 * P.half;
                        f4v v[4];
#pragma unroll
                        for (int q = 0; q < 4; ++q)
#pragma unroll
                            for (int e = 0; e < 4; ++e) v[q][e] = y[c][j][4 * q + e] * back[c][4 * q + e] * scale;
                        if (a.accumulate) {
#pragma unroll
                            for (int q = 0; q < 4; ++q) v[q] += *reinterpret_cast<const f4v*>(out + 16 * (q >> 1) + 4 * (q & 1));
                        }
                        if (r < n) {
#pragma unroll
                            for (int q = 0; q < 4; ++q) *reinterpret_cast<f4v*>(out + 16 * (q >> 1) + 4 * (q & 1)) = v[q];
                        }
                    }
                }
            });
        }
    }
}

// The weights of all products, scaled by columns, split and in the order in which the lanes take them, and the padded biases; a workgroup
// per 32 columns, which it holds between their largest values and the split where a column has no more than 512 (all loads are then on
// their way at once).
constexpr int kPackWaves = 8, kPackHeld = 4;         // chunks of a wavefront
struct PackProduct {
    const float* w[4];           // [k, n_out] as stored, or [n_out, k] (back)
    int k, n_out, blocks, chunks, end;       // end: running number of column blocks of all types
    bool back;
    int64_t at;
    int back_at;
};
struct PackArgs {
    PackProduct p[2 * kNetMaxLayers];
    const float *bias[kNetMaxLayers][4];
    int products, layers, widths[kNetMaxLayers + 1], fixed_at[kNetMaxLayers + 2], fixed_size;
    char* packed;
    float* fixed;
    unsigned char* backs;
    const float* top[4];
};
__global__ __launch_bounds__(64 * kPackWaves) void chain_pack_kernel(const PackArgs a)
{
    constexpr int kThreads = 64 * kPackWaves;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), number = static_cast<int>(blockIdx.x);
    if (number >= a.p[a.products - 1].end) {
        // behind the weights: the biases, a value to a thread
        const int i = (number - a.p[a.products - 1].end) * kThreads + static_cast<int>(threadIdx.x), t = i / a.fixed_size, at = i - t * a.fixed_size;
        if (t >= 4) return;
        float v = 0.f;
        const int H = a.layers - 1;
        if (at >= a.fixed_at[H + 1]) {
            if (at == a.fixed_at[H + 1] && a.bias[H][t]) v = a.bias[H][t][0];
        } else {
            int l = 0;
            while (at >= a.fixed_at[l + 1]) ++l;
            const int c = at - a.fixed_at[l];
            const float* const from = l < H ? a.bias[l][t] : a.top[t];
            if (from && c < a.widths[min(l + 1, H)]) v = from[c];
        }
        a.fixed[i] = v;
        return;
    }
    __shared__ unsigned largest[32];
    if (threadIdx.x < 32) largest[threadIdx.x] = 0u;
    __syncthreads();
    int m = 0;
    while (number >= a.p[m].end) ++m;
    const PackProduct& p = a.p[m];
    const int rel = number - (m == 0 ? 0 : a.p[m - 1].end), t = rel / p.blocks, cb = rel - t * p.blocks;
    const int col = 32 * cb + column_of(lane & 31);
    const float* const w = p.w[t];
    const bool wide = p.back && p.k % 8 == 0 && (reinterpret_cast<uintptr_t>(w) & 15u) == 0;      // sixteen bytes at a time
    float v[kPackHeld][8];
    const auto fetch = [&](int first) {
#pragma unroll
        for (int i = 0; i < kPackHeld; ++i) {
            const int k0 = 16 * (first + i * kPackWaves + wave) + 8 * (lane >> 5);
            if (wide) {
                const bool inside = w && col < p.n_out && k0 < p.k;          // (a type without rows has no weights)
                const f4v* const from = reinterpret_cast<const f4v*>(w + static_cast<size_t>(col) * p.k + k0);
#pragma unroll
                for (int q = 0; q < 2; ++q) {
                    const f4v x = inside ? from[q] : f4v(0.f);
#pragma unroll
                    for (int e = 0; e < 4; ++e) v[i][4 * q + e] = x[e];
                }
            } else {
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    const bool inside = w && col < p.n_out && k0 + e < p.k;
                    const size_t at = p.back ? static_cast<size_t>(col) * p.k + k0 + e : static_cast<size_t>(k0 + e) * p.n_out + col;
                    v[i][e] = inside ? w[at] : 0.f;
                }
            }
        }
    };
    constexpr int kGroup = kPackWaves * kPackHeld;
    float most = 0.f;
#pragma unroll 1
    for (int first = 0; first < p.chunks; first += kGroup) {
        fetch(first);
#pragma unroll
        for (int i = 0; i < kPackHeld; ++i)
#pragma unroll
            for (int e = 0; e < 8; ++e) most = fmaxf(most, fabsf(v[i][e]));
    }
    atomicMax(&largest[lane & 31], __float_as_uint(most));
    __syncthreads();
    const unsigned of_column = largest[lane & 31];
    const float scale = column_scale(of_column);
    if (wave == 0 && lane < 32) a.backs[p.back_at + 32 * rel + column_of(lane)] = static_cast<unsigned char>(__float_as_uint(column_back(of_column)) >> 23);
#pragma unroll 1
    for (int first = 0; first < p.chunks; first += kGroup) {
        if (p.chunks > kGroup) fetch(first);
#pragma unroll
        for (int i = 0; i < kPackHeld; ++i) {
            const int c = first + i * kPackWaves + wave;
            if (c >= p.chunks) break;
            u4v part[kParts];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                unsigned q[kParts];
                split_pair(v[i][2 * e] * scale, v[i][2 * e + 1] * scale, q[0], q[1]);
                part[0][e] = q[0], part[1][e] = q[1];
            }
            char* const to = a.packed + p.at + (static_cast<int64_t>(rel) * p.chunks + c) * kChunkBytes + lane * 16;
#pragma unroll
            for (int q = 0; q < kParts; ++q) *reinterpret_cast<u4v*>(to + q * 1024) = part[q];
        }
    }
}

// ---- host
int padded(int width) { return (width + 63) / 64 * 64; }

// 32 or 64 rows to a workgroup.  64 halve the weights' way from the L2, and are the faster form of full rounds (wide layers: 155 us forward
// for 512 tiles, 81 for half of their rows with 32; deep networks, 497 tiles, 418 us and 468 with 32, 442 tiles 409 and 449), but a last
// round that is not full takes nearly as long as a full one with 64 (368 tiles 375 us, with 32 354).  So with wide layers the full rounds are
// of 64 rows, and what is left, where it is no more than three quarters of a round, is a launch of its own with 32 (737 tiles with
// charges 1,196 us, all with 32 1,250; 644 tiles without 608 and 628).  Layers of up to 128 columns gain less from 64 rows (default networks
// with charges on 40,000 molecules, 14 rounds, 2,757 us and 2,830 with 32; 497 tiles 315 and 321) and lose as much to a round
// that is not full (736 tiles 427 and 396; divided 428): one form, of 64 where that round is more than half full or one of many.
struct Part {
    int rb, tiles, tile_end[4], first[4], n[4];          // rows first .. first + n of a type
    int64_t act_at[kNetMaxLayers];
};
constexpr int kRound = 512;                              // tiles of 64 rows that the chip holds

struct Layout {
    int hidden, parts;
    Part part[2];
    bool wide;                   // more than 128 columns: 64 to a wavefront of four, or of 32 rows 32 to one of eight
    ChainProduct f[kNetMaxLayers], r[kNetMaxLayers];
    int64_t fixed_bytes_at, backs_bytes_at, bytes;
    int fixed_at[kNetMaxLayers + 2], fixed_size, act_blocks[kNetMaxLayers];

    explicit Layout(const NetChain& net) : hidden(net.hidden), parts(0)
    {
        int widest = 0;
        for (int l = 1; l <= hidden; ++l) widest = std::max(widest, net.widths[l]);
        wide = widest > 128;
        // (the last chunks' places are loaded from ahead of need)
        int64_t at = 0;
        int backs = 0;
        const auto product = [&](int k, int n_out) {
            const ChainProduct p = {at, padded(n_out) / 32, padded(k) / 16, backs};
            at += 4ll * p.blocks * p.chunks * kChunkBytes;
            backs += 4 * p.blocks * 32;
            return p;
        };
        for (int l = 0; l < hidden; ++l) f[l] = product(net.widths[l], net.widths[l + 1]);
        for (int l = 0; l < hidden && net.want_rows; ++l) r[l] = product(net.widths[hidden - l], net.widths[hidden - l - 1]);
        fixed_size = 0;
        for (int l = 0; l < hidden; ++l) {
            fixed_at[l] = fixed_size;
            fixed_size += padded(net.widths[l + 1]);
        }
        fixed_at[hidden] = fixed_size;
        fixed_at[hidden + 1] = fixed_size += padded(net.widths[hidden]);
        fixed_size += 4;
        fixed_bytes_at = at;
        at += (4ll * fixed_size * 4 + 255) / 256 * 256;
        backs_bytes_at = at;
        at += (backs + 255) / 256 * 256;
        for (int l = 0; l < hidden; ++l) act_blocks[l] = padded(net.widths[l + 1]) / 32;

        int64_t tiles64 = 0;
        for (int t = 0; t < 4; ++t) tiles64 += (net.n[t] + 63) / 64;
        const int64_t last = tiles64 % kRound;
        int64_t full = last > kRound / 4 * 3 ? tiles64 : tiles64 - last;       // tiles of 64 rows
        if (!wide) full = last == 0 || last > kRound / 2 || tiles64 >= 8 * kRound ? tiles64 : 0;
        int done[4] = {0, 0, 0, 0};
        const auto add = [&](int rb, int64_t most) {
            Part& p = part[parts++];
            p.rb = rb;
            p.tiles = 0;
            for (int t = 0; t < 4; ++t) {
                const int64_t tiles = std::min<int64_t>((net.n[t] - done[t] + 32 * rb - 1) / (32 * rb), most - p.tiles);
                p.first[t] = done[t];
                p.n[t] = static_cast<int>(std::min<int64_t>(net.n[t] - done[t], tiles * 32 * rb));
                p.tile_end[t] = p.tiles += static_cast<int>(tiles);
                done[t] += p.n[t];
            }
            for (int l = 0; l < hidden && net.want_rows; ++l) {
                p.act_at[l] = at;
                at += static_cast<int64_t>(p.tiles) * act_blocks[l] * rb * 4096;
            }
        };
        if (full > 0) add(2, full);
        if (full < tiles64) add(1, INT_MAX);
        bytes = at + 16;
    }
};

template <int kWaves, int kRB, int kCB, bool kBack>
hipError_t launch(const ChainArgs& a, int tiles, hipStream_t stream)
{
    chain_kernel<kWaves, kRB, kCB, kBack><<<dim3(static_cast<unsigned>(tiles)), dim3(64 * kWaves), 0, stream>>>(a);
    return hipGetLastError();
}
// one part after the other
template <bool kBack>
hipError_t launch_parts(const NetChain& net, const Layout& L, const void* workspace, float* const value[4], const float* const scale[4], float* const grad[4],
                        bool accumulate, hipStream_t stream)
{
    char* const ws = static_cast<char*>(const_cast<void*>(workspace));
    ChainArgs a = {};
    a.packed = ws;
    a.fixed = reinterpret_cast<const float*>(ws + L.fixed_bytes_at);
    a.backs = reinterpret_cast<const unsigned char*>(ws + L.backs_bytes_at);
    std::copy(kBack ? L.r : L.f, (kBack ? L.r : L.f) + L.hidden, a.p);
    std::copy(L.act_blocks, L.act_blocks + L.hidden, a.act_blocks);
    std::copy(L.fixed_at, L.fixed_at + kNetMaxLayers + 2, a.fixed_at);
    a.fixed_size = L.fixed_size;
    a.hidden = L.hidden;
    a.k0 = net.widths[0];
    a.absolute = net.absolute;
    a.alpha = net.alpha;
    a.inv_alpha = 1.0f / net.alpha;
    a.accumulate = accumulate;
    for (int i = 0; i < L.parts; ++i) {
        const Part& p = L.part[i];
        for (int l = 0; l < L.hidden; ++l) a.act[l] = net.want_rows ? reinterpret_cast<float*>(ws + p.act_at[l]) : nullptr;
        for (int t = 0; t < 4; ++t) {
            const size_t first = p.first[t], rows = first * net.widths[0];
            a.n[t] = p.n[t];
            a.tile_end[t] = p.tile_end[t];
            a.x[t] = p.n[t] > 0 ? net.x[t] + rows : nullptr;
            a.value[t] = value && p.n[t] > 0 ? value[t] + first : nullptr;
            a.scale[t] = scale && p.n[t] > 0 && scale[t] ? scale[t] + first : nullptr;
            a.grad[t] = grad && p.n[t] > 0 ? grad[t] + rows : nullptr;
        }
        const hipError_t e = L.wide ? p.rb == 2 ? launch<4, 2, 2, kBack>(a, p.tiles, stream) : launch<8, 1, 1, kBack>(a, p.tiles, stream)
                                    : p.rb == 2 ? launch<4, 2, 1, kBack>(a, p.tiles, stream) : launch<4, 1, 1, kBack>(a, p.tiles, stream);
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

}  // namespace

bool net_chain_fits(const int* widths, int hidden)
{
    if (hidden < 1 || hidden >= kNetMaxLayers || widths[0] <= 0 || widths[0] % kChainPiece) return false;
    for (int l = 1; l <= hidden; ++l)
        if (widths[l] < 1 || widths[l] > kChainWidth) return false;
    return true;
}

size_t net_chain_workspace(const NetChain& net) { return static_cast<size_t>(Layout(net).bytes); }

hipError_t launch_net_chain_values(const NetChain& net, void* workspace, float* const value[4], hipStream_t stream)
{
    const Layout L(net);
    if (L.parts == 0) return hipSuccess;
    PackArgs p = {};
    int end = 0;
    for (int back = 0; back < (net.want_rows ? 2 : 1); ++back)
        for (int l = 0; l < L.hidden; ++l) {
            PackProduct& q = p.p[p.products++];
            const ChainProduct& c = back ? L.r[l] : L.f[l];
            const int layer = back ? L.hidden - 1 - l : l;
            for (int t = 0; t < 4; ++t) q.w[t] = net.n[t] > 0 ? net.w[layer][t] : nullptr;
            q.k = net.widths[back ? layer + 1 : layer];
            q.n_out = net.widths[back ? layer : layer + 1];
            q.blocks = c.blocks;
            q.chunks = c.chunks;
            q.back = back != 0;
            q.at = c.at;
            q.back_at = c.back_at;
            q.end = end += 4 * c.blocks;
        }
    for (int l = 0; l <= L.hidden; ++l)
        for (int t = 0; t < 4; ++t) p.bias[l][t] = net.n[t] > 0 ? net.b[l][t] : nullptr;
    for (int t = 0; t < 4; ++t) p.top[t] = net.n[t] > 0 ? net.w[L.hidden][t] : nullptr;
    p.layers = L.hidden + 1;
    std::copy(net.widths, net.widths + kNetMaxLayers + 1, p.widths);
    std::copy(L.fixed_at, L.fixed_at + kNetMaxLayers + 2, p.fixed_at);
    p.fixed_size = L.fixed_size;
    p.packed = static_cast<char*>(workspace);
    p.fixed = reinterpret_cast<float*>(p.packed + L.fixed_bytes_at);
    p.backs = reinterpret_cast<unsigned char*>(p.packed + L.backs_bytes_at);
    chain_pack_kernel<<<dim3(static_cast<unsigned>(end + (4 * L.fixed_size + 64 * kPackWaves - 1) / (64 * kPackWaves))), dim3(64 * kPackWaves), 0, stream>>>(p);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    return launch_parts<false>(net, L, workspace, value, nullptr, nullptr, false, stream);
}

hipError_t launch_net_chain_rows(const NetChain& net, const void* workspace, const float* const scale[4], float* const grad[4], bool accumulate,
                                 hipStream_t stream)
{
    const Layout L(net);
    if (L.parts == 0) return hipSuccess;
    return launch_parts<true>(net, L, workspace, nullptr, scale, grad, accumulate, stream);
}

}  // namespace khan
