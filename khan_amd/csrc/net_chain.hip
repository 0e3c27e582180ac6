// Inference of float32 networks with CELU of up to twelve layers (khan/model/nn.py:38-68, khan/inference/energy_server.py:121-123), for
// the four atom types: all layers of the forward pass in one launch, and all layers of the way back to the feature rows in another.
// With the names of net_layers.hip, a_l = celu(a_{l-1} W_l + b_l), value = a_L w + b; d_L = w celu'(a_L), d_{l-1} = (d_l W_l^T)
// celu'(a_{l-1}), row gradient = s d_1 W_1^T.
//
// The products are those of layer_split_kernel (net_layers.hip): every operand the exact sum of three bfloat16 values, the six
// largest of the nine partial products accumulated in float32, the five small ones in accumulators of their own.  What differs is
// where the operands come from.  Layer by layer, the tiles of a launch run side by side, first all waiting for their rows, then
// all multiplying, then all storing: 43-49 us for 47,000 rows 256 -> 256, of which the products need 19.  Here a workgroup takes 64 (or
// 32) rows through all layers: the rows of the next product are split once, by the lanes that have just formed them, into three planes
// in LDS (98 KB for 64 rows of 256), and the weights, split and packed beforehand by a launch of their own, go from memory straight to
// registers, four chunks of 16 k ahead, across the ends of the layers.  A wavefront takes 32 columns of all 64 rows (of 32 where the layer
// is so narrow that its columns would leave wavefronts idle), so that no two of a workgroup load the same weights.
// The weights are the matrix instruction's first operand and the rows its second: a lane has one row and, with the columns packed in a
// suitable order, twice eight neighbouring columns of it, which go to the planes 16 bytes at a time.  The activations that the
// way back needs go to memory in the order in which the lanes hold them, a kilobyte at a time, and come back the same way.
// Widths are padded to multiples of 64 with weights and biases of zero.
// Measured, inference with gradients against layer by layer: deep networks (seven layers of 256, 128, 64 and 8 on 384) and a charge network
// on 4,001 organic molecules (47,000 atoms) 1,701 -> 1,493 us, the networks alone 100 molecules 224 -> 181; default networks
// (128 128 64) with charges on 16,384 molecules 1,376 -> 1,227, on 256 204 -> 162.  Relative errors against float64 of energies and gradients of the
// deep networks with charges on 1,000 6.2e-7 -> 3.6e-7 and 1.28e-6 -> 8.1e-7.
// Two half-precision values for an operand, scaled by rows and columns, need three products and 1,180 us, but hold 23 bits of it, and
// nothing of what is 2^-50 of its row's largest value or less.  Full rounds of 64-row tiles and the rest of 32 rows in two launches
// measured as one form (1,490; 1,500 molecules 440 for 427), 64 columns of 32 rows to each of four wavefronts 1,614.
// 340-347 us each way for those 47,000 rows (741 tiles of 64, three rounds of 256, at 2 GHz): matrix pipe busy 43 % forward and 42 % back, other vector
// instructions 21 and 15 %, wavefronts waiting half of their time (profiles/networks_chain_deep4001_counters.md).
#include <algorithm>

#include "khan_internal.h"
#include "net_chain.h"
#include "net_celu.h"
#include "split_bf16.h"

namespace khan {

namespace {

typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f4v __attribute__((ext_vector_type(4)));

constexpr int kChunkBytes = 3 * 1024;        // packed weights of 16 k x 32 columns: [part][lane][8 k]
constexpr int kRing = 4;                     // chunks of weights on their way
constexpr int kWaitLoads = 0x0f70;           // s_waitcnt vmcnt(0)

struct ChainProduct {
    int64_t at;                  // packed weights of type 0: [type][32 columns][16 k]
    int blocks, chunks;          // 32 columns, 16 k; multiples of 2 and 4
};
struct ChainArgs {
    const float* x[4];
    int n[4], tile_end[4];
    const char* packed;
    const float* fixed;          // per type: the hidden layers' biases one after the other, the output layer's weights, its bias
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

template <int kWaves, int kRB>
struct ChainLds {
    static constexpr int kRows = 32 * kRB;
    u4v planes[3][4 * kWaves][kRows + 1];        // [part][8 columns][row]
    float sums[kWaves][kRows];
    float fixed[kNetMaxLayers * 32 * kWaves + 4];        // the type's biases and output layer
};

struct Lane {
    int lane, wave, l32, half;
};
struct Ring {
    u4v part[kRing][3];
    __device__ __forceinline__ void load(int u, const char* chunk, unsigned lane16)
    {
#pragma unroll
        for (int m = 0; m < 3; ++m) part[u][m] = *reinterpret_cast<const u4v*>(chunk + m * 1024 + lane16);
    }
    __device__ __forceinline__ void start(const char* weights, unsigned lane16)
    {
#pragma unroll
        for (int u = 0; u < kRing; ++u) load(u, weights + u * kChunkBytes, lane16);
    }
};

// Which part of a product a wavefront forms: 32 columns (from column block `cb`) of RB blocks of 32 rows (from block rb0).
struct Share {
    int cb, rb0;
    bool active;
};
// half: the layer's columns are so few that two wavefronts share them, a block of rows each
template <int kWaves, int kRB>
__device__ __forceinline__ bool by_rows(int blocks) { return kRB == 2 && 2 * blocks <= kWaves; }
template <int kWaves, int kRB>
__device__ __forceinline__ Share share_of(int wave, int blocks)
{
    if (by_rows<kWaves, kRB>(blocks)) {
        const int rb0 = wave / blocks;
        return {wave - rb0 * blocks, min(rb0, kRB - 1), rb0 < kRB};
    }
    return {min(wave, blocks - 1), 0, wave < blocks};
}

// acc, small += the planes' columns from 8 first8 on (16 `chunks` of them) times the weights from `weights` on, whose first kRing chunks
// are in the ring; `next`: the weights that come after these
template <int kWaves, int kRB, int RB>
__device__ __forceinline__ void multiply(const ChainLds<kWaves, kRB>& S, const Lane& P, int first8, int rb0, int chunks, const char* weights, const char* next,
                                         Ring& ring, f32x16 (&acc)[RB], f32x16 (&small)[RB])
{
    const unsigned lane16 = P.lane * 16;
    const auto group = [&](int c) {
        const char* const ahead = c + kRing < chunks ? weights + (c + kRing) * kChunkBytes : next;
#pragma unroll
        for (int u = 0; u < kRing; ++u) {
            bf16x8 x[RB][3], w[3];
#pragma unroll
            for (int j = 0; j < RB; ++j)
#pragma unroll
                for (int m = 0; m < 3; ++m) x[j][m] = __builtin_bit_cast(bf16x8, S.planes[m][first8 + 2 * (c + u) + P.half][32 * (rb0 + j) + P.l32]);
#pragma unroll
            for (int m = 0; m < 3; ++m) w[m] = __builtin_bit_cast(bf16x8, ring.part[u][m]);
            const auto mul = [&](f32x16 (&to)[RB], int xi, int wi) {
#pragma unroll
                for (int j = 0; j < RB; ++j) to[j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(w[wi], x[j][xi], to[j], 0, 0, 0);
            };
            mul(small, 0, 2);
            mul(acc, 0, 0);
            mul(small, 1, 1);
            mul(small, 2, 0);
            mul(small, 0, 1);
            mul(small, 1, 0);
            ring.load(u, ahead + u * kChunkBytes, lane16);
            // the loads stay behind the chunk's products (vector, scalar and LDS instructions may pass): the compiler would gather
            // them behind the last one
            __builtin_amdgcn_sched_barrier(0x386);
        }
    };
    // (the first chunks apart: they have come, and wait for nothing that was asked for or stored after them)
    group(0);
#pragma unroll 1
    for (int c = kRing; c < chunks; c += kRing) group(c);
}

// a lane's values of a layer -> the planes, split
template <int kWaves, int kRB, int RB>
__device__ __forceinline__ void to_planes(ChainLds<kWaves, kRB>& S, const Lane& P, int cb, int rb0, const f32x16 (&y)[RB])
{
#pragma unroll
    for (int j = 0; j < RB; ++j)
#pragma unroll
        for (int g = 0; g < 2; ++g) {
            u4v p[3];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                unsigned q[3];
                split_pair(y[j][8 * g + 2 * e], y[j][8 * g + 2 * e + 1], q[0], q[1], q[2]);
                p[0][e] = q[0], p[1][e] = q[1], p[2][e] = q[2];
            }
#pragma unroll
            for (int m = 0; m < 3; ++m) S.planes[m][4 * cb + 2 * g + P.half][32 * (rb0 + j) + P.l32] = p[m];
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
// a lane's sixteen columns of a vector over the layer's columns (LDS)
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
__device__ __forceinline__ float slope_of(float a, float inv_alpha) { return a >= 0.f ? 1.f : fmaf(a, inv_alpha, 1.f); }

// wavefronts per SIMD: one workgroup of eight wavefronts with 64 rows of 256 (114 KB) on a compute unit or two of four with 64 of 128
// (57 KB; three would have 168 registers, 100 too few), and with 32 rows two and four
constexpr int chain_waves(int, int rb) { return rb == 2 ? 2 : 4; }

template <int kWaves, int kRB, bool kBack>
__global__ __launch_bounds__(64 * kWaves) __attribute__((amdgpu_waves_per_eu(chain_waves(kWaves, kRB), chain_waves(kWaves, kRB))))
void chain_kernel(const ChainArgs a)
{
    typedef ChainLds<kWaves, kRB> Lds;
    constexpr int kRows = Lds::kRows, kThreads = 64 * kWaves;
    __shared__ Lds S;
    float* const fixed = S.fixed;
    const int tid = threadIdx.x;
    const Lane P = {tid & 63, __builtin_amdgcn_readfirstlane(tid >> 6), tid & 31, (tid >> 5) & 1};
    const unsigned lane16 = P.lane * 16;
    const int tile = static_cast<int>(blockIdx.x);
    const int t = (tile >= a.tile_end[0]) + (tile >= a.tile_end[1]) + (tile >= a.tile_end[2]);
    const int row0 = (tile - (t == 0 ? 0 : a.tile_end[t - 1])) * kRows, n = a.n[t], H = a.hidden;
    const auto weights_of = [&](const ChainProduct& p, int cb) {
        return a.packed + p.at + (static_cast<int64_t>(t) * p.blocks + cb) * p.chunks * kChunkBytes;
    };
    const auto act_at = [&](int h, int cb, int rb) -> float* {
        return a.act[h] + (static_cast<size_t>(tile) * a.act_blocks[h] + cb) * kRB * 1024 + rb * 1024;
    };
    Ring ring;
    ring.start(weights_of(a.p[0], share_of<kWaves, kRB>(P.wave, min(a.p[0].blocks, kWaves)).cb), lane16);
    for (int i = tid; i < a.fixed_size; i += kThreads) fixed[i] = a.fixed[static_cast<size_t>(t) * a.fixed_size + i];

    // product l, column blocks from `cb0` on, in one of the two shares; `before(multiply)` may call it more than once
    const auto run = [&](auto rb_count, int l, int cb0, auto&& before, auto&& operands, auto&& finish) {
        constexpr int RB = decltype(rb_count)::value;
        const ChainProduct& p = a.p[l];
        const int blocks = min(p.blocks - cb0, kWaves);
        const Share s = share_of<kWaves, kRB>(P.wave, blocks);
        const char* const weights = weights_of(p, cb0 + s.cb);
        const char* next = weights;
        if (cb0 + kWaves < p.blocks) next = weights_of(p, cb0 + kWaves + share_of<kWaves, kRB>(P.wave, min(p.blocks - cb0 - kWaves, kWaves)).cb);
        else if (l + 1 < H) next = weights_of(a.p[l + 1], share_of<kWaves, kRB>(P.wave, min(a.p[l + 1].blocks, kWaves)).cb);
        f32x16 acc[RB], small[RB];
#pragma unroll
        for (int j = 0; j < RB; ++j) acc[j] = small[j] = f32x16(0.f);
        auto met = before(rb_count, s);
        operands(p, s, [&](int first8, int first, int chunks) {
            if (s.active) {
                const char* const from = weights + first * kChunkBytes;
                multiply<kWaves, kRB, RB>(S, P, first8, s.rb0, chunks, from, first + chunks < p.chunks ? from + chunks * kChunkBytes : next, ring, acc, small);
            }
        });
        if (!s.active) ring.start(next, lane16);
#pragma unroll
        for (int j = 0; j < RB; ++j) acc[j] += small[j];
        finish(rb_count, s, cb0, acc, met);
    };
    const auto run_any = [&](int l, int cb0, auto&& before, auto&& operands, auto&& finish) {
        if constexpr (kRB == 2) {
            if (by_rows<kWaves, kRB>(min(a.p[l].blocks - cb0, kWaves))) return run(std::integral_constant<int, 1>(), l, cb0, before, operands, finish);
        }
        run(std::integral_constant<int, kRB>(), l, cb0, before, operands, finish);
    };
    const auto nothing = [](auto, const Share&) { return 0; };
    const auto from_planes = [&](const ChainProduct& p, const Share&, auto&& mul) { mul(0, 0, p.chunks); };

    if constexpr (!kBack) {
        // ---- layer 1: the feature rows through the planes piece by piece.  kHeld: half the planes at a time, the next piece's loads
        // in flight during the products (the one workgroup of the compute unit would wait for them); otherwise there are
        // other workgroups, and no registers for it.
        constexpr bool kHeld = kWaves == 8 && kRB == 2;
        constexpr int kPiece = (kHeld ? 16 : 32) * kWaves, kUnits = kRows * kPiece / 8 / kThreads;       // 8 columns of a row
        const auto place = [&](int i, int& row, int& k8) {
            const int unit = tid + i * kThreads, rest = unit >> 3;
            row = rest % kRows;
            k8 = (unit & 7) + 8 * (rest / kRows);
        };
        const auto fetch = [&](int i, int piece, f4v (&x)[2]) {
            int row, k8;
            place(i, row, k8);
            const int column = min(piece * kPiece + 8 * k8, a.k0 - 8);           // (past the end: others again, not read)
            const float* const from = a.x[t] + static_cast<size_t>(min(row0 + row, n - 1)) * a.k0 + column;
            x[0] = *reinterpret_cast<const f4v*>(from);
            x[1] = *reinterpret_cast<const f4v*>(from + 4);
        };
        const auto stage = [&](int i, int first8, const f4v (&x)[2]) {
            int row, k8;
            place(i, row, k8);
            u4v p[3];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                unsigned q[3];
                split_pair(x[e >> 1][2 * (e & 1)], x[e >> 1][2 * (e & 1) + 1], q[0], q[1], q[2]);
                p[0][e] = q[0], p[1][e] = q[1], p[2][e] = q[2];
            }
#pragma unroll
            for (int m = 0; m < 3; ++m) S.planes[m][first8 + k8][row] = p[m];
        };
        const auto through_pieces = [&](const ChainProduct&, const Share&, auto&& mul) {
            if constexpr (kHeld) {
                const int pieces = a.k0 / kPiece;
                f4v held[kUnits][2];
#pragma unroll
                for (int i = 0; i < kUnits; ++i) {
                    fetch(i, 0, held[i]);
                    stage(i, 0, held[i]);
                }
#pragma unroll 1
                for (int piece = 0; piece < pieces; ++piece) {
                    __syncthreads();       // the piece is staged, and the other half of the planes has been read
#pragma unroll
                    for (int i = 0; i < kUnits; ++i) fetch(i, min(piece + 1, pieces - 1), held[i]);
                    mul((piece & 1) * (kPiece / 8), piece * (kPiece / 16), kPiece / 16);
#pragma unroll
                    for (int i = 0; i < kUnits; ++i) stage(i, ((piece + 1) & 1) * (kPiece / 8), held[i]);      // (behind the last: not read)
                }
            } else {
#pragma unroll 1
                for (int piece = 0; piece * kPiece < a.k0; ++piece) {
                    if (piece > 0) __syncthreads();         // the planes have been read
#pragma unroll
                    for (int i = 0; i < kUnits; ++i) {
                        f4v x[2];
                        fetch(i, piece, x);
                        stage(i, 0, x);
                    }
                    __syncthreads();
                    mul(0, piece * (kPiece / 16), min(kPiece, a.k0 - piece * kPiece) / 16);
                }
            }
        };
        const auto layer = [&](int l, auto&& operands) {
            run_any(l, 0, nothing, operands, [&](auto rb_count, const Share& s, int, auto& y, int) {
                constexpr int RB = decltype(rb_count)::value;
                if (s.active) {
                    const f32x16 bias = of_columns(fixed + a.fixed_at[l], P, s.cb);
                    const bool absolute = (a.absolute >> l) & 1u;
#pragma unroll
                    for (int j = 0; j < RB; ++j) {
                        if (absolute) {
#pragma unroll
                            for (int v = 0; v < 16; ++v) y[j][v] = celu_absolute(y[j][v] + bias[v], a.alpha, a.inv_alpha);
                        } else {
#pragma unroll
                            for (int v = 0; v < 16; ++v) y[j][v] = celu_exact(y[j][v] + bias[v], a.alpha, a.inv_alpha);
                        }
                    }
                }
                __syncthreads();           // the planes have been read
                if (s.active) {
                    if (l + 1 < H) {
                        to_planes<kWaves, kRB, RB>(S, P, s.cb, s.rb0, y);
                    } else {
                        const f32x16 w = of_columns(fixed + a.fixed_at[H], P, s.cb);
#pragma unroll
                        for (int j = 0; j < RB; ++j) {
                            float part[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
                            for (int v = 0; v < 16; ++v) part[v & 3] = fmaf(y[j][v], w[v], part[v & 3]);
                            float sum = (part[0] + part[1]) + (part[2] + part[3]);
                            sum += __shfl_xor(sum, 32, 64);
                            if (P.half == 0) S.sums[s.cb][32 * (s.rb0 + j) + P.l32] = sum;
                        }
                    }
                    if (a.act[l]) {
                        // loads and stores are waited for in the order they were issued: the next layer's first weights have to be
                        // there before the stores go out, which then have those chunks' time
                        __builtin_amdgcn_s_waitcnt(kWaitLoads);
#pragma unroll
                        for (int j = 0; j < RB; ++j) store_block(act_at(l, s.cb, s.rb0 + j), P, y[j]);
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
        for (int u = P.wave; u < a.act_blocks[H - 1] * kRB; u += kWaves) {
            const int cb = u / kRB, rb = u - cb * kRB;
            f32x16 y[1];
            load_block(act_at(H - 1, cb, rb), P, y[0]);
            const f32x16 w = of_columns(fixed + a.fixed_at[H], P, cb);
#pragma unroll
            for (int v = 0; v < 16; ++v) y[0][v] = w[v] * slope_of(y[0][v], a.inv_alpha);
            to_planes<kWaves, kRB, 1>(S, P, cb, rb, y);
        }
        __syncthreads();
        // ---- d_{L-1} .. d_1
#pragma unroll 1
        for (int l = 0; l + 1 < H; ++l) {
            const int h = H - 2 - l;               // the hidden layer whose activations are met
            const auto activations = [&](auto rb_count, const Share& s) {
                constexpr int RB = decltype(rb_count)::value;
                Blocks<RB> act;
#pragma unroll
                for (int j = 0; j < RB; ++j) load_block(act_at(h, s.cb, s.rb0 + j), P, act.v[j]);
                return act;
            };
            run_any(l, 0, activations, from_planes, [&](auto rb_count, const Share& s, int, auto& y, auto& act) {
                constexpr int RB = decltype(rb_count)::value;
#pragma unroll
                for (int j = 0; j < RB; ++j)
#pragma unroll
                    for (int v = 0; v < 16; ++v) y[j][v] *= slope_of(act.v[j][v], a.inv_alpha);
                __syncthreads();           // the planes have been read
                if (s.active) to_planes<kWaves, kRB, RB>(S, P, s.cb, s.rb0, y);
                __syncthreads();
            });
        }
        // ---- the rows
#pragma unroll 1
        for (int cb0 = 0; cb0 < a.p[H - 1].blocks; cb0 += kWaves) {
            run_any(H - 1, cb0, nothing, from_planes, [&](auto rb_count, const Share& s, int cb0, auto& y, int) {
                constexpr int RB = decltype(rb_count)::value;
                if (!s.active) return;
#pragma unroll
                for (int j = 0; j < RB; ++j) {
                    const int r = row0 + 32 * (s.rb0 + j) + P.l32;
                    const float scale = a.scale[t] ? a.scale[t][min(r, n - 1)] : 1.f;
                    float* const out = a.grad[t] + static_cast<size_t>(min(r, n - 1)) * a.k0 + 32 * (cb0 + s.cb) + 8 * P.half;
                    f4v v[4];
#pragma unroll
                    for (int q = 0; q < 4; ++q)
#pragma unroll
                        for (int e = 0; e < 4; ++e) v[q][e] = y[j][4 * q + e] * scale;
                    if (a.accumulate) {
#pragma unroll
                        for (int q = 0; q < 4; ++q) v[q] += *reinterpret_cast<const f4v*>(out + 16 * (q >> 1) + 4 * (q & 1));
                    }
                    if (r < n) {
#pragma unroll
                        for (int q = 0; q < 4; ++q) *reinterpret_cast<f4v*>(out + 16 * (q >> 1) + 4 * (q & 1)) = v[q];
                    }
                }
            });
        }
    }
}

// The weights of all products, split and in the order in which the lanes take them, and the padded biases; a wavefront per chunk.
struct PackProduct {
    const float* w[4];           // [k, n_out] as stored, or [n_out, k] (back)
    int k, n_out, blocks, chunks, end;       // end: running number of chunks of all types
    bool back;
    int64_t at;
};
struct PackArgs {
    PackProduct p[2 * kNetMaxLayers];
    const float *bias[kNetMaxLayers][4];
    int products, layers, widths[kNetMaxLayers + 1], fixed_at[kNetMaxLayers + 2], fixed_size;
    char* packed;
    float* fixed;
    const float* top[4];
};
__global__ __launch_bounds__(256) void chain_pack_kernel(const PackArgs a)
{
    const int lane = threadIdx.x & 63, number = static_cast<int>(blockIdx.x) * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    if (number >= a.p[a.products - 1].end) {
        // behind the weights: the biases, 64 values to a wavefront
        const int i = (number - a.p[a.products - 1].end) * 64 + lane, t = i / a.fixed_size, at = i - t * a.fixed_size;
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
    int m = 0;
    while (number >= a.p[m].end) ++m;
    const PackProduct& p = a.p[m];
    const int rel = number - (m == 0 ? 0 : a.p[m - 1].end), t = rel / (p.blocks * p.chunks), block = rel - t * p.blocks * p.chunks;
    const int cb = block / p.chunks, chunk = block - cb * p.chunks;
    const int col = 32 * cb + column_of(lane & 31), k0 = 16 * chunk + 8 * (lane >> 5);
    const float* const w = p.w[t];
    float v[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        const bool inside = w && col < p.n_out && k0 + e < p.k;
        const size_t at = p.back ? static_cast<size_t>(col) * p.k + k0 + e : static_cast<size_t>(k0 + e) * p.n_out + col;
        v[e] = inside ? w[inside ? at : 0] : 0.f;
    }
    u4v part[3];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        unsigned q[3];
        split_pair(v[2 * e], v[2 * e + 1], q[0], q[1], q[2]);
        part[0][e] = q[0], part[1][e] = q[1], part[2][e] = q[2];
    }
    char* const to = a.packed + p.at + static_cast<int64_t>(rel) * kChunkBytes + lane * 16;
#pragma unroll
    for (int q = 0; q < 3; ++q) *reinterpret_cast<u4v*>(to + q * 1024) = part[q];
}

// ---- host
int padded(int width) { return (width + 63) / 64 * 64; }

struct Layout {
    int waves, rb, hidden, tiles;
    ChainProduct f[kNetMaxLayers], r[kNetMaxLayers];
    int64_t fixed_bytes_at, act_at[kNetMaxLayers], bytes;
    int fixed_at[kNetMaxLayers + 2], fixed_size, act_blocks[kNetMaxLayers], tile_end[4];

    explicit Layout(const NetChain& net) : hidden(net.hidden)
    {
        int widest = 0;
        for (int l = 1; l <= hidden; ++l) widest = std::max(widest, net.widths[l]);
        waves = widest <= 128 ? 4 : 8;
        // (the last chunks' places are loaded from ahead of need)
        int64_t at = 0;
        const auto product = [&](int k, int n_out) {
            const ChainProduct p = {at, padded(n_out) / 32, padded(k) / 16};
            at += 4ll * p.blocks * p.chunks * kChunkBytes;
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
        int64_t tiles64 = 0;
        for (int t = 0; t < 4; ++t) tiles64 += (net.n[t] + 63) / 64;
        // 32 or 64 rows to a workgroup.  64 halve the weights' way from the L2 and are the faster form of a full chip (organic molecules;
        // 4 wavefronts: 943 against 995 us for 141,000 rows and 271 against 286 for 29,000; 8: 2,124 against 2,191 for 141,000); but with
        // half as many workgroups, they leave more of the chip idle in the last round, and 32 win where that round is up to half full
        // (4 wavefronts: 322 against 342 for 35,000 rows, 109 against 132 for 12; 8: 392 against 485 for 17,600, 138 against 207 for 12),
        // unless there are so many rounds that half of one is less than the forms differ.
        const int64_t round = 256 * (chain_waves(waves, 2) * 4 / waves), last = tiles64 % round;
        rb = last == 0 || last > round / 2 || tiles64 >= 8 * round ? 2 : 1;
        tiles = 0;
        for (int t = 0; t < 4; ++t) tile_end[t] = tiles += (net.n[t] + 32 * rb - 1) / (32 * rb);
        for (int l = 0; l < hidden; ++l) {
            act_blocks[l] = padded(net.widths[l + 1]) / 32;
            act_at[l] = at;
            if (net.want_rows) at += static_cast<int64_t>(tiles) * act_blocks[l] * rb * 4096;
        }
        bytes = at + 16;
    }
};

template <int kWaves, int kRB, bool kBack>
hipError_t launch(const ChainArgs& a, int tiles, hipStream_t stream)
{
    chain_kernel<kWaves, kRB, kBack><<<dim3(static_cast<unsigned>(tiles)), dim3(64 * kWaves), 0, stream>>>(a);
    return hipGetLastError();
}
template <bool kBack>
hipError_t launch_any(const ChainArgs& a, const Layout& L, hipStream_t stream)
{
    if (L.waves == 4) return L.rb == 2 ? launch<4, 2, kBack>(a, L.tiles, stream) : launch<4, 1, kBack>(a, L.tiles, stream);
    return L.rb == 2 ? launch<8, 2, kBack>(a, L.tiles, stream) : launch<8, 1, kBack>(a, L.tiles, stream);
}

ChainArgs args_of(const NetChain& net, const Layout& L, const void* workspace)
{
    ChainArgs a = {};
    char* const ws = static_cast<char*>(const_cast<void*>(workspace));
    for (int t = 0; t < 4; ++t) {
        a.x[t] = net.x[t];
        a.n[t] = net.n[t];
        a.tile_end[t] = L.tile_end[t];
    }
    a.packed = ws;
    a.fixed = reinterpret_cast<const float*>(ws + L.fixed_bytes_at);
    for (int l = 0; l < L.hidden; ++l) {
        a.act[l] = net.want_rows ? reinterpret_cast<float*>(ws + L.act_at[l]) : nullptr;
        a.act_blocks[l] = L.act_blocks[l];
    }
    std::copy(L.fixed_at, L.fixed_at + kNetMaxLayers + 2, a.fixed_at);
    a.fixed_size = L.fixed_size;
    a.hidden = L.hidden;
    a.k0 = net.widths[0];
    a.absolute = net.absolute;
    a.alpha = net.alpha;
    a.inv_alpha = 1.0f / net.alpha;
    return a;
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
    if (L.tiles == 0) return hipSuccess;
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
            q.end = end += 4 * c.blocks * c.chunks;
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
    const int waves = end + (4 * L.fixed_size + 63) / 64;
    chain_pack_kernel<<<dim3(static_cast<unsigned>((waves + 3) / 4)), dim3(256), 0, stream>>>(p);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    ChainArgs a = args_of(net, L, workspace);
    std::copy(L.f, L.f + L.hidden, a.p);
    for (int t = 0; t < 4; ++t) a.value[t] = value[t];
    return launch_any<false>(a, L, stream);
}

hipError_t launch_net_chain_rows(const NetChain& net, const void* workspace, const float* const scale[4], float* const grad[4], bool accumulate,
                                 hipStream_t stream)
{
    const Layout L(net);
    if (L.tiles == 0) return hipSuccess;
    ChainArgs a = args_of(net, L, workspace);
    std::copy(L.r, L.r + L.hidden, a.p);
    for (int t = 0; t < 4; ++t) {
        a.scale[t] = scale[t];
        a.grad[t] = grad[t];
    }
    a.accumulate = accumulate;
    return launch_any<true>(a, L, stream);
}

}  // namespace khan
