// The whole atomic network of the reference's default size, 384-128-128-64-1 with CELU (khan/model/nn.py:38-68,
// khan/model/activations.py:63-65; sizes: khan/inference/energy_server.py:121), for the four atom types in ONE launch,
// forward and -- on request -- back to the feature rows:
//     a1 = celu(x W1 + b1), a2 = celu(a1 W2 + b2), a3 = celu(a2 W3 + b3), e = a3 w4 + b4          (per feature row x)
//     g3 = s w4^T .* celu'(a3), g2 = (g3 W3^T) .* celu'(a2), g1 = (g2 W2^T) .* celu'(a1), dx = g1 W1^T
// with s the gradient with respect to each row's value e (1 when none is given: the gradient of the sum of the values,
// which is what forces need).  A feature row is read once and its gradient written once: the activations of a tile of
// rows never leave the compute unit.  Layer by layer the same pass moves 2.9 GB forward and 3.7 GB back per 767,292
// rows (every activation written, read again by the next layer and once more on the way back); this one moves the rows
// and their gradients, 2.4 GB, and the values.
//
// One workgroup of four wavefronts owns 64 rows at a time; two workgroups share a compute unit and, having no barriers in
// common, fill each other's waits.  A workgroup goes on to another tile of rows when it is through with one, and has the next
// tile's first rows and weights on their way before it stores the gradients of the last.  The products run on the 16-bit matrix instructions
// (v_mfma_f32_32x32x16_f16, sixteen times the rate of the float32 ones) with every float32 operand split into two
// half-precision parts:
//     x = h + 2^-11 l,   h = half(x),   l = half(2^11 (x - h))
// h carries 11 significant bits, x - h is exact in float32 and at most 2^-11 |x|, and l carries its 11 leading bits:
// |x - h - 2^-11 l| <= 2^-23 |x|, and 0 for three values of four (where x - h needs a twelfth bit, the last one goes).  The residual is scaled by 2^11 so that it has
// x's exponent and not one twelve binary orders below it, where half precision would run out of exponent for every
// |x| < 0.25.  Of the four partial products of x w three are kept, each an exact 22-bit product accumulated in
// float32, in two accumulators:
//     hi += h_x h_w,   lo += h_x l_w + l_x h_w,   x w ~ hi + 2^-11 lo      (left out: l_x l_w 2^-22 <= 2^-22 |x w|)
// which is a float32 product to within 2^-21 |x w| (a term of 2^-22 and two of 2^-23) from three matrix instructions;
// the three-way bfloat16 split of dense_first.hip, which keeps every bit of the operands, needs six.  What it costs is range: half precision ends at 65,504,
// so an operand (feature, activation, weight) of that size or more gives NaN -- never a wrong finite number -- and an
// |x| below 6e-5 keeps an absolute accuracy of 2^-36 instead of a relative one.  On the way back the gradient is
// carried for a unit upstream factor and multiplied by the row's factor only when it is stored (the pass is linear
// in it), so that the gradients' size inside the kernel does not depend on the caller's loss scale.
// A wavefront holds all 64 rows of 32 columns of a layer's 64 x 128 output
// (32 x 32 of the 64 x 64 one) in accumulator registers, and keeps its part of a1, a2 and a3 in registers for the way
// back, where the gradients arrive in the same places.  Between layers the activations (gradients) go to LDS already
// split, as two planes [row][k] of half precision: the next product's row operand, read straight from there.  The weights
// do not pass through LDS: every wavefront loads its operands of a chunk of 16 k straight into registers (layer_product)
// -- from the chunks the caller has had split once beforehand (launch_networks_pack), or from the float32 weights, which
// a lane then splits itself.  Layer 1's feature rows, float32 in memory, go through a double-buffered LDS stage in the
// space the activation planes take later.  LDS: 41 KB per workgroup; 2 wavefronts per SIMD (the accumulators, the
// saved activations and the weights on their way take 240 registers).
//
// 767,292 rows with gradients, one after another: 970 us -> 830 us (one tile per workgroup, weights asked for one chunk ahead and
// anew at each product, biases from memory, two vector instructions of address per load -> all that is said here).  Bound by power
// as much as by anything: 640 us with neither rows nor gradients in memory, at a clock of 1.8 GHz with the matrix units 55 % busy; with
// them the matrix units are 39 % busy at 1.9 to 2.0 GHz; the rows and gradients alone are 440 us of memory traffic.
// Tried and slower: gradients stored one run per chunk of the product after (4 %), stores marked as written once (18 %).
#include "dense_fused_tiles.h"
#include "khan_internal.h"
#include "khan_params.h"

namespace khan {

namespace {

typedef float v4 __attribute__((ext_vector_type(4)));
typedef float v16 __attribute__((ext_vector_type(16)));
typedef unsigned u2v __attribute__((ext_vector_type(2)));
typedef unsigned u4v __attribute__((ext_vector_type(4)));
typedef _Float16 h2v __attribute__((ext_vector_type(2)));
typedef _Float16 h8v __attribute__((ext_vector_type(8)));
typedef float f2v __attribute__((ext_vector_type(2)));

constexpr int kRows = kFusedRows;   // rows per workgroup
constexpr int kResident = 2 * kCUs; // workgroups that the chip holds
constexpr int kThreads = 256;       // four wavefronts: 64 rows x 32 columns each of a 128-wide output
constexpr int kK1 = kFusedK1, kN1 = kFusedN1, kN2 = kFusedN2, kN3 = kFusedN3;
constexpr int kActStride = 136;     // 16-bit elements between rows of the activation planes: 128 + 8 (16-byte reads without bank conflicts)
constexpr int kKC = kFusedKC;       // k per staged chunk
constexpr int kStStride = 40;       // 16-bit elements between staged rows: a pair of chunks (32 k) + 8
constexpr int kParts = kFusedParts;
constexpr float kResidualScale = 2048.0f, kResidualBack = 1.0f / 2048.0f;      // 2^11

struct FusedArgs {
    const float* rows[4];           // [n_t, 384] feature rows per type
    int n[4];
    int tile_end[4];                // running sum of the per-type row tiles
    const float* w1t[4];            // [128, 384]: layer 1's weights, the summed index contiguous (transposed)
    const float* w2t[4];            // [128, 128]
    const float* w3t[4];            // [64, 128]
    const float* w1[4];             // [384, 128]: as stored -- the transposed operand of the way back
    const float* w2[4];             // [128, 128]
    const float* w3[4];             // [128, 64]
    const float* b1[4];
    const float* b2[4];
    const float* b3[4];
    const float* w4[4];             // [64]
    const float* b4[4];             // one float
    const float* scale[4];          // [n_t] gradient with respect to each row's value, or null (ones)
    float* value[4];                // [n_t]
    float* grad[4];                 // [n_t, 384], or null
    const unsigned short* packed;   // the six weight matrices of every type already split (pack_weights_kernel), or null
};

// a type's biases and output layer, one after the other
constexpr int kAtB1 = 0, kAtB2 = kAtB1 + kN1, kAtB3 = kAtB2 + kN2, kAtW4 = kAtB3 + kN3, kAtB4 = kAtW4 + kN3, kFixed = kAtB4 + 4;

struct __align__(16) FusedLds {
    union {
        unsigned short act[kParts][kRows][kActStride];        // a layer's activations or gradients, split: [part][row][k]
        unsigned short astage[2][kParts][kRows][kStStride];   // layer 1: pairs of chunks of the feature rows
    };
    float rowval[2][kRows];                              // the output layer's partial sums
    // every type's biases and output layer: read from memory between two products they would be waited for behind the weights
    // already asked for (loads come back in order)
    float fixed[4][kFixed];
};

// two floats -> their two half-precision parts (the value rounded, and 2^11 times what the rounding left), each pair
// packed into one register (first value in the low half).  Both differences are exact in float32.
__device__ __forceinline__ void split_pair(float x0, float x1, unsigned& p1, unsigned& p2)
{
    const h2v h = __builtin_convertvector(f2v{x0, x1}, h2v);
    p1 = __builtin_bit_cast(unsigned, h);
    // 2^11 x - 2^11 h in one fused multiply-add that reads h and writes half precision as they are (both products are exact,
    // and so is the difference)
    h2v l;
    l[0] = static_cast<_Float16>(fmaf(static_cast<float>(h[0]), -kResidualScale, x0 * kResidualScale));
    l[1] = static_cast<_Float16>(fmaf(static_cast<float>(h[1]), -kResidualScale, x1 * kResidualScale));
    p2 = __builtin_bit_cast(unsigned, l);
}

// a chunk piece (four consecutive k of one row or column) split into the planes of a stage buffer
template <int kR>
__device__ __forceinline__ void stage_piece(unsigned short (&dst)[kParts][kR][kStStride], int r, int k4, const v4 x)
{
    unsigned lo[kParts], hi[kParts];
    split_pair(x[0], x[1], lo[0], lo[1]);
    split_pair(x[2], x[3], hi[0], hi[1]);
#pragma unroll
    for (int q = 0; q < kParts; ++q) *reinterpret_cast<u2v*>(&dst[q][r][k4]) = u2v{lo[q], hi[q]};
}

__device__ __forceinline__ float celu_of(float v, float alpha, float to_exp2)
{
    const float below = fmaf(alpha, __builtin_amdgcn_exp2f(v * to_exp2), -alpha);
    return v >= 0.f ? v : below;
}
// CELU' from CELU's own value: 1 for h >= 0, exp(z / alpha) = h / alpha + 1 below
__device__ __forceinline__ float celu_slope(float h, float inv_alpha) { return __builtin_elementwise_minimum(1.0f, fmaf(h, inv_alpha, 1.0f)); }

// Positions.  The weights are the matrix instruction's first operand and the rows its second, so that a lane has one row of
// a block and four times four neighbouring columns of it, and what follows a product works on runs of four: the activations go to
// LDS eight bytes at a time (with a row's columns spread over the lanes it was two bytes at a time, 64 writes a layer, and
// the output layer's sums sixteen reductions over 32 lanes), the gradients to memory sixteen.  A 128-wide output (kWide): the
// wavefront owns the tile's 64 rows x 32 columns as two 32 x 32 blocks, block j with row j*32 + l32, accumulator e with column
// wave*32 + 8 (e / 4) + 4 half + e % 4.  The 64-wide output of layer 3: one block per wavefront, rows wr*32 + l32, columns
// wc*32 + ...
struct Place {
    int tid, lane, wave, wr, wc, l32, half;
    template <bool kWide> __device__ __forceinline__ int row(int j) const { return (kWide ? j * 32 : wr * 32) + l32; }
    template <bool kWide> __device__ __forceinline__ int col(int q) const { return (kWide ? wave * 32 : wc * 32) + 8 * q + 4 * half; }      // of accumulators 4 q .. 4 q + 3
    template <bool kWide> __device__ __forceinline__ int operand_col() const { return (kWide ? wave * 32 : wc * 32) + l32; }               // of the weights this lane loads
};

// The products of the pass in their order; each is acc = A . B^T for this workgroup's 64 rows, A = 64 x K (rows), B = columns x K
// (one row per output column), chunk by chunk of 16 k.
enum Pass { kF1, kF2, kF3, kG3, kG2, kGx };          // layers 1 to 3, their data gradients back to a2, a1, and (128 columns at a time) the rows
template <int kP> struct ProductOf {
    static constexpr int kK = kP == kF1 ? kK1 : kP == kF2 ? kN1 : kP == kF3 ? kN2 : kP == kG3 ? kN3 : kP == kG2 ? kN2 : kN1;
    static constexpr bool kWide = kP != kF3;
    static constexpr int kCols = kWide ? 128 : 64;
    static constexpr int kChunks = kK / kKC;
    // the chunks of all products end to end, one after the other through the ring of register sets
    static constexpr int kRing0 = kP <= kG3 ? 0 : kN3 / kKC;
    static_assert(kN3 / kKC == 4 && kK1 / kKC % 8 == 0 && kN1 / kKC % 8 == 0 && kN2 / kKC % 8 == 0, "where each product's chunks begin in the ring");
};

// B never passes through LDS: a matrix instruction's operand is, per lane, eight consecutive k of one column -- 16
// bytes of a packed chunk, and the 64 lanes' pieces are one contiguous kilobyte -- so every wavefront loads its own
// operands straight into registers, kAhead chunks ahead, across the ends of the products: the wait for a product's first
// weights (2 us from L2 under this load, before every one of nine products) had been a third of the kernel, and the next product's
// weights are asked for before the gradients' stores, which a load behind them would wait for (loads and stores share one
// counter, in order).  In a 128-wide product a wavefront takes ALL 64 rows of 32
// columns: its weight operand serves two matrix instructions' worth of rows, no other wavefront loads the same
// columns, and the row operand -- from LDS, which has the bandwidth to spare -- is read twice as often instead.  (With
// 32 rows x 64 columns per wavefront the two wavefronts of a column half loaded the same weights: the weights' loads,
// 1.2 MB per tile through the compute unit's 64-byte-per-cycle load path, were the largest single part of the kernel.)
// With the weights staged in LDS (the first version) the kernel was bound by LDS traffic: nine kilobytes read and
// written per wavefront and chunk for six matrix instructions, and a barrier per chunk.
// kPacked: the matrices' packed chunks (half precision); otherwise float32 weights, of which a lane loads its eight values and
// splits them itself.
// A stretch of memory by descriptor: a load takes the lane's offset from one 32-bit register and the wavefront's from a
// scalar one, with no vector arithmetic (by address the compiler spends two vector instructions and two registers on each), and
// one whose lane's offset lies past the end gives zeros, a store there is dropped.  (Whether the scalar offset counts in that is not
// relied on: it always lies inside.)
struct Stretch {
    __amdgpu_buffer_rsrc_t r;
    __device__ __forceinline__ void set(const void* p, unsigned bytes) { r = __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, bytes, 0x00020000); }
    __device__ __forceinline__ u4v get(unsigned lane, unsigned uniform) const { return __builtin_amdgcn_raw_buffer_load_b128(r, lane, uniform, 0); }
    // of data read once: it does not take the place of the weights in L2 (767k rows: 866 -> 830 us)
    __device__ __forceinline__ u4v get_once(unsigned lane, unsigned uniform) const { return __builtin_amdgcn_raw_buffer_load_b128(r, lane, uniform, 2); }
    // The whole offset is in the lane's register: behind a 16-byte store with a scalar offset the compiler sees no need to wait before
    // it writes the data registers anew, and such stores were seen to take the new value (lanes 12 to 15 of each sixteen, the first
    // of the four floats).  Not marked as written once: the stores take 160 us longer so.
    __device__ __forceinline__ void put(const v4 x, unsigned lane) const
    {
        __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u4v, x), r, lane, 0, 0);
    }
};

struct BSet {
    u4v raw[2];      // a chunk's operand for this wavefront's columns, as loaded: the two parts (packed), or eight float32 weights
};
constexpr int kAhead = 8;
template <bool kPacked>
struct Weights {
    Stretch packed;                                      // every type's packed matrices
    const void* w[6];                                    // float32: of F1, F2, F3, G3, G2, Gx
    const void* w_next;                                  // of F1 for the workgroup's next tile
    int t, t_next;                                       // the types of this tile and of the workgroup's next one (without one: of this,
    unsigned skip_next;                                  // and what is asked for ahead for it lies this far past the end, where a load gives zeros)
    BSet set[kAhead];

    template <int kP>
    __device__ __forceinline__ void fetch(const Place& P, int c, BSet& x, int column_tile = 0) const
    {
        fetch_of<kP>(t, w[kP], 0, P, c, x, column_tile);
    }
    template <int kP>
    __device__ __forceinline__ void fetch_of(int type, const void* w, unsigned skip, const Place& P, int c, BSet& x, int column_tile) const
    {
        typedef ProductOf<kP> Q;
        const unsigned col = P.operand_col<Q::kWide>();
        if constexpr (kPacked) {
            constexpr int kAt[6] = {kPackF1, kPackF2, kPackF3, kPackB3, kPackB2, kPackB1};
            const unsigned at = packed_chunk_at(type, kAt[kP], Q::kCols, Q::kK, column_tile, c);
            const unsigned lane = (col * kKC + P.half * 8) * 2 + skip;
#pragma unroll
            for (int m = 0; m < kParts; ++m) x.raw[m] = packed.get(lane, at + m * Q::kCols * kKC * 2);
        } else {
            Stretch matrix;
            matrix.set(w, (kP == kGx ? kK1 : Q::kCols) * Q::kK * 4);
            const unsigned at = (column_tile * 128 * Q::kK + c * kKC) * 4, lane = (col * Q::kK + P.half * 8) * 4 + skip;
            x.raw[0] = matrix.get(lane, at);
            x.raw[1] = matrix.get(lane, at + 16);
        }
    }
    // the chunk kAhead behind chunk c of product kP (compile-time c apart from layer 1's and the last product's repetitions)
    template <int kP, bool kGrad>
    __device__ __forceinline__ void fetch_behind(const Place& P, int c, BSet& x, int column_tile)
    {
        typedef ProductOf<kP> Q;
        const int d = c + kAhead - Q::kChunks;           // in the product after this one
        if (d < 0) {
            fetch<kP>(P, c + kAhead, x, column_tile);
        } else if constexpr (kP == kF1) {
            fetch<kF2>(P, d, x);
        } else if constexpr (kP == kF2) {
            fetch<kF3>(P, d, x);
        } else if constexpr (!kGrad) {
            return;
        } else if constexpr (kP == kF3) {
            if (d < ProductOf<kG3>::kChunks) fetch<kG3>(P, d, x);
            else fetch<kG2>(P, d - ProductOf<kG3>::kChunks, x);
        } else if constexpr (kP == kG3) {
            fetch<kG2>(P, d, x);
        } else if constexpr (kP == kG2) {
            fetch<kGx>(P, d, x);
        } else {
            // (a tile's chunks are four more than a multiple of the sets: chunk d + 4 of the next tile's layer 1 belongs here)
            if (column_tile + 1 < kK1 / 128) fetch<kGx>(P, d, x, column_tile + 1);
            else fetch_of<kF1>(t_next, w_next, skip_next, P, (d + ProductOf<kGx>::kRing0) % kAhead, x, 0);
        }
    }
    static __device__ __forceinline__ void operand(const BSet& x, h8v (&bv)[kParts])
    {
        if constexpr (kPacked) {
#pragma unroll
            for (int m = 0; m < kParts; ++m) bv[m] = __builtin_bit_cast(h8v, x.raw[m]);
        } else {
            u4v part[kParts];
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const v4 f = __builtin_bit_cast(v4, x.raw[h]);
                unsigned a[kParts], b[kParts];
                split_pair(f[0], f[1], a[0], a[1]);
                split_pair(f[2], f[3], b[0], b[1]);
#pragma unroll
                for (int m = 0; m < kParts; ++m) {
                    part[m][2 * h] = a[m];
                    part[m][2 * h + 1] = b[m];
                }
            }
#pragma unroll
            for (int m = 0; m < kParts; ++m) bv[m] = __builtin_bit_cast(h8v, part[m]);
        }
    }
};

// Layer 1: the feature rows go through LDS a PAIR of chunks (32 k = one 128-byte line per row) at a time: eight lanes
// fetch a row's line together, a thread two rows' pieces (rows r8 and r8 + 32, k8..k8+3 of the pair), and a barrier
// closes a pair, not a chunk.  kPairsAhead pairs are in flight in registers (as many as chunks of weights: a weight's wait is
// one for the rows asked for before it).
constexpr int kPairsAhead = kAhead / 2;
static_assert(kRows == 64 && kThreads == 256, "a thread two rows' pieces");
struct Rows {
    struct Pair {
        v4 x[2];
    };
    Stretch tile;
    Pair pair[kPairsAhead];

    __device__ __forceinline__ void fetch(const Place& P, int q, Pair& a, unsigned skip = 0) const
    {
        // (rows past the end come back as zeros, and nothing of theirs is stored)
#pragma unroll
        for (int u = 0; u < 2; ++u) a.x[u] = __builtin_bit_cast(v4, tile.get_once(lane(P) + u * 32 * kK1 * 4 + skip, q * 2 * kKC * 4));
    }
    static __device__ __forceinline__ unsigned lane(const Place& P) { return ((P.tid >> 3) * kK1 + ((P.tid & 7) << 2)) * 4; }
    // the first pairs of a tile's rows (skip: kFusedSkip where there is no tile, and zeros come back)
    __device__ __forceinline__ void start(const Place& P, const float* rows, int row0, int n, unsigned skip = 0)
    {
        tile.set(rows + static_cast<size_t>(row0) * kK1, min(n - row0, kRows) * kK1 * 4);
#pragma unroll
        for (int q = 0; q < kPairsAhead; ++q) fetch(P, q, pair[q], skip);
    }
};

// A comes from the activation planes, with no barrier inside the product; or (layer 1) from `rows` in memory, started by the
// caller, through a double-buffered LDS stage (the rows are float32 and have to be split and regrouped), one barrier per pair of chunks.  Begins
// and ends with a barrier: the planes written before the call are complete, and afterwards nobody reads the planes or the stage
// any more.  The product's first kAhead chunks of weights have been asked for before.
template <int kP, bool kGrad, bool kPacked>
__device__ __forceinline__ void layer_product(FusedLds& S, const Place& P, v16 (&acc)[2], Weights<kPacked>& W, Rows& R, int column_tile = 0)
{
    typedef ProductOf<kP> Q;
    constexpr bool kAGlobal = kP == kF1, kWide = Q::kWide;
    constexpr int chunks = Q::kChunks;
    constexpr int kNB = kWide ? 2 : 1;                   // blocks (accumulators) of this wavefront
    auto astage_pair = [&](int q, const Rows::Pair& a) {
        const int r8 = P.tid >> 3, k8 = (P.tid & 7) << 2;
        stage_piece(S.astage[q & 1], r8, k8, a.x[0]);
        stage_piece(S.astage[q & 1], r8 + 32, k8, a.x[1]);
    };

    v16 lo[2];                   // the mixed partial products, 2^11 times their size
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int e = 0; e < 16; ++e) {
            acc[j][e] = 0.f;
            lo[j][e] = 0.f;
        }
    if constexpr (kAGlobal) {
        astage_pair(0, R.pair[0]);
        R.fetch(P, kPairsAhead, R.pair[0]);
    }
    __syncthreads();             // pair 0 of the rows is staged; the activation planes written before this call are complete
    // chunk c: (layer 1, first chunk of a pair: stage the rows' next pair into the other buffer, ask for the pair
    // kPairsAhead further on,) multiply chunk c, ask for the weights kAhead chunks behind it
    auto step = [&](int c, BSet& b, Rows::Pair& a_next) {
        h8v av[2][kParts];
#pragma unroll
        for (int j = 0; j < kNB; ++j) {
            const int arow_l = (kWide ? j * 32 : P.wr * 32) + P.l32;
#pragma unroll
            for (int m = 0; m < kParts; ++m) {
                if constexpr (kAGlobal)
                    av[j][m] = __builtin_bit_cast(h8v, *reinterpret_cast<const u4v*>(&S.astage[(c >> 1) & 1][m][arow_l][(c & 1) * kKC + P.half * 8]));
                else
                    av[j][m] = __builtin_bit_cast(h8v, *reinterpret_cast<const u4v*>(&S.act[m][arow_l][c * kKC + P.half * 8]));
            }
        }
        if constexpr (kAGlobal) {
            asm volatile("" ::: "memory");               // the reads above stay ahead of the stage's writes
            const int q = c >> 1;
            if ((c & 1) == 0 && 2 * (q + 1) < chunks) {
                astage_pair(q + 1, a_next);              // the other buffer: last read before the previous barrier
                if (2 * (q + 1 + kPairsAhead) < chunks) R.fetch(P, q + 1 + kPairsAhead, a_next);
            }
        }
        h8v bv[kParts];
        Weights<kPacked>::operand(b, bv);
        // independent accumulators alternate, so that no matrix instruction waits for the one before it
#pragma unroll
        for (int j = 0; j < kNB; ++j) lo[j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(bv[0], av[j][1], lo[j], 0, 0, 0);
#pragma unroll
        for (int j = 0; j < kNB; ++j) acc[j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(bv[0], av[j][0], acc[j], 0, 0, 0);
#pragma unroll
        for (int j = 0; j < kNB; ++j) lo[j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(bv[1], av[j][0], lo[j], 0, 0, 0);
        W.template fetch_behind<kP, kGrad>(P, c, b, column_tile);
        // the loads stay here, behind the chunk's products (0x386: vector, scalar and LDS instructions may pass): the compiler would
        // gather them all behind the last product, where the next one waits for them
        __builtin_amdgcn_sched_barrier(0x386);
        if constexpr (kAGlobal) {
            if (c & 1) __syncthreads();                  // the pair has been read, the next one is staged
        }
    };
    // (layer 1: chunk c + u belongs to pair c / 2 + u / 2, and the pair staged during it, one further on, sits in register
    // set (u / 2 + 1) % kPairsAhead)
    constexpr int kBody = chunks < kAhead ? chunks : kAhead;
#pragma unroll 1
    for (int c = 0; c < chunks; c += kBody) {
#pragma unroll
        for (int u = 0; u < kBody; ++u) step(c + u, W.set[(Q::kRing0 + u) % kAhead], R.pair[kAGlobal ? ((u >> 1) + 1) % kPairsAhead : 0]);
    }
    if constexpr (!kAGlobal) __syncthreads();
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int e = 0; e < 16; ++e) acc[j][e] = fmaf(lo[j][e], kResidualBack, acc[j][e]);
}

// a wavefront's values of a layer -> the activation planes, split; column = k of the next product
template <bool kWide>
__device__ __forceinline__ void to_planes(FusedLds& S, const Place& P, const v16 (&v)[2])
{
#pragma unroll
    for (int j = 0; j < (kWide ? 2 : 1); ++j) {
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            unsigned lo[kParts], hi[kParts];
            split_pair(v[j][4 * q], v[j][4 * q + 1], lo[0], lo[1]);
            split_pair(v[j][4 * q + 2], v[j][4 * q + 3], hi[0], hi[1]);
#pragma unroll
            for (int m = 0; m < kParts; ++m) *reinterpret_cast<u2v*>(&S.act[m][P.row<kWide>(j)][P.col<kWide>(q)]) = u2v{lo[m], hi[m]};
        }
    }
}

// the four runs of four columns of this lane from a vector over the layer's columns
template <bool kWide>
__device__ __forceinline__ void of_columns(const Place& P, const float* __restrict__ from, float (&to)[16])
{
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const v4 f = *reinterpret_cast<const v4*>(from + P.col<kWide>(q));
#pragma unroll
        for (int e = 0; e < 4; ++e) to[4 * q + e] = f[e];
    }
}

template <bool kGrad, bool kPacked>
__global__ __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(2, 2)))
void networks_fused_kernel(FusedArgs args, float alpha, float inv_alpha, float to_exp2)
{
    static_assert(kRows == 64 && kThreads == 256, "four wavefronts: 64 rows x 32 columns each of a 128-wide output");
    __shared__ FusedLds S;
    Place P;
    P.tid = threadIdx.x;
    P.lane = P.tid & 63;
    P.wave = P.tid >> 6;
    P.wr = P.wave >> 1;
    P.wc = P.wave & 1;
    P.l32 = P.lane & 31;
    P.half = P.lane >> 5;
    Weights<kPacked> W;
    Rows R;
    W.packed.set(args.packed, kPackBytes);
    FusedTile at = fused_tile(args.tile_end, static_cast<int>(blockIdx.x));
    const auto start = [&](int t, int row0) {
        R.start(P, args.rows[t], row0, args.n[t]);
#pragma unroll
        for (int c = 0; c < kAhead; ++c) W.template fetch_of<kF1>(t, args.w1t[t], 0, P, c, W.set[c], 0);
    };
    {
        static_assert(kThreads == kN1 + kN2 && kAtB2 == kN1 && kAtW4 == kAtB3 + kN3, "two values per thread");
        float v[4][2], b4[4];
        const int i = P.tid;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            if (args.n[k] <= 0) continue;
            v[k][0] = i < kN1 ? args.b1[k][i] : args.b2[k][i - kN1];
            if (i < 2 * kN3) v[k][1] = i < kN3 ? args.b3[k][i] : args.w4[k][i - kN3];
            b4[k] = args.b4[k] ? args.b4[k][0] : 0.f;
        }
        start(at.type, at.row0);
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            if (args.n[k] <= 0) continue;
            S.fixed[k][kAtB1 + i] = v[k][0];
            if (i < 2 * kN3) S.fixed[k][kAtB3 + i] = v[k][1];
            if (i == 0) S.fixed[k][kAtB4] = b4[k];
        }
    }
    // Of two workgroups on a compute unit the older one's wavefronts are served first, and it would be through its tiles long
    // before the other (29 against 45 us a tile): every other tile the later workgroups have the precedence.
    bool high = blockIdx.x >= kCUs;
#pragma unroll 1
    for (;;) {
        if (high) __builtin_amdgcn_s_setprio(1); else __builtin_amdgcn_s_setprio(0);
        high = !high;
        const FusedTile next = fused_next(args.tile_end, at, static_cast<int>(gridDim.x));
        const bool more = next.tile != at.tile;
        const int t = at.type, row0 = at.row0, n = args.n[t];
        W.t = t;
        W.t_next = next.type;
        W.skip_next = more ? 0u : kFusedSkip;
        if constexpr (!kPacked) {
            W.w[kF1] = args.w1t[t];
            W.w[kF2] = args.w2t[t];
            W.w[kF3] = args.w3t[t];
            W.w[kG3] = args.w3[t];
            W.w[kG2] = args.w2[t];
            W.w[kGx] = args.w1[t];
            W.w_next = args.w1t[next.type];
        }

        v16 acc[2], a1[2], a2[2], a3[2];
        // ------------------------------------------------------------ layer 1: 384 -> 128
        layer_product<kF1, kGrad>(S, P, acc, W, R);
        {
            float b[16];
            of_columns<true>(P, S.fixed[t] + kAtB1, b);
#pragma unroll
            for (int j = 0; j < 2; ++j)
#pragma unroll
                for (int e = 0; e < 16; ++e) a1[j][e] = celu_of(acc[j][e] + b[e], alpha, to_exp2);
        }
        to_planes<true>(S, P, a1);
        // ------------------------------------------------------------ layer 2: 128 -> 128
        layer_product<kF2, kGrad>(S, P, acc, W, R);
        {
            float b[16];
            of_columns<true>(P, S.fixed[t] + kAtB2, b);
#pragma unroll
            for (int j = 0; j < 2; ++j)
#pragma unroll
                for (int e = 0; e < 16; ++e) a2[j][e] = celu_of(acc[j][e] + b[e], alpha, to_exp2);
        }
        to_planes<true>(S, P, a2);
        // ------------------------------------------------------------ layer 3: 128 -> 64, and the output layer 64 -> 1
        layer_product<kF3, kGrad>(S, P, acc, W, R);
        if constexpr (!kGrad) {
            if (more) start(next.type, next.row0);
        }
        float w4[16];
        of_columns<false>(P, S.fixed[t] + kAtW4, w4);
        {
            float b[16], part[4];
            of_columns<false>(P, S.fixed[t] + kAtB3, b);
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                part[q] = 0.f;
#pragma unroll
                for (int e = 4 * q; e < 4 * q + 4; ++e) {
                    a3[0][e] = celu_of(acc[0][e] + b[e], alpha, to_exp2);
                    part[q] = fmaf(a3[0][e], w4[e], part[q]);
                }
            }
            float sum = (part[0] + part[1]) + (part[2] + part[3]);
            sum += __shfl_xor(sum, 32, 64);                  // over this wavefront's 32 of the 64 columns
            if (P.half == 0) S.rowval[P.wc][P.row<false>(0)] = sum;
        }
        __syncthreads();
        if (P.tid < kRows) {
            const int gr = row0 + P.tid;
            const float value = S.rowval[0][P.tid] + S.rowval[1][P.tid] + S.fixed[t][kAtB4];
            if (gr < n) args.value[t][gr] = value;
        }
        if constexpr (!kGrad) {
            if (!more) return;
            at = next;
            continue;
        }
        // ------------------------------------------------------------ the way back
        const bool given = args.scale[t] != nullptr;
        float upstream[2];                                   // the upstream factors of this lane's rows, used after the products
        {
            Stretch scale;
            scale.set(args.scale[t] + (given ? row0 : 0), given ? min(n - row0, kRows) * 4 : 0);
#pragma unroll
            for (int j = 0; j < 2; ++j)
                upstream[j] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(scale.r, P.row<true>(j) * 4, 0, 0));
        }
        {
            v16 g3[2];
#pragma unroll
            for (int e = 0; e < 16; ++e) g3[0][e] = w4[e] * celu_slope(a3[0][e], inv_alpha);     // for a unit upstream factor
            to_planes<false>(S, P, g3);
        }
        // g2 = (g3 W3^T) .* celu'(a2): 64 -> 128
        layer_product<kG3, kGrad>(S, P, acc, W, R);
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int e = 0; e < 16; ++e) acc[j][e] *= celu_slope(a2[j][e], inv_alpha);
        to_planes<true>(S, P, acc);
        // g1 = (g2 W2^T) .* celu'(a1): 128 -> 128
        layer_product<kG2, kGrad>(S, P, acc, W, R);
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int e = 0; e < 16; ++e) acc[j][e] *= celu_slope(a1[j][e], inv_alpha);
        to_planes<true>(S, P, acc);
        // dx = g1 W1^T: 128 -> 384, three column tiles of 128
#pragma unroll
        for (int j = 0; j < 2; ++j) upstream[j] = given ? upstream[j] : 1.f;
        Stretch out;
        out.set(args.grad[t] + static_cast<size_t>(row0) * kK1, min(n - row0, kRows) * kK1 * 4);    // rows past the end are not stored
        const auto store = [&](int ct) {
            const unsigned lane = (P.row<true>(0) * kK1 + ct * 128 + P.col<true>(0)) * 4;
#pragma unroll
            for (int j = 0; j < 2; ++j)
#pragma unroll
                for (int q = 0; q < 4; ++q)
                    out.put(v4{acc[j][4 * q] * upstream[j], acc[j][4 * q + 1] * upstream[j], acc[j][4 * q + 2] * upstream[j], acc[j][4 * q + 3] * upstream[j]},
                            lane + j * 32 * kK1 * 4 + 32 * q);
        };
#pragma unroll 1
        for (int ct = 0; ct < kK1 / 128 - 1; ++ct) {
            layer_product<kGx, kGrad>(S, P, acc, W, R, ct);
            store(ct);
        }
        R.start(P, args.rows[next.type], next.row0, args.n[next.type], W.skip_next);
        layer_product<kGx, kGrad>(S, P, acc, W, R, kK1 / 128 - 1);
        store(kK1 / 128 - 1);
        if (!more) return;
        at = next;
    }
}

// one float32 weight -> its two half-precision parts in the packed buffer; a thread per weight of one type's six matrices.
// kStored: the transposed matrices are read from the stored ones, neighbouring threads along a stored row (a transposed copy
// of twelve matrices is twelve launches; the strided two-byte writes stay in L2).
template <bool kStored>
__global__ __launch_bounds__(256) void pack_weights_kernel(FusedArgs args, unsigned short* __restrict__ packed)
{
    const int t = blockIdx.y;
    const int i = blockIdx.x * 256 + threadIdx.x;           // index among the type's 147,456 weights
    constexpr int n1 = kN1 * kK1, n2 = kN2 * kN1, n3 = kN3 * kN2;
    if (i >= 2 * (n1 + n2 + n3)) return;
    const float* src;
    int at, cols, k_len, j = i;      // the matrix: where it starts in the packed buffer, its columns and its summed length
    bool across = kStored;           // src is [k][column]
    if (j < n1) { src = kStored ? args.w1[t] : args.w1t[t]; at = kPackF1; cols = kN1; k_len = kK1; }
    else if ((j -= n1) < n2) { src = kStored ? args.w2[t] : args.w2t[t]; at = kPackF2; cols = kN2; k_len = kN1; }
    else if ((j -= n2) < n3) { src = kStored ? args.w3[t] : args.w3t[t]; at = kPackF3; cols = kN3; k_len = kN2; }
    else if ((j -= n3) < n1) {       // layer 1 as stored, [384][128]: three matrices of 128 columns
        across = false;
        src = args.w1[t];
        const int ct = j / (128 * kN1);
        src += ct * 128 * kN1;
        j -= ct * 128 * kN1;
        at = kPackB1 + ct * kParts * 128 * kN1;
        cols = 128;
        k_len = kN1;
    }
    else if ((j -= n1) < n2) { across = false; src = args.w2[t]; at = kPackB2; cols = kN1; k_len = kN2; }
    else { j -= n2; across = false; src = args.w3[t]; at = kPackB3; cols = kN2; k_len = kN3; }
    unsigned p1, p2;
    split_pair(src[j], 0.f, p1, p2);
    const int line = across ? cols : k_len, major = j / line, minor = j - major * line;
    const int r = across ? minor : major, k = across ? major : minor;
    unsigned short* dst = packed + static_cast<size_t>(t) * kPackPerType + at + ((k / kKC) * kParts * cols + r) * kKC + (k % kKC);
    dst[0] = static_cast<unsigned short>(p1 & 0xffffu);
    dst[cols * kKC] = static_cast<unsigned short>(p2 & 0xffffu);
}

}  // namespace

size_t networks_packed_bytes() { return kPackBytes; }

// the six weight matrices of each type (three transposed, three as stored) split into `packed` (networks_packed_bytes());
// w*t null: the transposed ones from the stored ones
hipError_t launch_networks_pack(const float* const* w1t, const float* const* w2t, const float* const* w3t,
                                const float* const w1[4], const float* const w2[4], const float* const w3[4],
                                void* packed, hipStream_t stream)
{
    FusedArgs a = {};
    for (int t = 0; t < 4; ++t) {
        if (w1t) { a.w1t[t] = w1t[t]; a.w2t[t] = w2t[t]; a.w3t[t] = w3t[t]; }
        a.w1[t] = w1[t]; a.w2[t] = w2[t]; a.w3[t] = w3[t];
    }
    constexpr int per_type = 2 * (kN1 * kK1 + kN2 * kN1 + kN3 * kN2);
    const dim3 grid((per_type + 255) / 256, 4);
    if (w1t) pack_weights_kernel<false><<<grid, dim3(256), 0, stream>>>(a, static_cast<unsigned short*>(packed));
    else pack_weights_kernel<true><<<grid, dim3(256), 0, stream>>>(a, static_cast<unsigned short*>(packed));
    return hipGetLastError();
}

// rows[t]: [n[t], 384]; w*t: transposed weights ([out, in]); w*: as stored ([in, out]); value[t]: [n[t]];
// grad[t]: [n[t], 384] or null pointers (then only the values are formed; w1, w2, w3 and scale are not read).
// packed: the weights as launch_networks_pack left them (then w*t and w* are not read), or null.
hipError_t launch_networks_fused(const float* const rows[4], const int32_t n[4],
                                 const float* const w1t[4], const float* const w2t[4], const float* const w3t[4],
                                 const float* const w1[4], const float* const w2[4], const float* const w3[4],
                                 const float* const b1[4], const float* const b2[4], const float* const b3[4],
                                 const float* const w4[4], const float* const b4[4], const float* const scale[4],
                                 float alpha, float* const value[4], float* const grad[4], const void* packed,
                                 hipStream_t stream)
{
    FusedArgs a = {};
    a.packed = static_cast<const unsigned short*>(packed);
    int tiles = 0;
    bool want_grad = false;
    for (int t = 0; t < 4; ++t) {
        a.rows[t] = rows[t];
        a.n[t] = n[t];
        tiles += (n[t] + kRows - 1) / kRows;
        a.tile_end[t] = tiles;
        a.w1t[t] = w1t ? w1t[t] : nullptr; a.w2t[t] = w2t ? w2t[t] : nullptr; a.w3t[t] = w3t ? w3t[t] : nullptr;
        a.w1[t] = w1 ? w1[t] : nullptr; a.w2[t] = w2 ? w2[t] : nullptr; a.w3[t] = w3 ? w3[t] : nullptr;
        a.b1[t] = b1[t]; a.b2[t] = b2[t]; a.b3[t] = b3[t];
        a.w4[t] = w4[t];
        a.b4[t] = b4 ? b4[t] : nullptr;
        a.scale[t] = scale ? scale[t] : nullptr;
        a.value[t] = value[t];
        a.grad[t] = grad ? grad[t] : nullptr;
        want_grad = want_grad || (grad && grad[t]);
    }
    if (tiles == 0) return hipSuccess;
    const dim3 grid(static_cast<unsigned>(tiles < kResident ? tiles : kResident)), block(kThreads);
    const float to_exp2 = static_cast<float>(1.4426950408889634 / alpha);      // log2(e) / alpha
    if (want_grad) {
        if (packed) networks_fused_kernel<true, true><<<grid, block, 0, stream>>>(a, alpha, 1.0f / alpha, to_exp2);
        else networks_fused_kernel<true, false><<<grid, block, 0, stream>>>(a, alpha, 1.0f / alpha, to_exp2);
    } else {
        if (packed) networks_fused_kernel<false, true><<<grid, block, 0, stream>>>(a, alpha, 1.0f / alpha, to_exp2);
        else networks_fused_kernel<false, false><<<grid, block, 0, stream>>>(a, alpha, 1.0f / alpha, to_exp2);
    }
    return hipGetLastError();
}

}  // namespace khan
