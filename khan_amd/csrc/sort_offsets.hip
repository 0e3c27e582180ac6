// Integer part of the featurization path on gfx950: molecule offsets and the atom-type sort.
//
// ani_sort (reference: gpu_featurizer/ani_sort.cpp:71-115, a host std::stable_sort) is a stable
// 4-bin counting sort, i.e. four exclusive prefix sums over the atom array:
//     atom_counts[t]  = #{A == t}
//     scatter_idxs[g] = #{g' < g : A[g'] == A[g]}                       (rank inside its type)
//     gather_idxs[g]  = sum_{t < A[g]} atom_counts[t] + scatter_idxs[g]  (stable sort position)
// Two launches: per-tile histograms (wave ballot + popcount), and a rank pass that redoes the ballots and adds lane /
// wave / tile prefixes (above 4 million atoms a scan of the tile histograms in between).  Results are integers and
// identical to the host algorithm.
//
// mol_offsets (reference: tf.segment_sum(ones_like(m), m) and tf.cumsum(exclusive=True),
// khan/training/trainer_multi_tower.py:302-303) turns sorted per-atom molecule ids into per-molecule
// atom counts and exclusive offsets by locating the segment boundaries.
//
// A batch needs both and the size order at the bottom of this file before its first pass.  Each is a few microseconds of
// work and was two or three launches (nine in all, 62 us of GPU time for 65,536 organic molecules, 50 us for 1,024, and two
// copies to the host behind them); launch_prepare does the three together in three launches (24 us for 65,536), and in one for
// a batch of up to 16,384 atoms (9 us for 1,024 molecules, 5 us for a few hundred).
#include "khan_internal.h"
#include "khan_params.h"

namespace khan {

namespace {

constexpr int kSortThreads = 256;
constexpr int kSortSubTiles = 8;
constexpr int kSortTile = kSortThreads * kSortSubTiles;   // atoms per workgroup
// Up to this many tiles (4 million atoms) every workgroup of the rank pass adds up the tile histograms before its own by
// itself, at most eight 16-byte loads per thread; above it a scan of the histograms runs in between, because the sum of
// those loads grows with the square of the tiles.
constexpr int64_t kScanTiles = 2048;

// counts of each type among the 64 lanes, and this lane's rank among earlier lanes of its type
__device__ __forceinline__ void wave_type_masks(int type, bool valid, unsigned long long m[4])
{
#pragma unroll
    for (int t = 0; t < 4; ++t) m[t] = wave_ballot(valid && type == t);
}

// MOs[m] for the molecules that start at atom g (g = n: the ones behind the last atom): every molecule id in
// (id of atom g - 1, id of atom g]; ids skipped by the input are empty molecules
__device__ __forceinline__ void mol_starts(int64_t prev, int64_t cur, int64_t g, int32_t n_mols, int32_t* __restrict__ MOs)
{
    if (cur > n_mols - 1) cur = n_mols - 1;   // also keeps ids beyond n_mols from writing out of range
    if (prev < -1) prev = -1;
    for (int64_t m = prev + 1; m <= cur; ++m) MOs[m] = static_cast<int32_t>(g);
}
__device__ __forceinline__ void mol_bounds(const int32_t* __restrict__ mol_idxs, int64_t g, int64_t n, int32_t n_mols,
                                           int32_t* __restrict__ MOs)
{
    mol_starts(g > 0 ? mol_idxs[g - 1] : -1, g < n ? mol_idxs[g] : n_mols, g, n_mols, MOs);
}

// First pass over the atoms, a tile per workgroup: the tile's type histogram (A non-null), the molecules' first atoms
// (mol_idxs non-null), and zeros in the counters of the size order (size_scratch non-null).
__global__ __launch_bounds__(kSortThreads) void prep_count_kernel(const int32_t* __restrict__ A, const int32_t* __restrict__ mol_idxs,
                                                                  int64_t n, int32_t n_mols, int32_t* __restrict__ tile_counts,
                                                                  int32_t* __restrict__ MOs, int32_t* __restrict__ size_scratch)
{
    __shared__ int32_t wave_counts[4][4];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int64_t tile0 = static_cast<int64_t>(blockIdx.x) * kSortTile;
    if (size_scratch && blockIdx.x == 0)
        for (int k = threadIdx.x; k < kSizeOrderScratch; k += kSortThreads) size_scratch[k] = 0;
    int32_t cnt[4] = {0, 0, 0, 0};
    int32_t type[kSortSubTiles], id[kSortSubTiles], before[kSortSubTiles];
#pragma unroll
    for (int s = 0; s < kSortSubTiles; ++s) {        // every load in flight before the first is used
        const int64_t g = tile0 + s * kSortThreads + threadIdx.x;
        type[s] = A && g < n ? A[g] : -1;
        id[s] = mol_idxs && g < n ? mol_idxs[g] : -1;
        before[s] = mol_idxs && g < n && g > 0 ? mol_idxs[g - 1] : -1;
    }
#pragma unroll
    for (int s = 0; s < kSortSubTiles; ++s) {
        const int64_t g = tile0 + s * kSortThreads + threadIdx.x;
        if (A) {
            const bool valid = g < n;
            unsigned long long m[4];
            wave_type_masks(fold_type(type[s]), valid, m);
#pragma unroll
            for (int t = 0; t < 4; ++t) cnt[t] += __popcll(m[t]);
        }
        if (mol_idxs && g < n) mol_starts(before[s], id[s], g, n_mols, MOs);
    }
    // molecules behind the last atom (n = 0: all of them)
    if (MOs && blockIdx.x == 0 && threadIdx.x == 0) mol_bounds(mol_idxs, n, n, n_mols, MOs);
    if (!A) return;
    if (lane == 0) {
#pragma unroll
        for (int t = 0; t < 4; ++t) wave_counts[wave][t] = cnt[t];
    }
    __syncthreads();
    if (threadIdx.x < 4) {
        const int t = threadIdx.x;
        tile_counts[static_cast<int64_t>(blockIdx.x) * 4 + t] =
            wave_counts[0][t] + wave_counts[1][t] + wave_counts[2][t] + wave_counts[3][t];
    }
}

// Exclusive scan over tiles of the 4 per-tile counts, in place; totals[0..3] = atom_counts and
// totals[4..7] = exclusive type bases.  One workgroup; tiles are consumed 256 at a time.
__global__ __launch_bounds__(256) void sort_scan_kernel(int32_t* __restrict__ tile_counts,
                                                        int64_t n_tiles,
                                                        int32_t* __restrict__ totals,
                                                        int32_t* __restrict__ counts_out)
{
    __shared__ int32_t wave_tot[4][4];
    __shared__ int32_t carry[4];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    if (threadIdx.x < 4) carry[threadIdx.x] = 0;
    __syncthreads();
    for (int64_t base = 0; base < n_tiles; base += 256) {
        const int64_t b = base + threadIdx.x;
        int32_t v[4] = {0, 0, 0, 0};
        if (b < n_tiles) {
#pragma unroll
            for (int t = 0; t < 4; ++t) v[t] = tile_counts[b * 4 + t];
        }
        int32_t incl[4];
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            int32_t x = v[t];
#pragma unroll
            for (int d = 1; d < 64; d <<= 1) {
                const int32_t y = __shfl_up(x, d, 64);
                if (lane >= d) x += y;
            }
            incl[t] = x;
        }
        if (lane == 63) {
#pragma unroll
            for (int t = 0; t < 4; ++t) wave_tot[wave][t] = incl[t];
        }
        __syncthreads();
        int32_t prefix[4], chunk_total[4];
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            int32_t p = carry[t];
            for (int w = 0; w < wave; ++w) p += wave_tot[w][t];
            prefix[t] = p;
            chunk_total[t] = wave_tot[0][t] + wave_tot[1][t] + wave_tot[2][t] + wave_tot[3][t];
        }
        if (b < n_tiles) {
#pragma unroll
            for (int t = 0; t < 4; ++t) tile_counts[b * 4 + t] = prefix[t] + incl[t] - v[t];
        }
        __syncthreads();
        if (threadIdx.x < 4) carry[threadIdx.x] += chunk_total[threadIdx.x];
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        int32_t run = 0;
        for (int t = 0; t < 4; ++t) {
            totals[t] = carry[t];
            totals[4 + t] = run;
            counts_out[t] = carry[t];
            run += carry[t];
        }
    }
}

// Second pass.  Workgroups 0 .. n_tiles - 1: an atom's rank in its type = atoms of the type in earlier tiles + in earlier
// wavefronts of the tile + in earlier lanes.  `totals` null: tile_counts holds the tiles' histograms, which every
// workgroup adds up; otherwise tile_counts holds their exclusive sums and totals the type counts and bases (the scan
// below).  The workgroups behind them: atom counts of 256 molecules each, and the molecules per size (size_scratch
// non-null).
__global__ __launch_bounds__(kSortThreads) void prep_rank_kernel(
    const int32_t* __restrict__ A, int64_t n, unsigned n_tiles, const int32_t* __restrict__ tile_counts,
    const int32_t* __restrict__ totals, int32_t* __restrict__ scatter, int32_t* __restrict__ gather,
    int32_t* __restrict__ counts_out, const int32_t* __restrict__ MOs, int32_t n_mols, int32_t* __restrict__ MACs,
    int32_t* __restrict__ size_scratch)
{
    __shared__ int32_t shared[kSizeBins];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    if (blockIdx.x >= n_tiles) {                     // molecules
        if (size_scratch) {
            for (int k = threadIdx.x; k < kSizeBins; k += kSortThreads) shared[k] = 0;
            __syncthreads();
        }
        const int64_t m = static_cast<int64_t>(blockIdx.x - n_tiles) * kSortThreads + threadIdx.x;
        if (m < n_mols) {
            const int32_t next = (m + 1 < n_mols) ? MOs[m + 1] : static_cast<int32_t>(n);
            const int32_t count = next - MOs[m];
            MACs[m] = count;
            if (size_scratch) atomicAdd(&shared[size_bin(count)], 1);
        }
        if (size_scratch) {
            __syncthreads();
            for (int k = threadIdx.x; k < kSizeBins; k += kSortThreads)
                if (shared[k] > 0) atomicAdd(&size_scratch[k], shared[k]);
        }
        return;
    }
    const int64_t tile0 = static_cast<int64_t>(blockIdx.x) * kSortTile;
    const unsigned long long lt_mask = (1ull << lane) - 1ull;
    int types[kSortSubTiles];
#pragma unroll
    for (int s = 0; s < kSortSubTiles; ++s) {        // the tile's types, in flight while the histograms are added up
        const int64_t g = tile0 + s * kSortThreads + threadIdx.x;
        types[s] = g < n ? fold_type(A[g]) : -1;
    }
    int32_t running[4], type_base[4];
    if (totals) {
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            running[t] = tile_counts[static_cast<int64_t>(blockIdx.x) * 4 + t];
            type_base[t] = totals[4 + t];
        }
    } else {
        int32_t sum[8] = {0, 0, 0, 0, 0, 0, 0, 0};   // per type: in earlier tiles, and in all
        for (unsigned b = threadIdx.x; b < n_tiles; b += kSortThreads) {
            const int4 c = reinterpret_cast<const int4*>(tile_counts)[b];
            const bool before = b < blockIdx.x;
            sum[4] += c.x; sum[5] += c.y; sum[6] += c.z; sum[7] += c.w;
            if (before) { sum[0] += c.x; sum[1] += c.y; sum[2] += c.z; sum[3] += c.w; }
        }
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            sum[k] = wave_sum(sum[k]);
            if (lane == 0) shared[wave * 8 + k] = sum[k];
        }
        __syncthreads();
        int32_t base = 0;
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            running[t] = shared[t] + shared[8 + t] + shared[16 + t] + shared[24 + t];
            const int32_t all = shared[4 + t] + shared[12 + t] + shared[20 + t] + shared[28 + t];
            type_base[t] = base;
            base += all;
            if (blockIdx.x == 0 && threadIdx.x == 0) counts_out[t] = all;
        }
        __syncthreads();
    }
#pragma unroll
    for (int s = 0; s < kSortSubTiles; ++s) {
        const int64_t g = tile0 + s * kSortThreads + threadIdx.x;
        const int type = types[s];
        unsigned long long m[4];
        wave_type_masks(type, true, m);
        int32_t* const wave_counts = shared + (s & 1) * 16;          // two places in turn: one barrier per step
        if (lane == 0) {
#pragma unroll
            for (int t = 0; t < 4; ++t) wave_counts[wave * 4 + t] = __popcll(m[t]);
        }
        __syncthreads();
        int32_t rank = 0, tbase = 0;
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            int32_t before = running[t], all = running[t];
#pragma unroll
            for (int w = 0; w < 4; ++w) {
                const int32_t c = wave_counts[w * 4 + t];
                before += w < wave ? c : 0;
                all += c;
            }
            if (type == t) {
                rank = before + __popcll(m[t] & lt_mask);
                tbase = type_base[t];
            }
            running[t] = all;
        }
        if (type >= 0) {
            scatter[g] = rank;
            gather[g] = tbase + rank;
        }
    }
}

__global__ void zero_counts_kernel(int32_t* counts4)
{
    if (threadIdx.x < 4) counts4[threadIdx.x] = 0;
}

// clears the class counts and cursors behind a size order (a kernel and not a memset node, so that the
// sequence can be recorded into a graph)
__global__ __launch_bounds__(kSizeOrderScratch) void size_clear_kernel(int32_t* __restrict__ scratch)
{
    scratch[threadIdx.x] = 0;
}

// zeros for outputs that no molecule covers (a kernel, not a memset node: see size_clear_kernel)
template <typename T>
__global__ __launch_bounds__(256) void zero_fill_kernel(T* __restrict__ a, int64_t n)
{
    for (int64_t i = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x; i < n; i += static_cast<int64_t>(gridDim.x) * 256)
        a[i] = T(0);
}

}  // namespace

template <typename T>
hipError_t launch_zero(T* a, int64_t n, hipStream_t stream)
{
    if (n <= 0) return hipSuccess;
    const int64_t want = (n + 255) / 256;
    zero_fill_kernel<T><<<dim3(static_cast<unsigned>(want < 8192 ? want : 8192)), dim3(256), 0, stream>>>(a, n);
    return hipGetLastError();
}
template hipError_t launch_zero<float>(float*, int64_t, hipStream_t);
template hipError_t launch_zero<double>(double*, int64_t, hipStream_t);

namespace {
unsigned blocks_for(int64_t n, int64_t per) { return static_cast<unsigned>((n + per - 1) / per); }
unsigned tiles_of(int64_t n_atoms) { return n_atoms > 0 ? blocks_for(n_atoms, kSortTile) : 1u; }
}  // namespace

hipError_t launch_mol_offsets(const int32_t* mol_idxs, int64_t n_atoms, int32_t n_mols,
                              int32_t* MACs, int32_t* MOs, hipStream_t stream)
{
    if (n_mols <= 0) return hipSuccess;
    prep_count_kernel<<<dim3(tiles_of(n_atoms)), dim3(kSortThreads), 0, stream>>>(nullptr, mol_idxs, n_atoms, n_mols, nullptr, MOs, nullptr);
    prep_rank_kernel<<<dim3(blocks_for(n_mols, kSortThreads)), dim3(kSortThreads), 0, stream>>>(
        nullptr, n_atoms, 0u, nullptr, nullptr, nullptr, nullptr, nullptr, MOs, n_mols, MACs, nullptr);
    return hipGetLastError();
}

hipError_t launch_ani_sort(const int32_t* A, int64_t n_atoms, int32_t* scatter, int32_t* gather,
                           int32_t* counts4, hipStream_t stream)
{
    if (n_atoms <= 0) {
        zero_counts_kernel<<<dim3(1), dim3(64), 0, stream>>>(counts4);
        return hipGetLastError();
    }
    const unsigned n_tiles = tiles_of(n_atoms);
    int32_t* ws = nullptr;   // [n_tiles*4] tile counts (above kScanTiles then their exclusive sums), then [8] totals and type bases
    hipError_t e = hipMallocAsync(reinterpret_cast<void**>(&ws), sizeof(int32_t) * (static_cast<size_t>(n_tiles) * 4 + 8), stream);
    if (e != hipSuccess) return e;
    int32_t* totals = n_tiles > kScanTiles ? ws + static_cast<size_t>(n_tiles) * 4 : nullptr;
    prep_count_kernel<<<dim3(n_tiles), dim3(kSortThreads), 0, stream>>>(A, nullptr, n_atoms, 0, ws, nullptr, nullptr);
    if (totals) sort_scan_kernel<<<dim3(1), dim3(256), 0, stream>>>(ws, n_tiles, totals, counts4);
    prep_rank_kernel<<<dim3(n_tiles), dim3(kSortThreads), 0, stream>>>(A, n_atoms, n_tiles, ws, totals, scatter, gather, counts4,
                                                                       nullptr, 0, nullptr, nullptr);
    e = hipGetLastError();
    const hipError_t e2 = hipFreeAsync(ws, stream);
    return (e != hipSuccess) ? e : e2;
}

// ---- molecules in order of decreasing atom count ----
// Counting sort of the molecule indices by min(atom count, 257), largest first.  Two passes over the
// molecules, 1,024 per workgroup: the first adds workgroup histograms (LDS integer atomics) into a global
// one; the second recomputes its histogram, reserves a range per size class with one global atomic, and
// places its molecules inside the ranges.  The order inside a size class is whatever the atomics give,
// which no result depends on.  The one-wavefront kernels take molecule order[b] in workgroup b (the
// workgroup-per-molecule kernels walk the same order with the grid's stride): the dispatcher hands out
// workgroups in index order, so the expensive molecules start first and a launch does not end on a few
// long waves.
namespace {
constexpr int kOrderThreads = 1024;

__global__ __launch_bounds__(kOrderThreads) void size_hist_kernel(const int32_t* __restrict__ MACs, int32_t n_mols,
                                                                   int32_t* __restrict__ ghist)
{
    __shared__ int hist[kSizeBins];
    const int tid = threadIdx.x;
    if (tid < kSizeBins) hist[tid] = 0;
    __syncthreads();
    const int m = blockIdx.x * kOrderThreads + tid;
    if (m < n_mols) atomicAdd(&hist[size_bin(MACs[m])], 1);
    __syncthreads();
    if (tid < kSizeBins && hist[tid] > 0) atomicAdd(&ghist[tid], hist[tid]);
}

// Exclusive prefix sums of total[0 .. kSizeBins) into start (shared arrays), by the first wavefront, 64 bins at a time
__device__ __forceinline__ void bin_starts(const int* total, int* start)
{
    if (threadIdx.x < 64) {
        int carry = 0;
        for (int b0 = 0; b0 < kSizeBins; b0 += 64) {
            const int b = b0 + static_cast<int>(threadIdx.x);
            const int v = b < kSizeBins ? total[b] : 0;
            int x = v;
#pragma unroll
            for (int d = 1; d < 64; d <<= 1) {
                const int y = __shfl_up(x, d, 64);
                if (static_cast<int>(threadIdx.x) >= d) x += y;
            }
            if (b < kSizeBins) start[b] = carry + x - v;
            carry += __shfl(x, 63, 64);
        }
    }
}

// Molecules of up to 32, of 33..64, of 65..256 and of more atoms (class c), from the starts of the bins (largest sizes
// first) and the number of molecules.
__device__ __forceinline__ int class_total(int c, const int* start, int n_mols)
{
    const int lo = c == 0 ? 0 : c == 1 ? 33 : c == 2 ? 65 : 257;          // atom counts of the class
    const int hi = c == 0 ? 32 : c == 1 ? 64 : c == 2 ? 256 : 257;
    const int last = size_bin(lo);
    return (last + 1 < kSizeBins ? start[last + 1] : n_mols) - start[size_bin(hi)];
}

// host8 (may be null): host memory that the GPU can write, for the four atom counts and the four class totals
__global__ __launch_bounds__(kOrderThreads) void size_place_kernel(const int32_t* __restrict__ MACs, int32_t n_mols,
                                                                    const int32_t* __restrict__ ghist,
                                                                    int32_t* __restrict__ gcursor,
                                                                    int32_t* __restrict__ order,
                                                                    const int32_t* __restrict__ counts4, int32_t* __restrict__ host8)
{
    __shared__ int hist[kSizeBins];     // this workgroup's molecules per class, then its cursor inside the range
    __shared__ int start[kSizeBins];    // first position of the class in the order, then of this workgroup's range
    __shared__ int total[kSizeBins];    // molecules per class in the whole batch
    const int tid = threadIdx.x;
    if (tid < kSizeBins) {
        hist[tid] = 0;
        total[tid] = ghist[tid];
    }
    __syncthreads();
    const int m = blockIdx.x * kOrderThreads + tid;
    int bin = 0;
    if (m < n_mols) {
        bin = size_bin(MACs[m]);
        atomicAdd(&hist[bin], 1);
    }
    bin_starts(total, start);
    __syncthreads();
    // the four totals that tell a host which kernels have work (behind the cursors)
    if (blockIdx.x == 0 && tid < kSizeClasses) {
        const int sum = class_total(tid, start, n_mols);
        gcursor[kSizeBins + tid] = sum;
        if (host8) {
            host8[tid] = counts4[tid];
            host8[kSizeClasses + tid] = sum;
        }
    }
    __syncthreads();
    if (tid < kSizeBins) {
        const int mine = hist[tid];
        if (mine > 0) start[tid] += atomicAdd(&gcursor[tid], mine);
        hist[tid] = 0;
    }
    __syncthreads();
    if (m < n_mols) order[start[bin] + atomicAdd(&hist[bin], 1)] = m;
}

// The whole preparation of a small batch in one workgroup: what prep_count, prep_rank and size_place do, with barriers in
// place of launches.  A wavefront ranks 64 kPer consecutive atoms, 64 at a time; where it counts them, the four types'
// counts ride in one 64-bit word, 16 bits each.  What bounds it is latency: its loads are all in flight at once, and the
// rest is one compute unit's instruction rate.
constexpr int kSmallPrepPer = 16;            // most atoms per thread
constexpr int kSmallPrepAtoms = kSmallPrepPer * kOrderThreads, kSmallPrepMols = 2 * kOrderThreads;
template <int kPer>
__global__ __launch_bounds__(kOrderThreads) void prep_small_kernel(const int32_t* __restrict__ A, const int32_t* __restrict__ mol_idxs,
                                                                   int n, int32_t n_mols, int32_t* MACs, int32_t* MOs,
                                                                   int32_t* __restrict__ scatter, int32_t* __restrict__ gather,
                                                                   int32_t* __restrict__ counts4, int32_t* __restrict__ order,
                                                                   int32_t* __restrict__ host8)
{
    __shared__ int hist[kSizeBins], start[kSizeBins], mol_start[kSmallPrepMols + 1];
    __shared__ unsigned long long wave_total[kOrderThreads / 64];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    if (tid < kSizeBins) hist[tid] = 0;
    const int first = wave * 64 * kPer + lane;           // this lane's atoms: first, first + 64, ...
    int type[kPer];
    {
        int id[kPer], prev[kPer];
#pragma unroll
        for (int k = 0; k < kPer; ++k) {
            const int g = first + 64 * k;
            type[k] = g < n ? A[g] : -1;
            id[k] = g < n ? mol_idxs[g] : 0;
            prev[k] = g < n && g > 0 ? mol_idxs[g - 1] : -1;
        }
#pragma unroll
        for (int k = 0; k < kPer; ++k) {
            const int g = first + 64 * k;
            if (g < n) {
                type[k] = fold_type(type[k]);
                if (id[k] != prev[k]) mol_starts(prev[k], id[k], g, n_mols, mol_start);
            }
        }
    }
    if (tid == 0) {
        mol_bounds(mol_idxs, n, n, n_mols, mol_start);
        mol_start[n_mols] = n;
    }
    unsigned long long mine = 0;
#pragma unroll
    for (int k = 0; k < kPer; ++k) mine += type[k] >= 0 ? 1ull << (16 * type[k]) : 0ull;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) mine += __shfl_xor(mine, d, 64);
    if (lane == 0) wave_total[wave] = mine;
    __syncthreads();                    // the molecules' starts and the wavefronts' totals are complete
    int bin[kSmallPrepMols / kOrderThreads];
#pragma unroll
    for (int k = 0; k < kSmallPrepMols / kOrderThreads; ++k) {
        const int m = k * kOrderThreads + tid;
        if (m < n_mols) {
            const int at = mol_start[m], c = mol_start[m + 1] - at;
            MOs[m] = at;
            MACs[m] = c;
            bin[k] = size_bin(c);
            atomicAdd(&hist[bin[k]], 1);
        }
    }
    unsigned long long before = 0, all = 0;
#pragma unroll
    for (int w = 0; w < kOrderThreads / 64; ++w) {
        if (w < wave) before += wave_total[w];
        all += wave_total[w];
    }
    int count[4], base[4], running[4];
#pragma unroll
    for (int t = 0; t < 4; ++t) {
        count[t] = static_cast<int>((all >> (16 * t)) & 0xffffu);
        running[t] = __builtin_amdgcn_readfirstlane(static_cast<int>((before >> (16 * t)) & 0xffffu));
        base[t] = t == 0 ? 0 : base[t - 1] + count[t - 1];
    }
    __syncthreads();                    // the molecules per size are complete
    int32_t* const scratch = order + n_mols;         // the counts, the cursors (as they end), the class totals
    if (wave == 0) {
        // what a host waits for comes first: it prepares its next launch while the ranks are still written
        bin_starts(hist, start);
        __threadfence_block();
        if (lane < kSizeClasses) {
            const int sum = class_total(lane, start, n_mols);
            const int c = lane == 0 ? count[0] : lane == 1 ? count[1] : lane == 2 ? count[2] : count[3];
            if (host8) {
                host8[lane] = c;
                host8[kSizeClasses + lane] = sum;
            }
            scratch[2 * kSizeBins + lane] = sum;
            counts4[lane] = c;
        }
    }
#pragma unroll
    for (int k = 0; k < kPer; ++k) {
        const int g = first + 64 * k;
        if (wave * 64 * kPer + 64 * k >= n) break;
        int rank = 0, at = 0;
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            const unsigned long long m = wave_ballot(type[k] == t);
            const int r = running[t] + static_cast<int>(__builtin_amdgcn_mbcnt_hi(static_cast<unsigned>(m >> 32),
                                                                                  __builtin_amdgcn_mbcnt_lo(static_cast<unsigned>(m), 0u)));
            rank = type[k] == t ? r : rank;
            at = type[k] == t ? base[t] + r : at;
            running[t] += __popcll(m);
        }
        if (g < n && type[k] >= 0) {
            scatter[g] = rank;
            gather[g] = at;
        }
    }
    __syncthreads();                    // the sizes' first positions are complete
    if (tid < kSizeBins) {
        scratch[tid] = hist[tid];
        scratch[kSizeBins + tid] = hist[tid];
    }
#pragma unroll
    for (int k = 0; k < kSmallPrepMols / kOrderThreads; ++k) {
        const int m = k * kOrderThreads + tid;
        if (m < n_mols) order[atomicAdd(&start[bin[k]], 1)] = m;
    }
}
}  // namespace

// `order` holds n_mols + kSizeOrderScratch entries of device memory owned by the caller: the indices, the class
// counts, the cursors.
hipError_t launch_size_order(const int32_t* MACs, int32_t n_mols, int32_t* order, hipStream_t stream)
{
    if (n_mols <= 0) return hipSuccess;
    int32_t* scratch = order + n_mols;
    size_clear_kernel<<<dim3(1), dim3(kSizeOrderScratch), 0, stream>>>(scratch);
    const unsigned blocks = (static_cast<unsigned>(n_mols) + kOrderThreads - 1) / kOrderThreads;
    size_hist_kernel<<<dim3(blocks), dim3(kOrderThreads), 0, stream>>>(MACs, n_mols, scratch);
    size_place_kernel<<<dim3(blocks), dim3(kOrderThreads), 0, stream>>>(MACs, n_mols, scratch, scratch + kSizeBins, order, nullptr, nullptr);
    return hipGetLastError();
}

size_t prepare_workspace_bytes(int64_t n_atoms) { return sizeof(int32_t) * (static_cast<size_t>(tiles_of(n_atoms)) * 4 + 8); }

// launch_mol_offsets + launch_ani_sort + launch_size_order together, n_mols > 0.  `ws`: prepare_workspace_bytes(n_atoms)
// bytes, 16-byte aligned.
hipError_t launch_prepare(const int32_t* mol_idxs, const int32_t* A, int64_t n_atoms, int32_t n_mols, int32_t* MACs, int32_t* MOs,
                          int32_t* scatter, int32_t* gather, int32_t* counts4, int32_t* order, int32_t* ws, int32_t* host8,
                          hipStream_t stream)
{
    // one workgroup up to 16,384 atoms (the reference trainer's batch of 1,024 organic molecules is
    // 13,000: 9 us, where the three launches take 20 and the gaps between them), 5 us up to 4,096; above, one compute unit is slower
    if (n_atoms <= kSmallPrepAtoms && n_mols <= kSmallPrepMols) {
        const auto kernel = n_atoms <= 4 * kOrderThreads ? prep_small_kernel<4> : prep_small_kernel<kSmallPrepPer>;
        kernel<<<dim3(1), dim3(kOrderThreads), 0, stream>>>(A, mol_idxs, static_cast<int>(n_atoms), n_mols, MACs, MOs, scatter, gather,
                                                            counts4, order, host8);
        return hipGetLastError();
    }
    const unsigned n_tiles = tiles_of(n_atoms);
    int32_t* const totals = n_tiles > kScanTiles ? ws + static_cast<size_t>(n_tiles) * 4 : nullptr;
    int32_t* const scratch = order + n_mols;
    prep_count_kernel<<<dim3(n_tiles), dim3(kSortThreads), 0, stream>>>(A, mol_idxs, n_atoms, n_mols, ws, MOs, scratch);
    if (totals) sort_scan_kernel<<<dim3(1), dim3(256), 0, stream>>>(ws, n_tiles, totals, counts4);
    prep_rank_kernel<<<dim3(n_tiles + blocks_for(n_mols, kSortThreads)), dim3(kSortThreads), 0, stream>>>(
        A, n_atoms, n_tiles, ws, totals, scatter, gather, counts4, MOs, n_mols, MACs, scratch);
    size_place_kernel<<<dim3(blocks_for(n_mols, kOrderThreads)), dim3(kOrderThreads), 0, stream>>>(MACs, n_mols, scratch, scratch + kSizeBins,
                                                                                                  order, counts4, host8);
    return hipGetLastError();
}

}  // namespace khan
