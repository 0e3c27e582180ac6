// Sorted copies of the molecules of more than 256 atoms, for the workgroup-per-molecule AEV kernels (aev_large.h).
// One workgroup per molecule: a counting sort by (cell along a space-filling curve, atom type) that keeps the atoms'
// order inside a bin, and the box around every 64 consecutive sorted atoms; and the list of what those kernels share out among them.
#include <algorithm>

#include "aev_large.h"
#include "khan_params.h"

namespace khan {

namespace {

__device__ __forceinline__ int spread4(int v) { return (v & 1) | ((v & 2) << 2) | ((v & 4) << 4) | ((v & 8) << 6); }

// minimum / maximum over the wavefront
__device__ __forceinline__ float wave_min(float v)
{
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) v = fminf(v, __shfl_xor(v, d, 64));
    return v;
}
__device__ __forceinline__ float wave_maxf(float v)
{
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) v = fmaxf(v, __shfl_xor(v, d, 64));
    return v;
}

// Lists the units of the large molecules (SortedAtoms): kListers workgroups, each of which goes through all molecules, 2,048 at a time, and
// writes its share of every one's units (one workgroup alone takes 44 us for the 43,000 units of 64 boxes of 1,024-4,096 atoms).
constexpr int kListers = 16;
template <typename T>
__device__ __forceinline__ void list_units(const int32_t* __restrict__ MACs, int32_t n_mols, const int32_t* __restrict__ order, const SortedAtoms<T>& sorted,
                                           int (&wave_units)[4])
{
    constexpr int kEach = 8;                    // molecules of a thread, their loads in flight together (without an order all have to be looked at)
    const int tid = threadIdx.x, lane = tid & 63, wave = uniform(tid >> 6);
    const int count = order ? order[n_mols + size_bin(kMediumMaxAtoms + 1)] : n_mols;      // (they are the first of the order)
    int total = 0;
    for (int64_t m0 = 0; m0 < count; m0 += kEach * 256) {
        int mol[kEach], n[kEach], units = 0;
#pragma unroll
        for (int k = 0; k < kEach; ++k) {
            const int64_t m = m0 + k * 256 + tid;
            mol[k] = m < count ? (order ? order[m] : static_cast<int>(m)) : -1;
        }
#pragma unroll
        for (int k = 0; k < kEach; ++k) n[k] = mol[k] >= 0 ? MACs[mol[k]] : 0;
        const auto units_of = [](int atoms) { return atoms > kMediumMaxAtoms ? (atoms + kRunCentres - 1) >> kLogRunCentres : 0; };
#pragma unroll
        for (int k = 0; k < kEach; ++k) units += units_of(n[k]);
        int end = units;
#pragma unroll
        for (int d = 1; d < 64; d <<= 1) {
            const int before = __shfl_up(end, d, 64);
            end += lane >= d ? before : 0;
        }
        if (lane == 63) wave_units[wave] = end;
        __syncthreads();
        const int all[4] = {wave_units[0], wave_units[1], wave_units[2], wave_units[3]};
        int begin = total + (wave > 0 ? all[0] : 0) + (wave > 1 ? all[1] : 0) + (wave > 2 ? all[2] : 0) + end - units;
#pragma unroll
        for (int k = 0; k < kEach; ++k) {
            for (unsigned long long left = wave_ballot(n[k] > kMediumMaxAtoms); left; left &= left - 1) {
                const int b = lowest_bit(left), of = lane_read(mol[k], b), atoms = lane_read(n[k], b), at = lane_read(begin, b), most = units_of(atoms);
                for (int u = 64 * static_cast<int>(blockIdx.x) + lane; u < most; u += 64 * kListers) {
                    const int first = u << kLogRunCentres;
                    // (more than there is room for: the molecules overlap)
                    if (at + u < sorted.most_units) sorted.unit[at + u] = make_int2(of, (first << kLogRunCentres) + min(atoms - first, kRunCentres) - 1);
                }
            }
            begin += units_of(n[k]);
        }
        total += (all[0] + all[1]) + (all[2] + all[3]);
        __syncthreads();                        // the next molecules' counts go to the same places
    }
    if (blockIdx.x == 0 && tid == 0) *sorted.n_units = min(total, sorted.most_units);
}

constexpr int kListedAtoms = 64;      // of a bin, at most, where atoms are ranked by their bins' lists

template <typename T>
__global__ __launch_bounds__(256) void large_sort_kernel(
    const T* __restrict__ X, const T* __restrict__ Y, const T* __restrict__ Z,
    const int32_t* __restrict__ A, const int32_t* __restrict__ MOs,
    const int32_t* __restrict__ MACs, int32_t n_mols, const int32_t* __restrict__ SIs,
    const T* __restrict__ VX, const T* __restrict__ VY, const T* __restrict__ VZ,
    T* __restrict__ gX, T* __restrict__ gY, T* __restrict__ gZ, const int32_t* __restrict__ order,
    SortedAtoms<T> sorted)
{
    __shared__ int hist[4 * kSortCells];       // atoms per (cell, type); after the scan each one's next free sorted position
    __shared__ int in_step[4 * kSortCells];    // atoms per (cell, type) among the 256 of the current step (zero between steps)
    __shared__ __align__(16) int2 shared_bin[256];           // (key, thread) of the step's atoms that share their bin with another
    __shared__ int wshared[4];                 // how many of them each wavefront holds
    __shared__ __align__(16) int step_key[256];              // keys of the 256 atoms of the current step
    __shared__ float ext[4][6];                // each wavefront's share of the molecule's extent
    __shared__ int wsum[4], wtop[4];
    __shared__ unsigned long long want[4];
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = uniform(tid >> 6);
    if (blockIdx.y == 0) {                     // (the first to start)
        if (blockIdx.x < kListers) list_units(MACs, n_mols, order, sorted, wsum);
        return;
    }
    for_each_molecule_in_range(MACs, n_mols, kMediumMaxAtoms + 1, INT32_MAX, want, order, order ? order + n_mols : nullptr, [&](int mol) {
        const int n = uniform(MACs[mol]);
        const int off = uniform(MOs[mol]);

        // ---- the molecule's extent, and the cell grid over it
        float lo[3] = {3.0e38f, 3.0e38f, 3.0e38f}, hi[3] = {-3.0e38f, -3.0e38f, -3.0e38f};
        // (one workgroup walks the whole molecule: eight atoms' loads in flight per thread in this and the next loops, past
        // the end the last atom again, because a load under a condition is waited for on the spot)
        for (int base = tid; base < n; base += 8 * 256) {
#pragma unroll
            for (int u = 0; u < 8; ++u) {
                const int j = off + min(base + 256 * u, n - 1);
                const float p[3] = {static_cast<float>(X[j]), static_cast<float>(Y[j]), static_cast<float>(Z[j])};
#pragma unroll
                for (int k = 0; k < 3; ++k) {
                    lo[k] = fminf(lo[k], p[k]);
                    hi[k] = fmaxf(hi[k], p[k]);
                }
            }
        }
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            lo[k] = wave_min(lo[k]);
            hi[k] = wave_maxf(hi[k]);
        }
        if (lane == 0) {
#pragma unroll
            for (int k = 0; k < 3; ++k) {
                ext[wave][k] = lo[k];
                ext[wave][3 + k] = hi[k];
            }
        }
        __syncthreads();
        // cells per dimension: 4, 8 or 16 by the molecule's size (a chunk of 64 atoms spans several cells either way,
        // and the bins' bookkeeping below grows with the cube of it)
        const int g = n <= 1024 ? 4 : n <= 8192 ? 8 : kSortCellsPerDim;
        const int cells = g * g * g, bins = 4 * cells, per_thread = bins / 256;
        float scale[3];
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            lo[k] = fminf(fminf(ext[0][k], ext[1][k]), fminf(ext[2][k], ext[3][k]));
            hi[k] = fmaxf(fmaxf(ext[0][3 + k], ext[1][3 + k]), fmaxf(ext[2][3 + k], ext[3][3 + k]));
            scale[k] = static_cast<float>(g) / fmaxf(hi[k] - lo[k], 1.0e-3f);
        }
        // (cell, type) of an atom: the cell's index along the space-filling curve, then the type
        auto bin_of = [&](T x, T y, T z, int type) -> int {
            const float p[3] = {static_cast<float>(x), static_cast<float>(y), static_cast<float>(z)};
            int c[3];
#pragma unroll
            for (int k = 0; k < 3; ++k) c[k] = min(max(static_cast<int>((p[k] - lo[k]) * scale[k]), 0), g - 1);
            return (spread4(c[0]) | (spread4(c[1]) << 1) | (spread4(c[2]) << 2)) * 4 + type;
        };
        // body(j, bin) for this thread's atoms j
        auto for_each_bin = [&](auto&& body) {
            for (int base = tid; base < n; base += 8 * 256) {
                int key[8];
#pragma unroll
                for (int u = 0; u < 8; ++u) {
                    const int j = off + min(base + 256 * u, n - 1);
                    key[u] = bin_of(X[j], Y[j], Z[j], fold_type(A[j]));
                }
#pragma unroll
                for (int u = 0; u < 8; ++u)
                    if (base + 256 * u < n) body(base + 256 * u, key[u]);
            }
        };

        // ---- atoms per (cell, type)
        for (int b = tid; b < bins; b += 256) {
            hist[b] = 0;
            in_step[b] = 0;
        }
        __syncthreads();
        for_each_bin([&](int, int key) { atomicAdd(&hist[key], 1); });
        __syncthreads();
        // ---- exclusive prefix sum over the bins: per_thread consecutive bins per thread
        {
            int local = 0, top = 0;
            for (int q = 0; q < per_thread; ++q) {
                local += hist[per_thread * tid + q];
                top = max(top, hist[per_thread * tid + q]);
            }
#pragma unroll
            for (int d = 1; d < 64; d <<= 1) top = max(top, __shfl_xor(top, d, 64));
            if (lane == 0) wtop[wave] = top;
            int incl = local;
#pragma unroll
            for (int d = 1; d < 64; d <<= 1) {
                const int v = __shfl_up(incl, d, 64);
                if (lane >= d) incl += v;
            }
            if (lane == 63) wsum[wave] = incl;
            __syncthreads();
            int run = incl - local;
            for (int w = 0; w < wave; ++w) run += wsum[w];
            for (int q = 0; q < per_thread; ++q) {
                const int c = hist[per_thread * tid + q];
                hist[per_thread * tid + q] = run;
                run += c;
            }
        }
        __syncthreads();

        // ---- place the atoms in index order inside a (cell, type): the result does not depend on timing.
        struct Fetched {
            T x, y, z, vx, vy, vz;
            int type, si;
        };
        auto fetch = [&](int j) -> Fetched {                      // (past the end: the last atom)
            const int at = off + min(j, n - 1);
            Fetched f;
            f.x = X[at];
            f.y = Y[at];
            f.z = Z[at];
            f.type = fold_type(A[at]);
            f.si = SIs[at];
            f.vx = f.vy = f.vz = T(0);
            if (sorted.vel) {
                f.vx = VX[at];
                f.vy = VY[at];
                f.vz = VZ[at];
            }
            return f;
        };
        auto place = [&](int j, int dest, const Fetched& f) {
            T word;
            set_atom_word(word, (f.type << kTypeShift) | f.si);
            sorted.atom[dest] = Fast<T>::make4(f.x, f.y, f.z, word);
            sorted.index[dest] = off + j;
            if (sorted.vel) sorted.vel[dest] = Fast<T>::make4(f.vx, f.vy, f.vz, T(0));
            if (gX) {
                if (sorted.force) sorted.force[dest] = Fast<T>::make4(T(0), T(0), T(0), T(0));
                gX[off + j] = T(0);
                gY[off + j] = T(0);
                gZ[off + j] = T(0);
            }
        };
        if (n <= 4 * kSortCells && max(max(wtop[0], wtop[1]), max(wtop[2], wtop[3])) <= kListedAtoms) {
            // The atoms' indices are listed by bin in whatever order they come (in LDS, one entry per atom), and an atom's
            // rank is the number of smaller indices in its bin: three passes over the atoms without a barrier inside,
            // where steps of 256 need five each.  The lists have room for 16,384 atoms, and a bin's are read by each of
            // its atoms: for bins of up to 64 (a few in a molecule that fills its extent; 1,024-4,096 atoms: 106 -> 37 us with the boxes below).
            int* list = in_step;
            for_each_bin([&](int j, int key) { list[atomicAdd(&hist[key], 1)] = j; });
            __syncthreads();                        // hist[b] is the end of bin b now
            for (int base = tid; base < n; base += 4 * 256) {
                Fetched f[4];
#pragma unroll
                for (int u = 0; u < 4; ++u) f[u] = fetch(base + 256 * u);
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    const int j = base + 256 * u;
                    if (j >= n) break;
                    const int key = bin_of(f[u].x, f[u].y, f[u].z, f[u].type);
                    const int first = key == 0 ? 0 : hist[key - 1], end = hist[key];
                    int rank = 0;
                    for (int q = first; q < end; ++q) rank += list[q] < j;
                    place(j, off + first + rank, f[u]);
                }
            }
        } else {
            // 256 per step; an atom's data are fetched one step ahead, so that the loads run under the previous step's ranking
            Fetched next = fetch(tid);
            for (int base = 0; base < n; base += 256) {
                const int j = base + tid;
                const bool have = j < n;
                const Fetched cur = next;
                next = fetch(j + 256);
                int key = -1 - tid;                                    // (no two threads without an atom match)
                if (have) key = bin_of(cur.x, cur.y, cur.z, cur.type);
                // Rank among the step's atoms of the same bin, by thread.  In a large molecule most atoms are alone in their
                // bin within a step: the atoms that are not are listed (in thread order) and only they compare keys, with
                // that list.  When the list is long (small molecules, few bins) every atom compares with the 255 others.
                step_key[tid] = key;
                if (have) atomicAdd(&in_step[key], 1);
                __syncthreads();
                const bool shares = have && in_step[key] > 1;
                const unsigned long long smask = wave_ballot(shares);
                if (lane == 0) wshared[wave] = popc64(smask);
                __syncthreads();
                int before = 0, n_shared = 0;
                for (int w = 0; w < 4; ++w) {
                    before += w < wave ? wshared[w] : 0;
                    n_shared += wshared[w];
                }
                if (shares) shared_bin[before + popc64(smask & ((1ull << lane) - 1ull))] = make_int2(key, tid);
                __syncthreads();
                int rank = 0;
                if (n_shared > 48) {
#pragma unroll 8
                    for (int t = 0; t < 256; t += 4) {
                        const int4 k4 = *reinterpret_cast<const int4*>(&step_key[t]);
                        rank += (k4.x == key && t < tid) + (k4.y == key && t + 1 < tid) + (k4.z == key && t + 2 < tid) +
                                (k4.w == key && t + 3 < tid);
                    }
                } else if (shares) {
                    for (int q = 0; q < n_shared; ++q) {
                        const int2 e = shared_bin[q];
                        rank += (e.x == key && e.y < tid);
                    }
                }
                const int dest = have ? off + hist[key] + rank : 0;
                __syncthreads();                    // every thread has read its bin's position and the step's counts
                if (have) in_step[key] = 0;
                if (have) {
                    atomicAdd(&hist[key], 1);
                    place(j, dest, cur);
                }
                __syncthreads();                    // the bins are up to date, the keys may be overwritten
            }
        }

        // ---- the box around every 64 consecutive sorted atoms
        // The barrier orders the workgroup's stores to sorted.atom before its loads of them: one compute unit's, through one cache.
        // (A fence for the whole device beside it had the second-level cache written back: 34.3 -> 29.7 us.)
        __syncthreads();
        const size_t cb = chunk_base(off, mol);
        const int n_chunks = (n + 63) >> 6;
        // four neighbouring lanes per chunk, sixteen atoms each, their loads in flight together (a wavefront per chunk spent
        // most of the kernel in its 36 lane exchanges: 4,096 atoms are 64 chunks on four wavefronts, 20 us of 56)
        for (int c0 = 0; c0 < n_chunks; c0 += 64) {
            const int c = c0 + (tid >> 2), sub = tid & 3;
            float blo[3] = {3.0e38f, 3.0e38f, 3.0e38f}, bhi[3] = {-3.0e38f, -3.0e38f, -3.0e38f};
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                // (past the end the last atom again, which is in the last chunk)
                const typename Fast<T>::vec4 a = sorted.atom[off + min(64 * c + 4 * i + sub, n - 1)];
                const float p[3] = {static_cast<float>(a.x), static_cast<float>(a.y), static_cast<float>(a.z)};
#pragma unroll
                for (int k = 0; k < 3; ++k) {
                    blo[k] = fminf(blo[k], p[k]);
                    bhi[k] = fmaxf(bhi[k], p[k]);
                }
            }
#pragma unroll
            for (int k = 0; k < 3; ++k)
#pragma unroll
                for (int d = 1; d < 4; d <<= 1) {
                    blo[k] = fminf(blo[k], __shfl_xor(blo[k], d, 64));
                    bhi[k] = fmaxf(bhi[k], __shfl_xor(bhi[k], d, 64));
                }
            if (sub == 0 && c < n_chunks) {
                sorted.box[2 * (cb + c)] = make_float4(blo[0], blo[1], blo[2], 0.0f);
                sorted.box[2 * (cb + c) + 1] = make_float4(bhi[0], bhi[1], bhi[2], 0.0f);
            }
        }
        __syncthreads();                        // the next molecule reuses the shared arrays
    });
}

}  // namespace

template <typename T>
hipError_t launch_large_sort(const T* X, const T* Y, const T* Z, const int32_t* A, const int32_t* MOs,
                             const int32_t* MACs, int32_t n_mols, const int32_t* SIs, const T* VX, const T* VY,
                             const T* VZ, T* gX, T* gY, T* gZ, const int32_t* order, SortedAtoms<T> sorted,
                             hipStream_t stream)
{
    if (n_mols <= 0) return hipSuccess;
    const unsigned blocks = static_cast<unsigned>(n_mols < 1024 ? n_mols : 1024);
    large_sort_kernel<T><<<dim3(std::max(blocks, static_cast<unsigned>(kListers)), 2), dim3(256), 0, stream>>>(X, Y, Z, A, MOs, MACs, n_mols, SIs, VX, VY, VZ, gX, gY, gZ,
                                                             order, sorted);
    return hipGetLastError();
}

template hipError_t launch_large_sort<float>(const float*, const float*, const float*, const int32_t*, const int32_t*, const int32_t*, int32_t, const int32_t*, const float*, const float*, const float*, float*, float*, float*, const int32_t*, SortedAtoms<float>, hipStream_t);
template hipError_t launch_large_sort<double>(const double*, const double*, const double*, const int32_t*, const int32_t*, const int32_t*, int32_t, const int32_t*, const double*, const double*, const double*, double*, double*, double*, const int32_t*, SortedAtoms<double>, hipStream_t);

}  // namespace khan
