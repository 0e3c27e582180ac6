// Molecules of more than 256 atoms: the sorted copy of their atoms that the workgroup-per-molecule kernels read in
// place of their LDS arrays, and the kernel that writes it.
//
// Up to 256 atoms a workgroup sorts its molecule into LDS itself.  Above that the sorted atoms live in device
// memory (a molecule of a few thousand atoms stays in L2), written once per call by large_sort_kernel, and a molecule's
// centres are dealt to single wavefronts in short runs.  The atoms are sorted along a space-filling curve (by type inside a cell),
// and every 64 consecutive ones have a box around them: for a run the atoms in its reach are listed from the chunks whose box
// reaches into its cutoff, a centre tests those, and puts the partners it finds in order of type afterwards.  The partner lists, the segment tables and the
// angular phases are those of the smaller molecules; only where an atom is read from differs.
#pragma once
#include "aev_small_common.h"
#include "khan_params.h"

namespace khan {

// The work of the kernels for large molecules: a workgroup is one wavefront and takes runs of 2^log_run (up to kRunCentres)
// consecutive sorted atoms of a molecule, which lie close together.
// (A molecule to a column of 64 workgroups and 32 columns side by side kept 62 % of the wavefront slots busy on 64 boxes of
// 1,024-4,096 atoms: a column's molecules add up as they come.)
constexpr int kLogRunCentres = 2, kRunCentres = 1 << kLogRunCentres;
constexpr int kMaxCandidates = 176;        // atoms in reach of a run's centres (list_candidates)

// Long runs share a list of candidates, short ones spread a small batch over the GPU, where a centre takes 8-10 us whatever goes on
// beside it.  By the atoms of the large molecules (forward / backward with the sort, us, runs of 4, 2 and 1; boxes of
// 1,024-4,096 atoms in float32: 171,000 atoms 277 / 348, 302 / 394, 377 / 503; 64,000 143 / 171, 145 / 180, 173 / 219; 21,000
// 103 / 111, 88 / 100, 91 / 111; 8,000 81 / 86, 63 / 71, 60 / 70; 2,700 78 / 83, 58 / 64, 48 / 53; in float64 43,000 211 / 241,
// 210 / 247, 245 / 303), and not by those of the batch.
__device__ __forceinline__ int log_run_for(int64_t atoms) { return atoms >= 40000 ? 2 : atoms >= 9000 ? 1 : 0; }

// An atom's type and its scatter index (the row inside its type's bucket) in one word, which travels with the coordinates: a
// partner's row and block are known where it is found.  (Rows fit 28 bits: 2^28 of them are 400 GB.)
constexpr int kTypeShift = 28;
constexpr int kPlaceMask = (1 << kTypeShift) - 1;
__device__ __forceinline__ int atom_word(float w) { return __float_as_int(w); }
__device__ __forceinline__ int atom_word(double w) { return static_cast<int>(w); }
__device__ __forceinline__ void set_atom_word(float& w, int word) { w = __int_as_float(word); }
__device__ __forceinline__ void set_atom_word(double& w, int word) { w = static_cast<double>(word); }

template <typename T>
struct SortedAtoms {
    typename Fast<T>::vec4* atom;   // x, y, z, and the word (atom_word) of the atom at MOs[mol] + sorted position
    typename Fast<T>::vec4* vel;    // its incoming vector (Jacobian-vector product only), else null
    typename Fast<T>::vec4* force;  // the sum of the forces on it (backward pass, see there), else null
    int* index;                     // its index in the batch
    float4* box;                    // per chunk of 64 sorted atoms: lowest x, y, z and highest x, y, z (two entries)
    // The large molecules cut into units of kRunCentres sorted atoms (the last one of a molecule may be shorter), one after the other: molecule,
    // and 4 x first sorted atom + atoms - 1.  A run is a unit or an even part of one.
    int2* unit;
    int* n_units;
    int most_units;                 // that there is room for
};

// The atoms are ordered along a space-filling curve (up to 16 x 16 x 16 cells over the molecule's extent, Morton order;
// by type inside a cell), so that 64 consecutive atoms sit close together and a centre can skip the chunks whose box lies beyond its
// cutoff.  The boxes of molecule `mol` (atoms from offset `off`) start at entry 2 * chunk_base(off, mol): molecule m has
// at most macs[m] / 64 + 1 chunks, so these ranges are disjoint as long as the offsets increase with the molecule index
// and the molecules do not overlap (the exclusive prefix sum of the atom counts; stated as a precondition in khan_aev.h).
__host__ __device__ __forceinline__ size_t chunk_base(int off, int mol) { return static_cast<size_t>(off >> 6) + static_cast<size_t>(mol); }
constexpr int kSortCellsPerDim = 16;
constexpr int kSortCells = kSortCellsPerDim * kSortCellsPerDim * kSortCellsPerDim;

__host__ __device__ __forceinline__ size_t round_up_256(size_t v) { return (v + 255u) & ~static_cast<size_t>(255u); }

// a unit per four atoms, and one more per molecule of more than 256
__host__ inline int64_t most_units(int64_t n_atoms) { return n_atoms / kRunCentres + n_atoms / (kMediumMaxAtoms + 1); }

template <typename T>
__host__ inline size_t sorted_atoms_bytes(int64_t n_atoms, int32_t n_mols, bool with_vectors)
{
    const size_t vec = round_up_256(sizeof(typename Fast<T>::vec4) * static_cast<size_t>(n_atoms));
    return vec * (with_vectors ? 2 : 1) + round_up_256(sizeof(int) * static_cast<size_t>(n_atoms)) +
           round_up_256(2 * sizeof(float4) * (static_cast<size_t>(n_atoms) / 64 + static_cast<size_t>(n_mols) + 1)) +
           256 + sizeof(int2) * static_cast<size_t>(most_units(n_atoms));
}

// the arrays inside one allocation of sorted_atoms_bytes (256-byte aligned)
template <typename T>
__host__ inline SortedAtoms<T> carve_sorted_atoms(void* scratch, int64_t n_atoms, int32_t n_mols, bool with_vel, bool with_force)
{
    typedef typename Fast<T>::vec4 vec4;
    char* p = static_cast<char*>(scratch);
    const size_t vec = round_up_256(sizeof(vec4) * static_cast<size_t>(n_atoms));
    SortedAtoms<T> s;
    s.atom = reinterpret_cast<vec4*>(p);
    p += vec;
    s.vel = with_vel ? reinterpret_cast<vec4*>(p) : nullptr;
    s.force = with_force ? reinterpret_cast<vec4*>(p) : nullptr;
    if (with_vel || with_force) p += vec;
    s.index = reinterpret_cast<int*>(p);
    p += round_up_256(sizeof(int) * static_cast<size_t>(n_atoms));
    s.box = reinterpret_cast<float4*>(p);
    p += round_up_256(2 * sizeof(float4) * (static_cast<size_t>(n_atoms) / 64 + static_cast<size_t>(n_mols) + 1));
    s.n_units = reinterpret_cast<int*>(p);
    s.unit = reinterpret_cast<int2*>(p + 256);
    s.most_units = static_cast<int>(most_units(n_atoms));
    return s;
}

// Does the box blo .. bhi come within the radial cutoff of the box lo .. hi?  Boxes are in float whatever the precision of the
// coordinates: the margin covers their rounding.
__device__ __forceinline__ bool in_reach(const float (&lo)[3], const float (&hi)[3], const float4& blo, const float4& bhi)
{
    const float dx = fmaxf(fmaxf(blo.x - hi[0], lo[0] - bhi.x), 0.0f);
    const float dy = fmaxf(fmaxf(blo.y - hi[1], lo[1] - bhi.y), 0.0f);
    const float dz = fmaxf(fmaxf(blo.z - hi[2], lo[2] - bhi.z), 0.0f);
    constexpr float reach = kR_Rc_f + 0.01f;
    return dx * dx + dy * dy + dz * dz < reach * reach;
}

// Workgroups for the runs of a batch of n_atoms.  Where the host does not know that it holds large molecules (`sure`) they are fewer: they
// mostly find nothing to do.
__host__ inline dim3 run_grid(int64_t n_atoms, bool sure)
{
    const int64_t most = sure ? 16384 : 4096;
    return dim3(static_cast<unsigned>(n_atoms < most ? (n_atoms + 7) / 8 * 8 : most));
}

// Calls body(molecule, first sorted atom of the run, log2 of a run's atoms) for the workgroup's runs.
// (The units are listed beside the sort, by a workgroup of its own.  Numbers for all atoms of the batch, a run's molecule found by
// bisection of the offsets, have most of the numbers of a mixed batch belong to no run, and the others may lie in one of the eight parts
// below: 100 molecules of 300 atoms behind 3,400 small ones, forward / backward with theirs, 308 / 387 us, so 103 / 134; one of
// 2,700 122 / 159 and 85 / 105; 64 boxes of 1,024-4,096 atoms alone 252 and 245, 312 and 305 the kernels by themselves.)
template <typename T, typename Body>
__device__ __forceinline__ void for_each_run(const SortedAtoms<T>& sorted, Body body)
{
    const int lane = threadIdx.x & 63;
    const int units = uniform(*sorted.n_units);
    const int log_run = log_run_for(static_cast<int64_t>(units) << kLogRunCentres), log_parts = kLogRunCentres - log_run;
    // Workgroup w is on XCD w % 8: an XCD's workgroups take consecutive runs, whose atoms and rows its L2 then holds (64 boxes of
    // 1,024-4,096 atoms, backward 371 -> 358 us).
    const int count = units << log_parts, each = (count + 7) >> 3;
    for (int base = blockIdx.x; base < 8 * each; base += static_cast<int>(gridDim.x) * 64) {
        const int number = base + lane * static_cast<int>(gridDim.x), at = (number & 7) * each + (number >> 3);
        int mol = 0, first = 0;
        bool mine = number < 8 * each && at < count;
        if (mine) {
            const int2 u = sorted.unit[at >> log_parts];
            const int part = (at & ((1 << log_parts) - 1)) << log_run;
            mol = u.x;
            first = (u.y >> kLogRunCentres) + part;
            mine = part <= (u.y & (kRunCentres - 1));
        }
        for (unsigned long long left = wave_ballot(mine); left; left &= left - 1) {
            const int b = lowest_bit(left);
            body(lane_read(mol, b), lane_read(first, b), log_run);
        }
    }
}

// Lists the sorted atoms of a molecule (n atoms at offset off) that may lie in the radial cutoff of one of its sorted atoms
// s0 .. s1 - 1 (at most kRunCentres), in their order: their sorted positions, the atoms themselves and with kVel their vectors (LDS,
// kMaxCandidates each) -> how many, or -1 if there are more than that.  A centre then tests these, in LDS, instead of the chunks
// in its reach: around four neighbours of a dense box about 145 atoms, three steps of 64, where the chunks in reach of one of them
// are nine, from memory.
template <typename T, bool kVel>
__device__ __forceinline__ int list_candidates(const SortedAtoms<T>& sorted, int off, int n, size_t first_chunk, int s0, int s1, int* positions,
                                               typename Fast<T>::vec4* atoms, typename Fast<T>::vec4* vels, int lane)
{
    typedef typename Fast<T>::vec4 vec4;
    constexpr int kAhead = 4;              // chunks whose loads are in flight together
    float lo[3], hi[3];
    {
        const vec4 a = sorted.atom[off + min(s0 + (lane & (kRunCentres - 1)), s1 - 1)];
        const float p[3] = {static_cast<float>(a.x), static_cast<float>(a.y), static_cast<float>(a.z)};
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            lo[k] = hi[k] = p[k];
#pragma unroll
            for (int d = 1; d < kRunCentres; d <<= 1) {
                lo[k] = fminf(lo[k], __shfl_xor(lo[k], d, 64));
                hi[k] = fmaxf(hi[k], __shfl_xor(hi[k], d, 64));
            }
        }
    }
    const float4* const boxes = sorted.box + 2 * first_chunk;
    const int n_chunks = (n + 63) >> 6;
    int count = 0;
    wave_lds_fence();                      // (what was in the arrays has been read)
    for (int ch0 = 0; ch0 < n_chunks; ch0 += 64) {
        const int chunk = min(ch0 + lane, n_chunks - 1);
        unsigned long long near = wave_ballot(ch0 + lane < n_chunks && in_reach(lo, hi, boxes[2 * chunk], boxes[2 * chunk + 1]));
        while (near) {
            int ch[kAhead];
            vec4 at[kAhead];
#pragma unroll
            for (int u = 0; u < kAhead; ++u) {
                ch[u] = -1;
                if (near) {
                    ch[u] = ch0 + lowest_bit(near);
                    near &= near - 1;
                }
            }
#pragma unroll
            for (int u = 0; u < kAhead; ++u) at[u] = sorted.atom[off + min(max(ch[u], 0) * 64 + lane, n - 1)];
#pragma unroll
            for (int u = 0; u < kAhead; ++u) {
                if (ch[u] < 0) break;
                const int j = ch[u] * 64 + lane;
                const float4 p = make_float4(static_cast<float>(at[u].x), static_cast<float>(at[u].y), static_cast<float>(at[u].z), 0.0f);
                const unsigned long long take = wave_ballot(j < n && in_reach(lo, hi, p, p));
                const int to = rank_in(take, count);
                if (((take >> lane) & 1ull) && to < kMaxCandidates) {
                    positions[to] = j;
                    atoms[to] = at[u];
                    if constexpr (kVel) vels[to] = sorted.vel[off + j];
                }
                count += popc64(take);
            }
            if (count > kMaxCandidates) return -1;
        }
    }
    wave_lds_fence();
    return count;
}

// Calls scan(sorted position, does this lane have an atom, atom, vel) for a centre's possible partners, 64 at a time: the run's
// candidates (kPair: two steps' LDS reads together, which has scan() in the code three times instead of once; forward 282 -> 277 us),
// or, without a list (n_candidates < 0), the chunks in the centre's reach.
template <typename T, bool kVel, bool kPair, typename Scan>
__device__ __forceinline__ void scan_partners(const SortedAtoms<T>& sorted, int off, int n, size_t first_chunk, const int* positions,
                                              const typename Fast<T>::vec4* atoms, const typename Fast<T>::vec4* vels, int n_candidates,
                                              const typename Fast<T>::vec4& centre, int lane, Scan scan)
{
    typedef typename Fast<T>::vec4 vec4;
    const vec4 none = Fast<T>::make4(T(0), T(0), T(0), T(0));
    if constexpr (kPair) {
        for (int q0 = 0; q0 < n_candidates; q0 += 128) {
            int j[2];
            vec4 atom[2], vel[2];
#pragma unroll
            for (int u = 0; u < 2; ++u) {
                const int q = min(q0 + 64 * u + lane, n_candidates - 1);
                j[u] = positions[q];
                atom[u] = atoms[q];
                vel[u] = none;
                if constexpr (kVel) vel[u] = vels[q];
            }
#pragma unroll
            for (int u = 0; u < 2; ++u)
                if (q0 + 64 * u < n_candidates) scan(j[u], q0 + 64 * u + lane < n_candidates, atom[u], vel[u]);
        }
        if (n_candidates >= 0) return;
    }
    const float at_centre[3] = {static_cast<float>(centre.x), static_cast<float>(centre.y), static_cast<float>(centre.z)};
    const float4* const boxes = sorted.box + 2 * first_chunk;
    const int n_chunks = (n + 63) >> 6;
    int q0 = 0;                            // the next candidate, or the first of the next 64 chunks
    unsigned long long near = 0;
    for (;;) {
        int j;
        bool have;
        vec4 atom, vel = none;
        if (!kPair && n_candidates >= 0) {
            if (q0 >= n_candidates) return;
            const int q = min(q0 + lane, n_candidates - 1);
            have = q0 + lane < n_candidates;
            j = positions[q];
            atom = atoms[q];
            if constexpr (kVel) vel = vels[q];
            q0 += 64;
        } else {
            while (near == 0) {
                if (q0 >= n_chunks) return;
                const int chunk = min(q0 + lane, n_chunks - 1);
                near = wave_ballot(q0 + lane < n_chunks && in_reach(at_centre, at_centre, boxes[2 * chunk], boxes[2 * chunk + 1]));
                q0 += 64;
            }
            const int at = (q0 - 64 + lowest_bit(near)) * 64 + lane;
            near &= near - 1;
            have = at < n;
            j = min(at, n - 1);
            atom = sorted.atom[off + j];
            if constexpr (kVel) vel = sorted.vel[off + j];
        }
        scan(j, have, atom, vel);
    }
}

// Fills `sorted` for every molecule of more than 256 atoms (stable counting sort by type and cell, one workgroup per
// molecule); with gX the molecule's gradients and the sorted atoms' forces are zeroed as well (the backward kernel then only adds).
template <typename T>
hipError_t launch_large_sort(const T* X, const T* Y, const T* Z, const int32_t* A, const int32_t* MOs,
                             const int32_t* MACs, int32_t n_mols, const int32_t* SIs, const T* VX, const T* VY,
                             const T* VZ, T* gX, T* gY, T* gZ, const int32_t* order, SortedAtoms<T> sorted,
                             hipStream_t stream);

}  // namespace khan
