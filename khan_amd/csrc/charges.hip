// Damped-Coulomb charge energy and its gradients on gfx950.
//
// Reference: gpu_featurizer/ani_charges.cpp:58-71 (energy), 138-160 (dE/dq):
//     E_m = sum_{i<j in m} K q_i q_j (1 - f_C(r_ij, R_Rc)) / r_ij,   K = 0.529176917f, R_Rc = 4.6f
//     dL/dq_i = g_m * sum_{j != i} K q_j (1 - f_C(r_ij)) / r_ij
// f_C(r) = 0.5 cos(pi r / Rc) + 0.5 for r <= Rc, else 0 (so pairs beyond Rc are plain K q q / r).
// The coordinate gradient has no reference counterpart (the reference returns None for x, y, z,
// khan/training/trainer_multi_tower.py:112-119); it is the closed form
//     dL/dx_i = g_m K q_i sum_{j != i} q_j d/dr[(1 - f_C)/r] (x_i - x_j)/r.
//
// One wavefront per molecule.  Up to 64 atoms a step evaluates 64 (i, j) pairs at once -- 4 atoms i x 16
// partners j for molecules of up to 16 atoms, 2 x 32 up to 32, 1 x 64 above -- with the partners' data
// held in the lanes, and the sums over j are in-wave DPP reductions (a lane per atom i walking all j
// would leave four fifths of the lanes idle on a 12-atom molecule).  Molecules of 65 to 256 atoms go to a
// workgroup that tiles the molecule through LDS (charge_tile below).  Above 256 atoms several
// workgroups share a molecule: all pairs, the partners tiled through LDS (charge_large).  Each output
// element is written once, no atomics and no pre-zeroing -- except the energy of a molecule of more than 256 atoms,
// which is the sum of its workgroups' shares.
#include <algorithm>

#include "aev_small_common.h"

namespace khan {

namespace {

// What a pair at squared distance d2 contributes: u = (1 - f_C) / r and du = d/dr[(1 - f_C) / r] / r, both zero for
// coincident atoms.  kDamped = false drops the cutoff function: plain Coulomb pairs (the reference's op is the damped form).
// f_C is evaluated in every lane and selected: a branch would be taken by nearly every wavefront anyway.
// `Constants` are made once per kernel.
template <typename T, bool kDamped> struct PairTerms;
// float: the hardware reciprocal square root with one Newton step and the minimax cutoff polynomials of the AEV kernels
template <bool kDamped> struct PairTerms<float, kDamped> {
    struct Constants {};
    static __device__ __forceinline__ void of(const Constants&, float d2, float& u, float& du)
    {
        const float r = Fast<float>::sqrt_rn(d2);
        const float inv = d2 > 0.0f ? Fast<float>::rcp(r) : 0.0f;
        float fc = 0.0f, dfc = 0.0f;
        if constexpr (kDamped) {
            Fast<float>::cutoff_grad(r, kR_Rc_f, fc, dfc);
            const bool in = r <= kR_Rc_f;
            fc = in ? fc : 0.0f;
            dfc = in ? dfc : 0.0f;
        }
        u = (1.0f - fc) * inv;
        du = (-dfc * inv - u * inv) * inv;
    }
};
// double: no library call, no square root and no angle.  1/r from v_rsq_f64 (5e-8) and one third-order step.  1 - f_C =
// sin^2(pi r / 2 R_c) = d2 q(d2) and 2 d(1 - f_C)/d(d2) = (d/dr) / r are entire functions of d2: polynomials of degree
// nine in d2 (Chebyshev interpolation on [0, R_c^2]), exact to 4e-16 of q and 1e-16.  (Before: a square root, a folded half
// angle, its sine and cosine: 106 vector instructions per pair over the whole kernel by the counters, 92 with the polynomials'
// coefficients in vector registers, where every step of Horner's scheme copies one first, 72 with them in scalar registers.)
template <bool kDamped> struct PairTerms<double, kDamped> {
    struct Constants {
        double q[10], t[10];
        __device__ __forceinline__ Constants()
        {
            constexpr double kQ[10] = {0.11660686212575191, -0.004532386764938009, 7.046765314658188e-05, -5.869294224571146e-07,
                                       3.0417776911092683e-09, -1.0748245519813352e-11, 2.7545314816657834e-14,
                                       -5.3522125411118236e-17, 8.115026416218573e-20, -8.999642674693997e-23};
            constexpr double kT[10] = {0.23321372425150377, -0.018129547059751505, 0.0004228059188787524, -4.695435379265704e-06,
                                       3.0417776808067906e-08, -1.2897893108818512e-10, 3.856331055586389e-13,
                                       -8.562890949169944e-16, 1.4589662776261427e-18, -1.7805957172843363e-21};
            if constexpr (kDamped) {
#pragma unroll
                for (int k = 0; k < 10; ++k) {
                    q[k] = kQ[k];
                    t[k] = kT[k];
                    asm("" : "+s"(q[k]));          // (a value of its own in scalar registers)
                    asm("" : "+s"(t[k]));
                }
            }
        }
    };
    static __device__ __forceinline__ double poly(const double (&c)[10], double x)
    {
        double v = fma(c[9], x, c[8]);
#pragma unroll
        for (int k = 7; k >= 0; --k) v = fma(v, x, c[k]);
        return v;
    }
    static __device__ __forceinline__ void of(const Constants& k, double d2, double& u, double& du)
    {
        const double y = __builtin_amdgcn_rsq(d2);
        const double e = fma(-d2 * y, y, 1.0);
        double inv = fma(y * e, fma(e, 0.375, 0.5), y);
        inv = d2 > 0.0 ? inv : 0.0;
        double s = 1.0, t = 0.0;               // 1 - f_C, and its derivative in r over r
        if constexpr (kDamped) {
            constexpr double kRc2 = static_cast<double>(kR_Rc_f) * static_cast<double>(kR_Rc_f);
            const bool in = d2 <= kRc2;
            const double sq = d2 * poly(k.q, d2), tq = poly(k.t, d2);       // (without meaning outside)
            s = in ? sq : 1.0;
            t = in ? tq : 0.0;
        }
        u = s * inv;
        du = fma(t, inv, -u * (inv * inv));
    }
};

template <typename T>
struct ChargeArgs {
    const T *X, *Y, *Z, *Q;
    const int32_t *MOs, *MACs;
    int32_t n_mols;
    const T* grads;          // gradients only
    T K;
    T *E, *q_grads, *gX, *gY, *gZ;      // with gradients each of E, q_grads and (gX, gY, gZ) may be null
    const int32_t* order;               // the molecules of 65 to 256 atoms by decreasing size in front (charge_begin_kernel), or null
};

// A molecule of up to 64 atoms in one wavefront.
template <typename T, bool kDamped, bool kGrad>
__device__ __forceinline__ void charge_small(const ChargeArgs<T>& a, const typename PairTerms<T, kDamped>::Constants& constants, int mol, int n)
{
    const int lane = threadIdx.x & 63;
    const int off = a.MOs[mol];
    const int logW = n <= 16 ? 4 : n <= 32 ? 5 : 6;
    const int W = 1 << logW, G = 64 >> logW;
    const int grp = lane >> logW, jl = lane & (W - 1);
    const bool jok = jl < n;
    const T xj = jok ? a.X[off + jl] : T(0), yj = jok ? a.Y[off + jl] : T(0), zj = jok ? a.Z[off + jl] : T(0),
            qj = jok ? a.Q[off + jl] : T(0);
    T gK = T(0);
    if constexpr (kGrad) gK = a.grads[mol] * a.K;
    T acc = T(0);                // the energy / K; with gradients twice that: q_i sum_j q_j u_ij over the atoms
    for (int i0 = 0; i0 < n; i0 += G) {
        const int i = i0 + grp;                      // lane i of the first group holds atom i
        const T xi = __shfl(xj, i & 63, 64), yi = __shfl(yj, i & 63, 64), zi = __shfl(zj, i & 63, 64), qi = __shfl(qj, i & 63, 64);
        const bool valid = (i < n) && jok && (kGrad ? jl != i : jl > i);
        const T dx = xi - xj, dy = yi - yj, dz = zi - zj;
        T u, du;
        PairTerms<T, kDamped>::of(constants, dx * dx + dy * dy + dz * dz, u, du);
        if constexpr (!kGrad) {
            acc += valid ? qi * qj * u : T(0);
        } else {
            const T w = valid ? qj * du : T(0);
            // sums over the W partners of the group end up in its last lane
            const T dq = group_sum_to_last_lane(valid ? qj * u : T(0), logW);
            const T fx = group_sum_to_last_lane(w * dx, logW);
            const T fy = group_sum_to_last_lane(w * dy, logW);
            const T fz = group_sum_to_last_lane(w * dz, logW);
            if (jl == W - 1 && i < n) {
                acc = fma(qi, dq, acc);
                if (a.q_grads) a.q_grads[off + i] = gK * dq;
                if (a.gX) {
                    a.gX[off + i] = gK * qi * fx;
                    a.gY[off + i] = gK * qi * fy;
                    a.gZ[off + i] = gK * qi * fz;
                }
            }
        }
    }
    if (a.E) {
        acc = wave_sum(acc);
        if (lane == 0) a.E[mol] = (kGrad ? T(0.5) : T(1)) * a.K * acc;
    }
}

// Molecules of 65 to 256 atoms: one workgroup of four wavefronts per molecule, the molecule (x, y, z, q) in LDS.  A
// wavefront takes a block of 64 atoms, one atom i per lane; in round d a lane pairs its atom with atom j = (i + d) mod n,
// read from the tile: after (n-1)/2 rounds (plus half a round when n is even) of every block each unordered pair has been
// evaluated exactly once -- half the pair evaluations of a walk over all j != i.  The blocks' rounds are dealt to the four
// wavefronts in equal shares (a block per wavefront left a quarter of them without work on average: dense boxes of 64-256
// atoms).  In a round the partners j of a wavefront's atoms are distinct, so what a pair contributes to its partner
// (dE/dq_j and the force on j) is added to the partner's slot in LDS by plain read-add-write, without atomics, while the
// atom's own side stays in registers until the block's share ends.  Every wavefront adds into a copy of its own of the
// slots, so the four never wait for each other inside the rounds (a barrier per round would be the alternative); the
// copies are summed at the end.  Every output element is written once.
template <typename T, bool kGrad> struct ChargeTile;
// (pairs of values in arrays of their own: 16-byte accesses 32 bytes apart would meet in half of the banks)
template <typename T> struct __align__(16) ChargeTile<T, false> {
    typename Fast<T>::vec2 in[2][kMediumMaxAtoms];     // x, y and z, q
    T wpart[4];
};
// (in double these are 40,960 bytes, a quarter of a compute unit's LDS to the byte: the wavefronts' partial energies
// go into the tile's first entry once the rounds are over, not into four words more that would cost the fourth workgroup)
template <typename T> struct __align__(16) ChargeTile<T, true> {
    typename Fast<T>::vec2 in[2][kMediumMaxAtoms];     // x, y and z, q
    typename Fast<T>::vec2 acc[4][2][kMediumMaxAtoms]; // per wavefront: force x, y and force z, dE/dq
};

template <typename T, bool kDamped, bool kGrad>
__device__ __forceinline__ void charge_tile(const ChargeArgs<T>& a, const typename PairTerms<T, kDamped>::Constants& constants,
                                            ChargeTile<T, kGrad>& S, int mol, int n)
{
    typedef typename Fast<T>::vec2 vec2;
    static_assert(kMediumMaxAtoms == 256, "one atom per thread of a 256-thread workgroup");
    const int tid = threadIdx.x, lane = tid & 63, wave = uniform(tid >> 6);
    const int off = uniform(a.MOs[mol]);
    const bool have = tid < n;
    if (have) {
        S.in[0][tid] = Fast<T>::make2(a.X[off + tid], a.Y[off + tid]);
        S.in[1][tid] = Fast<T>::make2(a.Z[off + tid], a.Q[off + tid]);
    }
    if constexpr (kGrad) {
#pragma unroll
        for (int w = 0; w < 4; ++w) S.acc[w][0][tid] = S.acc[w][1][tid] = Fast<T>::make2(T(0), T(0));
    }
    __syncthreads();
    // the rounds of every block of 64 atoms, laid end to end and cut into four equal shares
    const int half = (n - 1) >> 1, rounds = half + ((n & 1) == 0 ? 1 : 0), blocks = (n + 63) >> 6;
    const int units = blocks * rounds;
    int unit = wave * units >> 2;
    const int last = (wave + 1) * units >> 2;
    T e_acc = T(0);
    while (unit < last) {
        const int block = unit / rounds, d0 = unit - block * rounds;             // rounds d0 + 1 .. d1
        const int d1 = min(rounds, d0 + (last - unit));
        unit += d1 - d0;
        const int i = block * 64 + lane;
        // a lane without an atom takes part with charge zero: everything it adds is zero, and its partners are, like
        // everyone's, distinct from those of the other lanes of its wavefront (n > 64)
        const vec2 own_xy = S.in[0][min(i, n - 1)], own_zq = S.in[1][min(i, n - 1)];
        const T q_own = i < n ? own_zq.y : T(0);
        int j = i + d0;                              // (i + d) mod n: i < n + 64, d0 < n / 2
        j -= j >= n ? n : 0;
        j -= j >= n ? n : 0;
        T fx = T(0), fy = T(0), fz = T(0), dq = T(0);
        // what a pair adds to either side, and where its partner's slot is
        struct Terms {
            int j;
            T q, u, wx, wy, wz;
        };
        auto terms = [&](T q_i, bool act) -> Terms {
            j = j + 1 == n ? 0 : j + 1;
            const vec2 xy = S.in[0][j], zq = S.in[1][j];
            const T dx = own_xy.x - xy.x, dy = own_xy.y - xy.y, dz = own_zq.x - zq.x;
            T u, du;
            PairTerms<T, kDamped>::of(constants, dx * dx + dy * dy + dz * dz, u, du);
            const T qq = q_i * zq.y;
            if constexpr (!kGrad) {
                e_acc = fma(qq, u, e_acc);
                return {};
            } else {
                dq = fma(act ? zq.y : T(0), u, dq);
                const T wq = qq * du;                    // q_i q_j d/dr[(1-f_C)/r] / r
                const Terms p = {j, q_i, u, wq * dx, wq * dy, wq * dz};
                fx += p.wx;
                fy += p.wy;
                fz += p.wz;
                return p;
            }
        };
        auto give = [&](const Terms& p) {
            if constexpr (kGrad) {
                vec2 pa = S.acc[wave][0][p.j], pb = S.acc[wave][1][p.j];     // distinct j across the lanes of this wavefront
                pa.x -= p.wx;
                pa.y -= p.wy;
                pb.x -= p.wz;
                pb.y = fma(p.q, p.u, pb.y);
                S.acc[wave][0][p.j] = pa;
                S.acc[wave][1][p.j] = pb;
                wave_lds_fence();                        // the next round may touch slots written here
            }
        };
        // two rounds' terms side by side (their chains of dependent multiply-adds fill each other's waits), then their sums
        const int full = min(d1, half);
        int d = d0;
        for (; d + 1 < full; d += 2) {
            const Terms p0 = terms(q_own, true), p1 = terms(q_own, true);
            give(p0);
            give(p1);
        }
        if (d < full) give(terms(q_own, true));
        if (d1 > half) give(terms(i < (n >> 1) ? q_own : T(0), i < (n >> 1)));      // the half round of an even n: the lower half only
        if constexpr (kGrad) {
            if (i < n) {                                 // the atoms' own side joins this wavefront's copy
                vec2 pa = S.acc[wave][0][i], pb = S.acc[wave][1][i];
                pa.x += fx;
                pa.y += fy;
                pb.x += fz;
                pb.y += dq;
                S.acc[wave][0][i] = pa;
                S.acc[wave][1][i] = pb;
            }
            wave_lds_fence();
        }
    }
    T p[4] = {T(0), T(0), T(0), T(0)};
    T* wpart;
    if constexpr (kGrad) {
        __syncthreads();                             // every wavefront's partner sides are complete, the tile is free
        if (have) {
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const vec2 p0 = S.acc[0][h][tid], p1 = S.acc[1][h][tid], p2 = S.acc[2][h][tid], p3 = S.acc[3][h][tid];
                p[2 * h] = (p0.x + p1.x) + (p2.x + p3.x);
                p[2 * h + 1] = (p0.y + p1.y) + (p2.y + p3.y);
            }
        }
        // the energy: half of q_i sum_j q_j u_ij over the atoms
        e_acc = have ? T(0.5) * S.in[1][tid].y * p[3] : T(0);
        __syncthreads();                             // (the first entry is overwritten below)
        wpart = reinterpret_cast<T*>(&S.in[0][0]);
    } else {
        wpart = S.wpart;
    }
    if (a.E) {
        e_acc = wave_sum(e_acc);
        if (lane == 0) wpart[wave] = e_acc;
        __syncthreads();
        if (tid == 0) a.E[mol] = a.K * ((wpart[0] + wpart[1]) + (wpart[2] + wpart[3]));
    }
    if constexpr (kGrad) {
        if (have) {
            const T gK = a.grads[mol] * a.K;
            if (a.q_grads) a.q_grads[off + tid] = gK * p[3];
            if (a.gX) {
                // the force sums carry q_i already (wq = q_i q_j ...)
                a.gX[off + tid] = gK * p[0];
                a.gY[off + tid] = gK * p[1];
                a.gZ[off + tid] = gK * p[2];
            }
        }
    }
}

// Molecules of more than 256 atoms: all pairs, the partners tiled through LDS 256 at a time.  A thread owns one atom i
// of a block of 256 and sums over every partner j (each pair is evaluated from both ends: no exchange between threads, and
// every per-atom output is written once, by its owner); the `parts` workgroups of a column share a molecule's
// blocks.  The energy is half the sum over atoms of q_i times the atom's sum, added to E[mol] (zeroed before the launch)
// by one floating-point atomic per workgroup and block: its last bits depend on the order of those additions.
template <typename T, bool kDamped, bool kGrad>
__device__ __forceinline__ void charge_large(const ChargeArgs<T>& a, const typename PairTerms<T, kDamped>::Constants& constants,
                                             typename Fast<T>::vec4* tile, T* wpart, int column, int columns, int part, int parts)
{
    typedef typename Fast<T>::vec4 vec4;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    for (int64_t base = column; base < a.n_mols; base += static_cast<int64_t>(columns) * 256) {
        // the next 256 molecules of this column, one per thread: is there a large one?
        const int64_t mine = base + static_cast<int64_t>(tid) * columns;
        const bool large = mine < a.n_mols && a.MACs[mine] > kMediumMaxAtoms;
        const bool some = wave_ballot(large) != 0ull;
        if (lane == 0) wpart[wave] = some ? T(1) : T(0);
        __syncthreads();
        const bool any = wpart[0] + wpart[1] + wpart[2] + wpart[3] > T(0);
        __syncthreads();
        if (!any) continue;
        for (int k = 0; k < 256; ++k) {
            const int64_t m = base + static_cast<int64_t>(k) * columns;
            if (m >= a.n_mols) break;
            const int mol = static_cast<int>(m);
            const int n = uniform(a.MACs[mol]);
            if (n <= kMediumMaxAtoms) continue;
            const int off = uniform(a.MOs[mol]);
            for (int i0 = part * 256; i0 < n; i0 += parts * 256) {
                const int i = i0 + tid;
                const bool have = i < n;
                const T xi = have ? a.X[off + i] : T(0), yi = have ? a.Y[off + i] : T(0), zi = have ? a.Z[off + i] : T(0),
                        qi = have ? a.Q[off + i] : T(0);
                T su = T(0), fx = T(0), fy = T(0), fz = T(0);      // sums over j of q_j u and of q_j du (x_i - x_j)
                for (int j0 = 0; j0 < n; j0 += 256) {
                    __syncthreads();                               // the previous tile has been used
                    const int j = j0 + tid;
                    // (places beyond the molecule: charge zero)
                    tile[tid] = j < n ? Fast<T>::make4(a.X[off + j], a.Y[off + j], a.Z[off + j], a.Q[off + j])
                                      : Fast<T>::make4(T(0), T(0), T(0), T(0));
                    __syncthreads();
                    const int cnt = min(256, n - j0);
#pragma unroll sizeof(T) == 4 ? 4 : 2
                    for (int t = 0; t < cnt; ++t) {
                        const vec4 aj = tile[t];                   // the same address in every lane
                        const T dx = xi - aj.x, dy = yi - aj.y, dz = zi - aj.z;
                        T u, du;
                        PairTerms<T, kDamped>::of(constants, dx * dx + dy * dy + dz * dz, u, du);      // zero for the atom itself (r = 0)
                        su = fma(aj.w, u, su);
                        if constexpr (kGrad) {
                            const T w = aj.w * du;
                            fx = fma(w, dx, fx);
                            fy = fma(w, dy, fy);
                            fz = fma(w, dz, fz);
                        }
                    }
                }
                if (a.E) {                                         // (the same for every thread)
                    const T share = wave_sum(have ? qi * su : T(0));
                    __syncthreads();                               // wpart is free
                    if (lane == 0) wpart[wave] = share;
                    __syncthreads();
                    if (tid == 0) atomicAdd(&a.E[mol], T(0.5) * a.K * (wpart[0] + wpart[1] + wpart[2] + wpart[3]));
                }
                if (kGrad && have) {
                    const T gK = a.grads[mol] * a.K;
                    if (a.q_grads) a.q_grads[off + i] = gK * su;
                    if (a.gX) {
                        a.gX[off + i] = gK * qi * fx;
                        a.gY[off + i] = gK * qi * fy;
                        a.gZ[off + i] = gK * qi * fz;
                    }
                }
            }
        }
    }
}

// One launch for every size.  Workgroups 0 .. large - 1 (columns x parts of them) share the molecules of more than 256 atoms.
// Behind them come, with per = 1, a workgroup for every four molecules, whose wavefronts take those of up to 64 atoms, and one
// for every molecule, which takes those of 65 to 256 (in the first ones' places a wavefront with 64 atoms had the compute unit
// that came upon it last work for 35 us after all others).  With per = 4 a workgroup does both for its four molecules.
// (Three launches, one per size, cost 10 us where two of them found nothing to do.)  Four workgroups per compute unit, which
// LDS allows.  4,096 boxes of 64 to 256 atoms in double, energy and both gradients with the launch before: 217 -> 148 us
// (coefficients in scalar registers, size order, first places for the small molecules, two rounds side by side; 170 in batch
// order).  Vector issue binds: by the counters 72 instructions a pair keep it 76 % busy, with an LDS instruction executing on
// a compute unit 82 % of the time (7.7 a pair).
template <typename T, bool kDamped, bool kGrad>
__global__ __launch_bounds__(256, 4) void charge_kernel(ChargeArgs<T> a, int columns, int parts, int per)
{
    __shared__ ChargeTile<T, kGrad> S;
    const typename PairTerms<T, kDamped>::Constants constants;
    const int large = columns * parts;
    const int b = static_cast<int>(blockIdx.x) - large;
    if (b < 0) {
        const int g = static_cast<int>(blockIdx.x);
        T* wpart;
        if constexpr (kGrad) wpart = reinterpret_cast<T*>(S.acc[0]);
        else wpart = S.wpart;
        charge_large<T, kDamped, kGrad>(a, constants, reinterpret_cast<typename Fast<T>::vec4*>(&S.in[0][0]), wpart, g % columns, columns, g / columns, parts);
        return;
    }
    const int wave = uniform(threadIdx.x >> 6);
    const int fours = (a.n_mols - 1) / 4 + 1;
    if (b < fours) {
        const int64_t mol = 4 * static_cast<int64_t>(b) + wave;
        if (mol < a.n_mols) {
            const int n = uniform(a.MACs[mol]);
            if (n <= kSmallMaxAtoms) charge_small<T, kDamped, kGrad>(a, constants, static_cast<int>(mol), n);
        }
        if (per == 1) return;
    }
    const int64_t first = per == 1 ? b - fours : 4 * static_cast<int64_t>(b);
    for (int64_t at = first; at < min(first + per, static_cast<int64_t>(a.n_mols)); ++at) {
        const int mol = a.order ? a.order[at] : static_cast<int>(at);
        const int n = uniform(a.MACs[mol]);
        if (n > kSmallMaxAtoms && n <= kMediumMaxAtoms) {
            charge_tile<T, kDamped, kGrad>(a, constants, S, mol, n);
            __syncthreads();         // the next molecule reuses the tile
        }
    }
}

// Before the launch: zeros in the outputs (atoms outside every molecule keep them, and the energies of molecules of more than
// 256 atoms are added up), and by the first workgroup the molecules of 65 to 256 atoms by
// decreasing size, the others behind them: a counting sort, in no particular order inside a size (every molecule's results
// are its own).  A launch lasts only a few molecules' time and in batch order ended with a third of the wavefronts' places empty.
// From two workgroups a compute unit on in float32 and from one on in float64, though four find a place: those that share a unit
// share its arithmetic, and in decreasing size the units' shares come out alike.  Boxes of 64 to 256 atoms, fill and pass in
// batch order -> sorting launch and pass, us: float32 257 molecules 24.9 -> 27.4, 400 31.7 -> 34.1, 600 36.4 -> 34.7, 1,000
// 46 -> 37, 4,096 103 -> 88; float64 257 35.5 -> 35.3, 400 45.7 -> 43.4, 600 56 -> 45, 1,000 67 -> 54, 4,096 170 -> 148.
template <typename T> constexpr int kOrderFrom = (sizeof(T) == 4 ? 2 : 1) * kCUs;
constexpr int kOrderMost = 16384;
template <typename T>
__global__ __launch_bounds__(1024) void charge_begin_kernel(const int32_t* __restrict__ MACs, int n_mols, int32_t* __restrict__ order,
                                                            T* __restrict__ outputs, int64_t n_outputs)
{
    const int tid = threadIdx.x;
    if (blockIdx.x > 0) {
        const int64_t step = static_cast<int64_t>(gridDim.x - 1) * 1024;
        for (int64_t i = static_cast<int64_t>(blockIdx.x - 1) * 1024 + tid; i < n_outputs; i += step) outputs[i] = T(0);
        return;
    }
    constexpr int kBins = kMediumMaxAtoms + 1, kEach = kOrderMost / 1024;
    __shared__ int bin[2][512];
    if (tid < 512) bin[0][tid] = 0;
    __syncthreads();
    int key[kEach];
#pragma unroll
    for (int k = 0; k < kEach; ++k) {
        const int mol = k * 1024 + tid;
        const int n = mol < n_mols ? MACs[mol] : 0;
        key[k] = mol >= n_mols ? -1 : n > kSmallMaxAtoms && n <= kMediumMaxAtoms ? kMediumMaxAtoms - n : kBins - 1;
    }
#pragma unroll
    for (int k = 0; k < kEach; ++k)
        if (key[k] >= 0) atomicAdd(&bin[0][key[k]], 1);
    __syncthreads();
    int from = 0;
    for (int d = 1; d < kBins; d <<= 1) {                 // inclusive sums
        if (tid < 512) bin[from ^ 1][tid] = bin[from][tid] + (tid >= d ? bin[from][tid - d] : 0);
        from ^= 1;
        __syncthreads();
    }
    if (tid < 512) bin[from ^ 1][tid] = tid > 0 ? bin[from][tid - 1] : 0;
    __syncthreads();
#pragma unroll
    for (int k = 0; k < kEach; ++k)
        if (key[k] >= 0) order[atomicAdd(&bin[from ^ 1][key[k]], 1)] = k * 1024 + tid;
}

// a workgroup per four molecules where they are small, per molecule where a workgroup has to work on each: 4,096 boxes on a
// quarter of the workgroups end when the compute unit with the largest boxes does
int charge_mols_per_workgroup(int32_t n_mols, int64_t n_atoms) { return n_atoms > 32 * static_cast<int64_t>(n_mols) ? 1 : 4; }

template <typename T, bool kGrad>
hipError_t launch_charges(const ChargeArgs<T>& a, int64_t n_atoms, bool damped, bool zeroed, hipStream_t stream)
{
    if (a.n_mols <= 0) return hipSuccess;
    int columns = 0, parts = 1;
    if (n_atoms > kMediumMaxAtoms) {          // there may be large ones: at most so many, of at most so many blocks
        columns = static_cast<int>(std::min<int64_t>({a.n_mols, 256, n_atoms / (kMediumMaxAtoms + 1)}));
        parts = static_cast<int>(std::min<int64_t>({columns >= 256 ? 4 : 1024 / columns, 256, (n_atoms + 255) / 256}));
        if (a.E && !zeroed) {
            const hipError_t e = launch_zero<T>(a.E, a.n_mols, stream);
            if (e != hipSuccess) return e;
        }
    }
    const int per = charge_mols_per_workgroup(a.n_mols, n_atoms);
    const int64_t blocks = (static_cast<int64_t>(a.n_mols) + 3) / 4 + (per == 1 ? a.n_mols : 0) + static_cast<int64_t>(columns) * parts;
    const auto kernel = damped ? charge_kernel<T, true, kGrad> : charge_kernel<T, false, kGrad>;
    kernel<<<dim3(static_cast<unsigned>(blocks)), dim3(256), 0, stream>>>(a, std::max(columns, 1), columns ? parts : 0, per);
    return hipGetLastError();
}

}  // namespace

template <typename T>
hipError_t launch_charge_energy(const T* X, const T* Y, const T* Z, const T* Q, const int32_t* MOs, const int32_t* MACs, int32_t n_mols,
                                int64_t n_atoms, bool damped, T K, T* E, hipStream_t stream)
{
    return launch_charges<T, false>(ChargeArgs<T>{X, Y, Z, Q, MOs, MACs, n_mols, nullptr, K, E, nullptr, nullptr, nullptr, nullptr, nullptr}, n_atoms, damped,
                                    false, stream);
}

template <typename T>
hipError_t launch_charge_grad(const T* X, const T* Y, const T* Z, const T* Q, const int32_t* MOs, const int32_t* MACs, int32_t n_mols,
                              int64_t n_atoms, const T* grads, bool damped, T K, T* q_grads, T* gX, T* gY, T* gZ, T* E, bool zeroed,
                              const int32_t* order, hipStream_t stream)
{
    return launch_charges<T, true>(ChargeArgs<T>{X, Y, Z, Q, MOs, MACs, n_mols, grads, K, E, q_grads, gX, gY, gZ, order}, n_atoms, damped, zeroed, stream);
}

// Zeros in `outputs`; `order` (n_mols ints): set to null where the size order does not pay.
template <typename T>
hipError_t launch_charge_begin(const int32_t* MACs, int32_t n_mols, int64_t n_atoms, int32_t*& order, T* outputs, int64_t n_outputs, hipStream_t stream)
{
    if (n_mols <= kOrderFrom<T> || n_mols > kOrderMost || charge_mols_per_workgroup(n_mols, n_atoms) != 1) order = nullptr;
    if (!order) return n_outputs > 0 ? launch_zero<T>(outputs, n_outputs, stream) : hipSuccess;
    const int64_t zeroing = std::min<int64_t>((n_outputs + 8191) / 8192, 512);
    charge_begin_kernel<T><<<dim3(static_cast<unsigned>(zeroing + 1)), dim3(1024), 0, stream>>>(MACs, n_mols, order, outputs, n_outputs);
    return hipGetLastError();
}
template hipError_t launch_charge_begin<float>(const int32_t*, int32_t, int64_t, int32_t*&, float*, int64_t, hipStream_t);
template hipError_t launch_charge_begin<double>(const int32_t*, int32_t, int64_t, int32_t*&, double*, int64_t, hipStream_t);

template hipError_t launch_charge_energy<float>(const float*, const float*, const float*, const float*, const int32_t*, const int32_t*, int32_t, int64_t, bool, float, float*, hipStream_t);
template hipError_t launch_charge_energy<double>(const double*, const double*, const double*, const double*, const int32_t*, const int32_t*, int32_t, int64_t, bool, double, double*, hipStream_t);
template hipError_t launch_charge_grad<float>(const float*, const float*, const float*, const float*, const int32_t*, const int32_t*, int32_t, int64_t, const float*, bool, float, float*, float*, float*, float*, float*, bool, const int32_t*, hipStream_t);
template hipError_t launch_charge_grad<double>(const double*, const double*, const double*, const double*, const int32_t*, const int32_t*, int32_t, int64_t, const double*, bool, double, double*, double*, double*, double*, double*, bool, const int32_t*, hipStream_t);

}  // namespace khan
