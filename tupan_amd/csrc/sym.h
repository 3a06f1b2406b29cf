// Symmetric all-pairs engine: a set against itself, each unordered pair once.
//
// A pair's separation, 1/R and the terms built from them are the same for
// both particles up to a sign, so a call whose i-set is its j-set evaluates
// them once per unordered pair and adds the result to both particles' sums:
// an FP64 AccJerk pair takes 39 instructions and one v_rsq_f64 for its two
// interactions where the tile engine (engine.h) takes 2 x 32 and two.  Both
// engines are bound by vector-ALU issue, so that ratio is the gain.
//
// Decomposition.  The set is cut into nb blocks of BI = 256 W particles, and
// block I meets the blocks I + d (mod nb), d = 1 .. nb/2 (for even nb the
// last distance belongs to the first nb/2 blocks), each once, and itself
// (d = 0, where all ordered pairs run and only the i sums are kept).  A
// workgroup of four waves holds block I, W particles per lane in registers,
// and walks a contiguous share ("chunk") of the row's j tiles.
//
// Inside a tile every wave takes 64 j-particles at a time: in step s lane l
// meets particle l - s (mod 64) of the 64, read from LDS (field arrays, each
// value stored twice so the rotating index needs no wrap and the reads are
// conflict free), applies it to its W particles, and adds the pairs' terms
// to the j-particle's running sums, which move one lane per step (DPP
// wave_ror:1) and so visit every lane with their particle.  A rotation costs
// one FP64 issue slot per 32-bit register, shared by the lane's W pairs
// (W = 4: 3 of 42 slots in FP64 AccJerk).  After 64 steps the four waves'
// j sums are added in wave order through LDS and written to the slot (d, j)
// of a partial-sum array, the i sums go to (chunk, i), and sym_reduce_kernel
// adds each particle's slots in a fixed order: the same result on every run.
//
// FP32 arithmetic (split-FP32 and the float build) moves its i sums into
// FP64 every 64 pairs and its j sums every 64 / W steps (64 pairs), as the
// tile engine does for the split ops.
#pragma once

#include "ops.h"

namespace tupan {

constexpr int kSymBlock = 256;
constexpr int kSymWaves = kSymBlock / kWave;

// -- interactions -------------------------------------------------------------
// A policy S over the tile engine's op Base: T (pair arithmetic), kF fields
// per particle in the order `load` fills them, kK sums, interact(I, J, ai,
// aj, e2u, eta) adding the pair to both particles' sums.  kU: the pair
// softening is e2u; kM: pairs at zero separation are masked.

// A padding particle is a copy of the set's last one without mass, softened
// enough that no pair with it overflows (infinity times its zero mass would
// be NaN in the real particle's sum).  A uniform tile has the set's softening
// for it too, where that is enough (pad_ok; an unmasked tile runs only where
// every pair is finite); else the tile takes the general loop.  kPadSafe: a
// policy whose padding needs none of this (1/R of a potential does not
// overflow; a padding particle without position has no time step).
template <int kM0, int kE2, class T, int F>
__device__ __forceinline__ void sym_pad(T (&f)[F])
{
    f[kM0] = T(0);
    f[kE2] = T(1);
}

template <class P>
struct SymPhi {
    using Base = OpPhi<P>;
    using T = typename P::T;
    static constexpr int kF = 5, kK = 1, kE2 = 4, kM0 = 0;
    static constexpr bool kMax1 = false, kPadSafe = true;
    __device__ static void load(const typename Base::Args& a, const typename Base::Frame&, int i,
                                T (&f)[kF])
    {
#pragma unroll
        for (int k = 0; k < kF; ++k) f[k] = a.ip[k][i];
    }
    __device__ static void pad(T (&f)[kF]) { f[0] = T(0); }
    template <bool kU, bool kM>
    __device__ static __forceinline__ void interact(const T (&I)[kF], const T (&J)[kF],
                                                    T (&ai)[kK], T (&aj)[kK], T e2u, T)
    {
        const T dx = I[1] - J[1], dy = I[2] - J[2], dz = I[3] - J[3];
        const T e2 = kU ? e2u : I[4] + J[4];
        const T r2 = dot3<P>(dx, dy, dz, dx, dy, dz);
        T q1, q2;
        P::q12(r2, e2, r2 > T(0), q1, q2);
        ai[0] = nmad<P>(J[0], q1, ai[0]);
        aj[0] = nmad<P>(I[0], q1, aj[0]);
    }
    __device__ static constexpr double scale() { return 1.0; }
};

template <class P>
struct SymAcc {
    using Base = OpAcc<P>;
    using T = typename P::T;
    static constexpr int kF = 5, kK = 3, kE2 = 4, kM0 = 0;
    static constexpr bool kMax1 = false, kPadSafe = false;
    __device__ static void load(const typename Base::Args& a, const typename Base::Frame&, int i,
                                T (&f)[kF])
    {
#pragma unroll
        for (int k = 0; k < kF; ++k) f[k] = a.ip[k][i];
    }
    __device__ static void pad(T (&f)[kF]) { sym_pad<kM0, kE2>(f); }
    template <bool kU, bool kM>
    __device__ static __forceinline__ void interact(const T (&I)[kF], const T (&J)[kF],
                                                    T (&ai)[kK], T (&aj)[kK], T e2u, T)
    {
        const T dx = I[1] - J[1], dy = I[2] - J[2], dz = I[3] - J[3];
        const T e2 = kU ? e2u : I[4] + J[4];
        const T r2 = dot3<P>(dx, dy, dz, dx, dy, dz);
        T q1, q2;
        P::q12(r2, e2, kM ? r2 > T(0) : true, q1, q2);
        const T q3 = q2 * q1;
        const T wj = q3 * J[0], wi = q3 * I[0];
        ai[0] = nmad<P>(wj, dx, ai[0]);
        ai[1] = nmad<P>(wj, dy, ai[1]);
        ai[2] = nmad<P>(wj, dz, ai[2]);
        aj[0] = mad<P>(wi, dx, aj[0]);
        aj[1] = mad<P>(wi, dy, aj[1]);
        aj[2] = mad<P>(wi, dz, aj[2]);
    }
    __device__ static constexpr double scale() { return 1.0; }
};

template <class P>
struct SymAccJerk {
    using Base = OpAccJerk<P>;
    using T = typename P::T;
    static constexpr int kF = 8, kK = 6, kE2 = 4, kM0 = 0;
    static constexpr bool kMax1 = false, kPadSafe = false;
    __device__ static void load(const typename Base::Args& a, const typename Base::Frame&, int i,
                                T (&f)[kF])
    {
#pragma unroll
        for (int k = 0; k < kF; ++k) f[k] = a.ip[k][i];
    }
    __device__ static void pad(T (&f)[kF]) { sym_pad<kM0, kE2>(f); }
    template <bool kU, bool kM>
    __device__ static __forceinline__ void interact(const T (&I)[kF], const T (&J)[kF],
                                                    T (&ai)[kK], T (&aj)[kK], T e2u, T)
    {
        const T dx = I[1] - J[1], dy = I[2] - J[2], dz = I[3] - J[3];
        const T e2 = kU ? e2u : I[4] + J[4];
        T ux = I[5] - J[5], uy = I[6] - J[6], uz = I[7] - J[7];
        const T r2 = dot3<P>(dx, dy, dz, dx, dy, dz);
        const T rv = dot3<P>(dx, dy, dz, ux, uy, uz);
        T q1, q2;
        P::q12(r2, e2, kM ? r2 > T(0) : true, q1, q2);
        const T q3 = q2 * q1;
        const T alpha = T(3) * rv * q2;
        ux = nmad<P>(alpha, dx, ux);
        uy = nmad<P>(alpha, dy, uy);
        uz = nmad<P>(alpha, dz, uz);
        const T wj = q3 * J[0], wi = q3 * I[0];
        ai[0] = nmad<P>(wj, dx, ai[0]);
        ai[1] = nmad<P>(wj, dy, ai[1]);
        ai[2] = nmad<P>(wj, dz, ai[2]);
        ai[3] = nmad<P>(wj, ux, ai[3]);
        ai[4] = nmad<P>(wj, uy, ai[4]);
        ai[5] = nmad<P>(wj, uz, ai[5]);
        aj[0] = mad<P>(wi, dx, aj[0]);
        aj[1] = mad<P>(wi, dy, aj[1]);
        aj[2] = mad<P>(wi, dz, aj[2]);
        aj[3] = mad<P>(wi, ux, aj[3]);
        aj[4] = mad<P>(wi, uy, aj[4]);
        aj[5] = mad<P>(wi, uz, aj[5]);
    }
    __device__ static constexpr double scale() { return 1.0; }
};

template <class P>
struct SymSnapCrackle {
    using Base = OpSnapCrackle<P>;
    using T = typename P::T;
    static constexpr int kF = 14, kK = 6, kE2 = 4, kM0 = 0;
    static constexpr bool kMax1 = false, kPadSafe = false;
    __device__ static void load(const typename Base::Args& a, const typename Base::Frame&, int i,
                                T (&f)[kF])
    {
#pragma unroll
        for (int k = 0; k < kF; ++k) f[k] = a.ip[k][i];
    }
    __device__ static void pad(T (&f)[kF]) { sym_pad<kM0, kE2>(f); }
    template <bool kU, bool kM>
    __device__ static __forceinline__ void interact(const T (&I)[kF], const T (&J)[kF],
                                                    T (&ai)[kK], T (&aj)[kK], T e2u, T)
    {
        // both particles' terms are the same six values times 1/R^3 and the
        // other's mass
        typename Base::IReg r;
        typename Base::Slot s;
        typename Base::Acc c;
#pragma unroll
        for (int k = 1; k < kF; ++k) {
            r.v[k - 1] = I[k];
            s.v[k] = J[k];
        }
        T q3;
        Base::pair_terms(r, s, c.s, q3);
        const T wj = q3 * J[0], wi = q3 * I[0];
#pragma unroll
        for (int k = 0; k < kK; ++k) {
            ai[k] = nmad<P>(wj, c.s[k], ai[k]);
            aj[k] = mad<P>(wi, c.s[k], aj[k]);
        }
    }
    __device__ static constexpr double scale() { return 1.0; }
};

// The pair frequency w^2 is the same for both particles.  A padding particle
// has no position (NaN), so its pairs fail the r^2 > 0 test and add zero.
template <class P>
struct SymTstep {
    using Base = OpTstep<P>;
    using T = typename P::T;
    static constexpr int kF = 8, kK = 2, kE2 = 4, kM0 = 0;
    static constexpr bool kMax1 = true, kPadSafe = true;
    __device__ static void load(const typename Base::Args& a, const typename Base::Frame&, int i,
                                T (&f)[kF])
    {
#pragma unroll
        for (int k = 0; k < kF; ++k) f[k] = a.ip[k][i];
    }
    __device__ static void pad(T (&f)[kF]) { f[1] = T(__builtin_nanf("")); }
    template <bool kU, bool kM>
    __device__ static __forceinline__ void interact(const T (&I)[kF], const T (&J)[kF],
                                                    T (&ai)[kK], T (&aj)[kK], T e2u, T eta)
    {
        typename Base::IReg r;
        typename Base::Slot s;
        r.m = I[0]; r.x = I[1]; r.y = I[2]; r.z = I[3]; r.e2 = I[4];
        r.vx = I[5]; r.vy = I[6]; r.vz = I[7]; r.eta = eta;
#pragma unroll
        for (int k = 0; k < kF; ++k) s.v[k] = J[k];
        const T w2 = Base::template pair_w2<kU>(r, s, e2u);
        ai[0] += w2;
        ai[1] = fmax_t(w2, ai[1]);
        aj[0] += w2;
        aj[1] = fmax_t(w2, aj[1]);
    }
    __device__ static constexpr double scale() { return 1.0; }
};

// Split-FP32: fields xh yh zh m xl yl zl e2 [vx vy vz], relative to the
// workgroup's frame.
template <class Op, int F>
__device__ __forceinline__ void split_fields(const PairArgs<double>& a,
                                             const typename Op::Frame& fr, int i, float (&f)[F])
{
    typename Op::Slot s;
    Op::load_j(a, fr, i, s);
#pragma unroll
    for (int k = 0; k < F; ++k) f[k] = s.v[k];
}

struct SymSplitAcc {
    using Base = OpSplitAcc;
    using T = float;
    static constexpr int kF = 8, kK = 3, kE2 = 7, kM0 = 3;
    static constexpr bool kMax1 = false, kPadSafe = false;
    __device__ static void load(const Base::Args& a, const Base::Frame& fr, int i, T (&f)[kF])
    {
        split_fields<Base>(a, fr, i, f);
    }
    __device__ static void pad(T (&f)[kF]) { sym_pad<kM0, kE2>(f); }
    template <bool kU, bool kM>
    __device__ static __forceinline__ void interact(const T (&I)[kF], const T (&J)[kF],
                                                    T (&ai)[kK], T (&aj)[kK], T e2u, T)
    {
        const float dx = (I[0] - J[0]) + (I[4] - J[4]);
        const float dy = (I[1] - J[1]) + (I[5] - J[5]);
        const float dz = (I[2] - J[2]) + (I[6] - J[6]);
        const float y = split_rsqrt<kSplitRefine, kM>(dx, dy, dz, kU ? e2u : I[7] + J[7]);
        const float q2 = y * y;
        const float wj = q2 * (y * J[3]), wi = q2 * (y * I[3]);
        ai[0] = __builtin_fmaf(-wj, dx, ai[0]);
        ai[1] = __builtin_fmaf(-wj, dy, ai[1]);
        ai[2] = __builtin_fmaf(-wj, dz, ai[2]);
        aj[0] = __builtin_fmaf(wi, dx, aj[0]);
        aj[1] = __builtin_fmaf(wi, dy, aj[1]);
        aj[2] = __builtin_fmaf(wi, dz, aj[2]);
    }
    __device__ static constexpr double scale() { return split_scale<kSplitRefine>(); }
};

struct SymSplitAccJerk {
    using Base = OpSplitAccJerk;
    using T = float;
    static constexpr int kF = 11, kK = 6, kE2 = 7, kM0 = 3;
    static constexpr bool kMax1 = false, kPadSafe = false;
    __device__ static void load(const Base::Args& a, const Base::Frame& fr, int i, T (&f)[kF])
    {
        split_fields<Base>(a, fr, i, f);
    }
    __device__ static void pad(T (&f)[kF]) { sym_pad<kM0, kE2>(f); }
    template <bool kU, bool kM>
    __device__ static __forceinline__ void interact(const T (&I)[kF], const T (&J)[kF],
                                                    T (&ai)[kK], T (&aj)[kK], T e2u, T)
    {
        const float dx = (I[0] - J[0]) + (I[4] - J[4]);
        const float dy = (I[1] - J[1]) + (I[5] - J[5]);
        const float dz = (I[2] - J[2]) + (I[6] - J[6]);
        float ux = I[8] - J[8], uy = I[9] - J[9], uz = I[10] - J[10];
        const float rv = __builtin_fmaf(dz, uz, __builtin_fmaf(dy, uy, dx * ux));
        const float y = split_rsqrt<kSplitRefine, kM>(dx, dy, dz, kU ? e2u : I[7] + J[7]);
        const float q2 = y * y;
        const float alpha = 3.0f * rv * q2;
        ux = __builtin_fmaf(-alpha, dx, ux);
        uy = __builtin_fmaf(-alpha, dy, uy);
        uz = __builtin_fmaf(-alpha, dz, uz);
        const float wj = q2 * (y * J[3]), wi = q2 * (y * I[3]);
        ai[0] = __builtin_fmaf(-wj, dx, ai[0]);
        ai[1] = __builtin_fmaf(-wj, dy, ai[1]);
        ai[2] = __builtin_fmaf(-wj, dz, ai[2]);
        ai[3] = __builtin_fmaf(-wj, ux, ai[3]);
        ai[4] = __builtin_fmaf(-wj, uy, ai[4]);
        ai[5] = __builtin_fmaf(-wj, uz, ai[5]);
        aj[0] = __builtin_fmaf(wi, dx, aj[0]);
        aj[1] = __builtin_fmaf(wi, dy, aj[1]);
        aj[2] = __builtin_fmaf(wi, dz, aj[2]);
        aj[3] = __builtin_fmaf(wi, ux, aj[3]);
        aj[4] = __builtin_fmaf(wi, uy, aj[4]);
        aj[5] = __builtin_fmaf(wi, uz, aj[5]);
    }
    __device__ static constexpr double scale() { return split_scale<kSplitRefine>(); }
};

struct SymSplitTstep {
    using Base = OpSplitTstep;
    using T = float;
    static constexpr int kF = 11, kK = 2, kE2 = 7, kM0 = 3;
    static constexpr bool kMax1 = true, kPadSafe = true;
    // masses held doubled, as OpSplitTstep's
    __device__ static void load(const Base::Args& a, const Base::Frame& fr, int i, T (&f)[kF])
    {
        split_fields<Base>(a, fr, i, f);
    }
    __device__ static void pad(T (&f)[kF]) { f[0] = __builtin_nanf(""); }
    template <bool kU, bool kM>
    __device__ static __forceinline__ void interact(const T (&I)[kF], const T (&J)[kF],
                                                    T (&ai)[kK], T (&aj)[kK], T e2u, T eta)
    {
        Base::IReg r;
        Base::Slot s;
        r.xh = I[0]; r.yh = I[1]; r.zh = I[2]; r.m = I[3];
        r.xl = I[4]; r.yl = I[5]; r.zl = I[6]; r.e2 = I[7];
        r.vx = I[8]; r.vy = I[9]; r.vz = I[10]; r.eta = eta;
#pragma unroll
        for (int k = 0; k < kF; ++k) s.v[k] = J[k];
        const float w2 = Base::pair_w2<kU>(r, s, e2u);
        ai[0] += w2;
        ai[1] = __builtin_fmaxf(w2, ai[1]);
        aj[0] += w2;
        aj[1] = __builtin_fmaxf(w2, aj[1]);
    }
    __device__ static constexpr double scale() { return 1.0; }
};

// The policy of a tile-engine op, where there is one.
template <class Op>
struct SymOf {
    using type = void;
};
template <> struct SymOf<OpPhi<Fast64>> { using type = SymPhi<Fast64>; };
template <> struct SymOf<OpAcc<Fast64>> { using type = SymAcc<Fast64>; };
template <> struct SymOf<OpAccJerk<Fast64>> { using type = SymAccJerk<Fast64>; };
template <> struct SymOf<OpSnapCrackle<Fast64>> { using type = SymSnapCrackle<Fast64>; };
template <> struct SymOf<OpTstep<Fast64>> { using type = SymTstep<Fast64>; };
template <> struct SymOf<OpPhi<Fast32>> { using type = SymPhi<Fast32>; };
template <> struct SymOf<OpAcc<Fast32>> { using type = SymAcc<Fast32>; };
template <> struct SymOf<OpAccJerk<Fast32>> { using type = SymAccJerk<Fast32>; };
template <> struct SymOf<OpSnapCrackle<Fast32>> { using type = SymSnapCrackle<Fast32>; };
template <> struct SymOf<OpTstep<Fast32>> { using type = SymTstep<Fast32>; };
template <> struct SymOf<OpSplitAcc> { using type = SymSplitAcc; };
template <> struct SymOf<OpSplitAccJerk> { using type = SymSplitAccJerk; };
template <> struct SymOf<OpSplitTstep> { using type = SymSplitTstep; };
template <class Op>
constexpr bool kHasSym = !std::is_void<typename SymOf<Op>::type>::value;
// Largest set an op leaves to the tile engine whatever the plan below says.
// Initial conditions are drawn from the FP64 Phi, and the 1e-14 comparison of
// two pair solvers on the 16384-particle realisation depends on its last
// bits, so a seed's realisation keeps the tile engine's summation order (and
// its j-splits: pairwise.hip, launch_tuned) up to 2^15 particles, where a
// potential costs under 0.7 ms (n = 32768: 0.67 there, 0.40 here); beyond,
// the time counts (n = 50000: 1.49 against 0.87 ms).
template <class Op>
inline constexpr int kSymOpAbove = 0;
template <>
inline constexpr int kSymOpAbove<OpPhi<Fast64>> = 32768;

// -- plan ---------------------------------------------------------------------
// Shapes {W, TJ}: W particles per lane, TJ j-particles per LDS tile.
constexpr int kNumSymShapes = 3;
constexpr int kSymShapeDims[kNumSymShapes][2] = {{4, 128}, {2, 64}, {1, 64}};

struct SymPlan {
    int shape;   // kSymShapeDims index, -1: the tile engine
    int nb;      // particle blocks
    int nchunk;  // workgroups per block row
};

// Tiles of row I: its own block and the blocks it meets.
__host__ __device__ inline int sym_row_tiles(int nb, int row, int tpb)
{
    int nd = (nb - 1) / 2;
    if (nb % 2 == 0 && row < nb / 2) ++nd;
    return (1 + nd) * tpb;
}

__host__ __device__ inline size_t sym_doubles(const SymPlan& p, int nk, int n)
{
    return static_cast<size_t>(p.nchunk + p.nb / 2) * nk * n;
}

// Smallest sets the symmetric engine takes, and where its shapes change.
// Up to kSymAbove the j tiles are too few to keep four waves on every SIMD
// and the tile engine's finer split is as fast or faster (split-FP32 Acc,
// n = 3000: 13 us of tile engine, 16 us here; FP64 AccJerk, n = 2300: 28 us
// and 17 us).  More particles per lane share each j rotation, fewer leave
// more workgroups: FP64 AccJerk takes 67, 70 us (W = 1, 2) at n = 7001, 113
// and 94 us at 9500, 824 and 873 us (W = 2, 4) at 32001, 1339 and 1285 us at
// 41000; the FP32 forms fill the ALU best with the four waves per SIMD that
// W = 2 leaves room for, and take W = 4 only where it halves a partial-sum
// array of several hundred MB at equal speed.  One rule serves every op of an
// arithmetic; off it by most is FP64 SnapCrackle, whose W = 4 holds one wave
// per SIMD: 2.97 ms at n = 37000, 2.58 under W = 2 (9.0 and 8.3 at 70000; tile
// engine 3.9 and 14.0).
// The bounds are multiples of the smaller shape's block, so every block
// count of a shape occurs at a whole multiple of its block.
constexpr int kSymAbove64 = 2048, kSymAbove32 = 4096;
constexpr int kSymW2Above = 9216;
constexpr int kSymW4Above64 = 36864, kSymW4Above32 = 131072;
// Partial sums of one call (4 GiB: FP64 AccJerk up to n = 420000); larger
// sets take the tile engine.
constexpr size_t kSymMaxBytes = static_cast<size_t>(4) << 30;

// kSymShapeDims index for n particles, -1 for the tile engine.
__host__ __device__ inline int sym_shape(int n, bool fp64)
{
    if (n <= (fp64 ? kSymAbove64 : kSymAbove32)) return -1;
    if (n > (fp64 ? kSymW4Above64 : kSymW4Above32)) return 0;
    return n > kSymW2Above ? 1 : 2;
}

// The plan of a set of n particles with nk sums on a device of cu CUs.
// Chunks per row: at least four workgroups per CU, eight where that leaves
// chunks of four tiles (the later ones even out what the CUs' speeds differ
// by), and of the counts up to four times that the one whose busiest CU has
// the least to do, a workgroup's fixed cost counted as half a tile.
__host__ __device__ inline SymPlan sym_plan(int n, int nk, bool fp64, int cu)
{
    SymPlan p{sym_shape(n, fp64), 0, 0};
    if (p.shape < 0) return p;
    const int bi = kSymBlock * kSymShapeDims[p.shape][0];
    p.nb = (n + bi - 1) / bi;
    const int tiles = sym_row_tiles(p.nb, 0, bi / kSymShapeDims[p.shape][1]);
    int lo = (8 * cu + p.nb - 1) / p.nb;
    if ((p.shape == 0 && fp64) || 4 * lo > tiles) lo = (4 * cu + p.nb - 1) / p.nb;
    if (lo > tiles) lo = tiles;
    long long best = -1;
    for (int nc = lo; nc <= tiles && nc <= 4 * lo; ++nc) {
        const long long cost =
            static_cast<long long>((p.nb * nc + cu - 1) / cu) * (2 * ((tiles + nc - 1) / nc) + 1);
        if (best < 0 || cost < best) {
            best = cost;
            p.nchunk = nc;
        }
    }
    if (sym_doubles(p, nk, n) > kSymMaxBytes / sizeof(double)) p.shape = -1;
    return p;
}

// -- kernels ------------------------------------------------------------------

// Every lane takes v of the lane below (lane 0 lane 63's).  The FP32 form is
// one block at raised priority (common.h: rsq_f32 has the reason); its s_nop
// is the wait a DPP read needs after a vector write of v.
#define TUPAN_ROR(k) "v_mov_b32_dpp %" #k ", %" #k " wave_ror:1 row_mask:0xf bank_mask:0xf\n\t"
template <int K>
__device__ __forceinline__ void wave_ror1(float (&v)[K])
{
    static_assert(K == 1 || K == 2 || K == 3 || K == 6, "one asm block per sum count");
    if constexpr (K == 1)
        asm("s_setprio 3\n\ts_nop 1\n\t" TUPAN_ROR(0) "s_setprio 0" : "+v"(v[0]));
    else if constexpr (K == 2)
        asm("s_setprio 3\n\ts_nop 1\n\t" TUPAN_ROR(0) TUPAN_ROR(1) "s_setprio 0" : "+v"(v[0]), "+v"(v[1]));
    else if constexpr (K == 3)
        asm("s_setprio 3\n\ts_nop 1\n\t" TUPAN_ROR(0) TUPAN_ROR(1) TUPAN_ROR(2) "s_setprio 0"
            : "+v"(v[0]), "+v"(v[1]), "+v"(v[2]));
    else
        asm("s_setprio 3\n\ts_nop 1\n\t" TUPAN_ROR(0) TUPAN_ROR(1) TUPAN_ROR(2) TUPAN_ROR(3) TUPAN_ROR(4) TUPAN_ROR(5) "s_setprio 0"
            : "+v"(v[0]), "+v"(v[1]), "+v"(v[2]), "+v"(v[3]), "+v"(v[4]), "+v"(v[5]));
}
#undef TUPAN_ROR
template <int K>
__device__ __forceinline__ void wave_ror1(double (&v)[K])
{
#pragma unroll
    for (int k = 0; k < K; ++k) {
        const unsigned long long b = __builtin_bit_cast(unsigned long long, v[k]);
        int lo = static_cast<int>(static_cast<unsigned>(b));
        int hi = static_cast<int>(static_cast<unsigned>(b >> 32));
        lo = __builtin_amdgcn_update_dpp(lo, lo, 0x13C, 0xf, 0xf, false);
        hi = __builtin_amdgcn_update_dpp(hi, hi, 0x13C, 0xf, 0xf, false);
        v[k] = __builtin_bit_cast(
            double, (static_cast<unsigned long long>(static_cast<unsigned>(hi)) << 32) |
                        static_cast<unsigned>(lo));
    }
}

// LDS written and read by one wave alone: its accesses happen in order, the
// compiler is told to keep them so.
__device__ __forceinline__ void wave_lds_sync()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

template <class S>
__device__ __forceinline__ double sym_join(double t, double v, int k)
{
    return S::kMax1 && k == 1 ? __builtin_fmax(t, v) : t + v;
}

// 64 j-particles against the lane's W particles.  `slot` is the sub-tile's
// field arrays (128 values each), `jp` the wave's j sums of the tile ([k][TJ],
// at this sub-tile).
template <class S, int W, int TJ, bool kU, bool kM>
__device__ __forceinline__ void sym_pass(const typename S::T* slot, int lane,
                                         const typename S::T (&I)[W][S::kF],
                                         typename S::T (&ai)[W][S::kK], double* jp,
                                         typename S::T e2u, typename S::T eta)
{
    using T = typename S::T;
    // FP32 j sums move to FP64 every 64 pairs, FP64 ones stay to the end
    constexpr int kRun = sizeof(T) == 4 ? kWave / W : kWave;
    constexpr int kUnroll = kRun < 4 ? kRun : 4;
    T aj[S::kK];
    for (int s0 = 0; s0 < kWave; s0 += kRun) {
#pragma unroll
        for (int k = 0; k < S::kK; ++k) aj[k] = T(0);
        for (int s1 = s0; s1 < s0 + kRun; s1 += kUnroll) {
            const T* base = slot + (kWave - s1) + lane;
#pragma unroll
            for (int u = 0; u < kUnroll; ++u) {
                T J[S::kF];
#pragma unroll
                for (int f = 0; f < S::kF; ++f) J[f] = base[f * 2 * kWave - u];
                wave_ror1(aj);
#pragma unroll
                for (int w = 0; w < W; ++w)
                    S::template interact<kU, kM>(I[w], J, ai[w], aj, e2u, eta);
            }
        }
        const int j = (lane - (s0 + kRun - 1)) & (kWave - 1);
        // j's sum of the runs before was written by another lane
        if (s0 > 0) wave_lds_sync();
#pragma unroll
        for (int k = 0; k < S::kK; ++k) {
            const double v = static_cast<double>(aj[k]) * S::scale();
            jp[k * TJ + j] = s0 == 0 ? v : sym_join<S>(jp[k * TJ + j], v, k);
        }
    }
}

template <class S, int W, int TJ>
__device__ __forceinline__ void sym_body(const typename S::Base::Args& a, int bid, int nb)
{
    using Op = typename S::Base;
    using T = typename S::T;
    constexpr int BI = kSymBlock * W;
    constexpr int kSub = TJ / kWave;
    constexpr int kSubLen = S::kF * 2 * kWave;
    static_assert(TJ % kWave == 0 && BI % TJ == 0 && TJ <= kSymBlock, "tile of whole sub-tiles");
    __shared__ T slots[kSub * kSubLen];
    __shared__ double jsum[kSymWaves * S::kK * TJ];

    const int n = a.ni;
    const int tid = static_cast<int>(threadIdx.x);
    const int lane = tid & (kWave - 1);
    const int wave = tid / kWave;
    const int row = bid / a.nsplit;
    const int chunk = bid % a.nsplit;
    const int ibase = row * BI;
    const typename Op::Frame fr = Op::frame(a, ibase);

    T I[W][S::kF];
    T ai[W][S::kK];
    double di[W][S::kK];
    [[maybe_unused]] T e2_i[W];
#pragma unroll
    for (int w = 0; w < W; ++w) {
        const int i = ibase + w * kSymBlock + tid;
        S::load(a, fr, i < n ? i : n - 1, I[w]);
        e2_i[w] = I[w][S::kE2];
        if (i >= n) S::pad(I[w]);
#pragma unroll
        for (int k = 0; k < S::kK; ++k) {
            ai[w][k] = T(0);
            di[w][k] = 0.0;
        }
    }

    // uniform softening and unmasked tiles, as in pair_body; both particles
    // of a pair must pass self_safe here
    constexpr bool kUni = HasUniformE2<Op>::value;
    constexpr bool kUnmask = kUni && HasUnmask<Op>::value;
    constexpr bool kSelf = kUnmask && HasSelfSafe<Op>::value;
    bool iuni = true;
    T e2_first = T(0);
    [[maybe_unused]] bool unmask = false;
    [[maybe_unused]] T y_self = T(0);
    [[maybe_unused]] bool pad_ok = true;  // no uniform tile overflows at a padding particle
    if constexpr (kUni) {
        e2_first = Op::e2_of_i(a, ibase);
        if constexpr (!kUnmask && !S::kPadSafe) {
            const T y = rsqrt_refined(e2_first + e2_first);
            pad_ok = __builtin_isfinite(y * y * y);
        }
#pragma unroll
        for (int w = 0; w < W; ++w) iuni = iuni && e2_i[w] == e2_first;
        iuni = iuni && (pad_ok || ibase + BI <= n);
    }
    if constexpr (kUnmask) unmask = Op::unmask_allowed(a);
    if constexpr (kSelf) {
        y_self = Op::self_y(e2_first + e2_first);
#pragma unroll
        for (int w = 0; w < W; ++w) unmask = unmask && Op::self_safe_m(y_self, I[w][S::kM0]);
    }
    const T eta = static_cast<T>(a.eta);

    const int row_tiles = sym_row_tiles(nb, row, BI / TJ);
    const int t0 = static_cast<int>(static_cast<long long>(row_tiles) * chunk / a.nsplit);
    const int t1 = static_cast<int>(static_cast<long long>(row_tiles) * (chunk + 1) / a.nsplit);
    double* jpart = a.partial + static_cast<size_t>(a.nsplit) * S::kK * n;
    // vmcnt(0): the i-particles' loads end here, or the compiler waits for
    // them in the pair loop, on every pass through it (float Phi: 2 %)
    __builtin_amdgcn_s_waitcnt(0x0f70);
    for (int t = t0; t < t1; ++t) {
        const int d = t / (BI / TJ);
        int jblock = row + d;
        if (jblock >= nb) jblock -= nb;
        const int j0 = jblock * BI + (t % (BI / TJ)) * TJ;
        if (j0 >= n) continue;
        __syncthreads();
        bool tuni = iuni;
        [[maybe_unused]] bool tsafe = unmask;
        if (tid < TJ) {
            T f[S::kF];
            const int j = j0 + tid;
            S::load(a, fr, j < n ? j : n - 1, f);
            if constexpr (kUni) tuni = tuni && f[S::kE2] == e2_first;
            if (j >= n) S::pad(f);
            if constexpr (kSelf) tsafe = tsafe && Op::self_safe_m(y_self, f[S::kM0]);
            T* dst = slots + (tid / kWave) * kSubLen + lane;
#pragma unroll
            for (int k = 0; k < S::kF; ++k) {
                dst[k * 2 * kWave] = f[k];
                dst[k * 2 * kWave + kWave] = f[k];
            }
        }
        bool special = false;
        if constexpr (kUnmask) {
            special = __syncthreads_and(tuni && tsafe);
        } else if constexpr (kUni) {
            special = __syncthreads_and(tuni) && (pad_ok || j0 + TJ <= n);
        } else {
            __syncthreads();
        }
        double* jp = jsum + wave * S::kK * TJ;
        for (int q = 0; q < kSub; ++q) {
            const T* slot = slots + q * kSubLen;
            if (kUni && special)
                sym_pass<S, W, TJ, true, !kUnmask>(slot, lane, I, ai, jp + q * kWave,
                                                   e2_first + e2_first, eta);
            else
                sym_pass<S, W, TJ, false, true>(slot, lane, I, ai, jp + q * kWave, e2_first, eta);
            if constexpr (sizeof(T) == 4) {
#pragma unroll
                for (int w = 0; w < W; ++w) {
#pragma unroll
                    for (int k = 0; k < S::kK; ++k) {
                        di[w][k] = sym_join<S>(di[w][k],
                                               static_cast<double>(ai[w][k]) * S::scale(), k);
                        ai[w][k] = T(0);
                    }
                }
            }
        }
        if (d > 0) {
            // the waves' j sums in wave order
            __syncthreads();
            for (int e = tid; e < S::kK * TJ; e += kSymBlock) {
                const int k = e / TJ, j = j0 + e % TJ;
                double v = jsum[e];
#pragma unroll
                for (int w = 1; w < kSymWaves; ++w)
                    v = sym_join<S>(v, jsum[w * S::kK * TJ + e], k);
                if (j < n) jpart[(static_cast<size_t>(d - 1) * S::kK + k) * n + j] = v;
            }
        }
    }
    double* ipart = a.partial + static_cast<size_t>(chunk) * S::kK * n;
#pragma unroll
    for (int w = 0; w < W; ++w) {
        const int i = ibase + w * kSymBlock + tid;
        if (i >= n) continue;
#pragma unroll
        for (int k = 0; k < S::kK; ++k)
            ipart[static_cast<size_t>(k) * n + i] =
                sizeof(T) == 4 ? di[w][k] : static_cast<double>(ai[w][k]);
    }
}

template <class S, int W, int TJ>
__global__ __launch_bounds__(kSymBlock) void sym_kernel(typename S::Base::Args a, int nb)
{
    sym_body<S, W, TJ>(a, static_cast<int>(blockIdx.x), nb);
}

// Adds each particle's partial sums: its chunks' i sums, then the j sums of
// the distances at which another block met its own, then Op's store.  Eight
// waves share 64 particles, wave g taking the slots g, g + 8, ... (batches of
// four, so that a lane has several slots' loads in flight), and wave 0 adds
// the eight totals in order.  A particle whose FP32 sums are not finite is
// evaluated again in FP64 by the whole wave.
constexpr int kSymReduceWaves = 8;

template <class S>
__device__ __forceinline__ void sym_reduce_body(const typename S::Base::Args& a, int bid, int nb,
                                                int bi)
{
    using Op = typename S::Base;
    constexpr int kBatch = 4;
    __shared__ double tots[kSymReduceWaves - 1][S::kK][kWave];
    const int n = a.ni;
    const int lane = static_cast<int>(threadIdx.x) & (kWave - 1);
    const int g = static_cast<int>(threadIdx.x) / kWave;
    const int i = bid * kWave + lane;
    const int ii = i < n ? i : n - 1;
    // the last distance of an even block count reaches the upper half only
    const int reach = nb / 2;
    const int nd = nb % 2 == 0 && ii / bi < nb / 2 ? reach - 1 : reach;
    const int terms = a.nsplit + nd;
    const size_t stride = static_cast<size_t>(S::kK) * n;
    double tot[S::kK];
#pragma unroll
    for (int k = 0; k < S::kK; ++k) tot[k] = 0.0;
    for (int s = g; s < terms; s += kSymReduceWaves * kBatch) {
        double part[kBatch][S::kK];
#pragma unroll
        for (int b = 0; b < kBatch; ++b) {
            const int q = s + b * kSymReduceWaves;
#pragma unroll
            for (int k = 0; k < S::kK; ++k)
                part[b][k] = q < terms ? a.partial[q * stride + static_cast<size_t>(k) * n + ii]
                                       : 0.0;
        }
#pragma unroll
        for (int b = 0; b < kBatch; ++b) {
#pragma unroll
            for (int k = 0; k < S::kK; ++k) tot[k] = sym_join<S>(tot[k], part[b][k], k);
        }
    }
    if (g > 0) {
#pragma unroll
        for (int k = 0; k < S::kK; ++k) tots[g - 1][k][lane] = tot[k];
    }
    __syncthreads();
    if (g > 0) return;
#pragma unroll
    for (int w = 0; w < kSymReduceWaves - 1; ++w) {
#pragma unroll
        for (int k = 0; k < S::kK; ++k) tot[k] = sym_join<S>(tot[k], tots[w][k][lane], k);
    }
    if constexpr (HasFallback<Op>::value) {
        unsigned long long bad = __ballot(i < n && !all_finite(tot));
        while (bad) {
            const int l = __ffsll(static_cast<long long>(bad)) - 1;
            bad &= bad - 1;
            double t[S::kK];
            fallback64<typename Op::Fallback64>(a, bid * kWave + l, lane, n, kWave, t);
#pragma unroll
            for (int off = kWave / 2; off > 0; off >>= 1) {
#pragma unroll
                for (int k = 0; k < S::kK; ++k) t[k] = sym_join<S>(t[k], __shfl_xor(t[k], off), k);
            }
            if (lane == l) {
#pragma unroll
                for (int k = 0; k < S::kK; ++k) tot[k] = t[k];
            }
        }
    }
    if (i < n) Op::store(a, i, tot);
}

template <class S>
__global__ __launch_bounds__(kSymReduceWaves * kWave) void sym_reduce_kernel(
    typename S::Base::Args a, int nb, int bi)
{
    sym_reduce_body<S>(a, static_cast<int>(blockIdx.x), nb, bi);
}

}  // namespace tupan
