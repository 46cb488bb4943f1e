// energy.hip — Eq.15 DG/Crank-Nicolson energy half step (psi^1, psi^2).
//
// Reference: energyDgCnKernel, eq15 branch (src/energy_solver.cu:41-161) and
// the copy-back in EnergyDepositionSolver::solve (src/energy_solver.cu:497-505).
//
// MI355X design:
//  * one thread per phase-space lane (s, m); lanes are contiguous for a fixed
//    group g, so every load/store of the sweep is a fully coalesced row;
//  * the sweep runs in place: the old values of g+1 (needed by the
//    straggling and slope couplings) and the new Delta_{g+1} are carried in
//    registers, so the reference's scratch arrays and D2D copy-back vanish;
//  * group coefficients come from a host-built FP64 table (wave-uniform, so
//    they are scalar loads) and the recurrence runs in FP64 for any state
//    type;
//  * loads run 16 groups (FP64 state: 8) ahead in a register ring to hide HBM
//    latency behind the serial recurrence (small grids leave only a few
//    waves per SIMD); per-group coefficients, dose weights included, come
//    through the scalar cache so they never queue behind the ring;
//  * grids of few lanes share a lane between two threads, one per linear form
//    (energy_split_kernel);
//  * the final E-half of a depth step also accumulates the Eq.24 dose and the
//    psi^2 proxy in FP64 (block partials, reduced deterministically later), so
//    the IDD costs no extra pass over the state.

#include "buffer.hpp"
#include "kernels.hpp"
#include "mfma.hpp"

#include <type_traits>

#include <utility>

namespace bfpn {
namespace {

constexpr int kBlock = 256;

__device__ inline double block_sum(double v, double* lds) {
    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off);
    const int wave = threadIdx.x >> 6;
    if ((threadIdx.x & 63) == 0) lds[wave] = v;
    __syncthreads();
    double t = 0.0;
    if (threadIdx.x == 0)
        for (int w = 0; w < kBlock / 64; ++w) t += lds[w];
    __syncthreads();
    return t;
}

__device__ inline int block_max(int v, int* lds) {
    for (int off = 32; off > 0; off >>= 1) v = max(v, __shfl_xor(v, off));
    const int wave = threadIdx.x >> 6;
    if ((threadIdx.x & 63) == 0) lds[wave] = v;
    __syncthreads();
    int t = -1;
    if (threadIdx.x == 0)
        for (int w = 0; w < kBlock / 64; ++w) t = max(t, lds[w]);
    __syncthreads();
    return t;
}

// Results below the smallest normal number of the state type are flushed to
// zero (what a flush-to-zero mode does).  Without it the upper energy tail of
// a beam never vanishes: a value at the smallest denormal, scaled by a decay
// factor above 1/2 each half step, rounds back to itself, so the top nonzero
// group could never fall as the beam slows.  The change is below 2^-126 of
// the state's scale in FP32 (2^-1022 in FP64).
template <typename T>
__device__ inline double flush_tiny(double v) {
    constexpr double tiny = sizeof(T) == 4 ? 1.1754943508222875e-38 : 2.2250738585072014e-308;
    return fabs(v) < tiny ? 0.0 : v;
}

// Top group of the state a sweep reads, and of a source made from a primary
// state with top *x (all groups when the tops are not tracked).
__device__ inline int state_top(const SweepTops& t, int Ng) { return t.in ? *t.in : Ng - 1; }
__device__ inline int source_top(const SweepTops& t, const int* x, int Ng) {
    const int top = (t.qmap && x) ? t.qmap[max(-1, min(Ng - 1, *x)) + 1] : Ng - 1;
    return max(-1, min(top, t.q_cap));
}
// Source row read at group g: rows above the source's top are masked where
// used, so their loads re-read the top row (an L2 hit) instead of HBM.
__device__ inline long long source_row(int g, int q_top) {
    return static_cast<long long>(max(min(g, q_top), 0));
}

// Presets the slots a later sweep writes (one thread of the grid).
__device__ inline void reset_tops(const SweepTops& t) {
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        if (t.reset) *t.reset = -1;
        if (t.reset_x) *t.reset_x = -1;
    }
}

// Publishes a block's highest nonzero output group (-1: none).
__device__ inline void publish_top(int top, int* out, int* out2, int* lds) {
    const int b = block_max(top, lds);
    if (threadIdx.x == 0 && b >= 0) {
        if (out) atomicMax(out, b);
        if (out2) atomicMax(out2, b);
    }
}

// LPT adjacent lanes per thread (4 with FP32 state on large lane counts):
// 16-byte row loads and stores, four independent recurrences in flight per
// thread, one set of coefficient loads for four lanes.
template <typename T, int LPT>
struct Pack {
    T v[LPT];
};

// f(integral_constant<int, 0>), ..., f(integral_constant<int, N - 1>)
template <typename F, int... I>
__device__ inline void unroll_seq(F&& f, std::integer_sequence<int, I...>) {
    (f(std::integral_constant<int, I>{}), ...);
}
template <int N, typename F>
__device__ inline void unroll(F&& f) {
    unroll_seq(f, std::make_integer_sequence<int, N>{});
}

// Loads and stores are non-temporal: every element is touched once per sweep
// and nothing the sweep moves is read again before the next operator has
// streamed the whole state through the caches, so keeping it out of L2 only
// frees the cache for the loads in flight (on the paper grid the paired
// sweeps ran 12 % faster with non-temporal stores and 3 % more with
// non-temporal loads).
template <typename T, int LPT>
__device__ inline Pack<T, LPT> load_pack(const T* p) {
    Pack<T, LPT> r;
    if constexpr (LPT == 4) {
        static_assert(sizeof(T) == 4, "4-lane packs are FP32");
        typedef float f32x4v __attribute__((ext_vector_type(4)));
        const f32x4v q = __builtin_nontemporal_load(reinterpret_cast<const f32x4v*>(p));
        r.v[0] = q[0];
        r.v[1] = q[1];
        r.v[2] = q[2];
        r.v[3] = q[3];
    } else {
        static_assert(LPT == 1, "one or four lanes per thread");
        r.v[0] = __builtin_nontemporal_load(p);
    }
    return r;
}

template <typename T, int LPT>
__device__ inline void store_pack(T* p, const double (&v)[LPT]) {
    if constexpr (LPT == 4) {
        typedef float f32x4v __attribute__((ext_vector_type(4)));
        const f32x4v q = {static_cast<float>(v[0]), static_cast<float>(v[1]),
                          static_cast<float>(v[2]), static_cast<float>(v[3])};
        __builtin_nontemporal_store(q, reinterpret_cast<f32x4v*>(p));
    } else {
        __builtin_nontemporal_store(static_cast<T>(v[0]), p);
    }
}

// Prefetch depth D (groups in flight per thread).  The register ring has
// D + 1 slots and the sweep is unrolled by D + 1, so slot indices are
// compile-time constants: the step on group g (slot k) loads group g - D
// into slot k - 1, which the previous step has finished with.  No load ever
// targets a register whose old value is still in use, so the compiler never
// has to copy a loaded value -- a copy waits for the load and would drain
// the ring.
template <typename T, int LPT>
constexpr int prefetch_depth() { return LPT == 4 ? 8 : (sizeof(T) == 4 ? 16 : 8); }

// Lanes per thread for a sweep over `lanes` lanes of `elem`-byte state.
inline int lanes_per_thread(long long lanes, size_t elem) {
    return (elem == 4 && lanes % 4 == 0 && lanes >= (1LL << 18)) ? 4 : 1;
}

// The two linear forms of a group (f_new = af.x, F_new = aF.x over
// x = (P_hi, R_hi, P, R, P_lo, Q, Delta_hi)), wave-uniform: scalar loads.
struct Forms {
    double af[7], aF[7];
};

__device__ inline Forms load_forms(const EnergyCoef* coef, int g) {
    Forms r;
#pragma unroll
    for (int i = 0; i < 7; ++i) {
        r.af[i] = coef[g].af[i];
        r.aF[i] = coef[g].aF[i];
    }
    return r;
}

// One group of one lane's recurrence: input (P, R) at g, carried input
// (P_hi, R_hi) and output difference hd at g+1; returns the outputs (a: psi^2,
// b: psi^1) and moves the carries to g.  Inputs are state values, so the
// carries are held in the state type C (exactly).
template <bool SRC, bool STRAG, typename C>
__device__ inline void recur(const Forms& c, C P, C R, double P_lo, double src, C& P_hi, C& R_hi,
                             double& hd, double& a, double& b) {
    const double Ph = P_hi, Rh = R_hi, Pd = P, Rd = R;
    // explicit FMAs: every kernel that inlines this evaluates it identically
    // (left to the compiler, contraction could differ between kernels and
    // break the paired sweep's bit-identity with two single sweeps)
    a = fma(c.af[3], Rd, fma(c.af[2], Pd, fma(c.af[1], Rh, c.af[0] * Ph)));
    b = fma(c.aF[3], Rd, fma(c.aF[2], Pd, fma(c.aF[1], Rh, c.aF[0] * Ph)));
    if (STRAG) {
        a = fma(c.af[4], P_lo, a);
        b = fma(c.aF[4], P_lo, b);
    }
    if (SRC) {
        a = fma(c.af[5], src, a);
        b = fma(c.aF[5], src, b);
    }
    a = flush_tiny<C>(fma(c.af[6], hd, a));
    b = flush_tiny<C>(fma(c.aF[6], hd, b));
    P_hi = P;
    R_hi = R;
    hd = b - a;
}

// Eq.24 dose of one group's result, accumulated with explicit FMAs (the same
// operations in every kernel, see recur).
__device__ inline double add_dose(double acc, double F, double f, double w1, double w2) {
    return fma(f, w2, fma(F, w1, acc));
}

// Everything a group needs besides the state (recurrence coefficients and the
// dose weights) sits in one EnergyCoef read through the scalar cache, so the
// vector loads in flight are the state ring alone: the in-order load counter
// then never waits on the ring to deliver a coefficient.
template <typename T, int LPT, bool SRC, bool STRAG, bool DOSE>
__global__ __launch_bounds__(kBlock) void energy_half_kernel(
    T* __restrict__ F, T* __restrict__ f, const EnergyCoef* __restrict__ coef,
    const T* __restrict__ Q1, int Ng, int lanes, const double* __restrict__ yzw, int nang,
    double* __restrict__ partials, int proxy, SweepTops tops) {
    constexpr int D = prefetch_depth<T, LPT>(), RING = D + 1;
    __shared__ double lds[kBlock / 64];
    __shared__ int ldi[kBlock / 64];
    const int lane = (blockIdx.x * kBlock + threadIdx.x) * LPT;  // first of LPT lanes
    reset_tops(tops);
    // Groups above G0 are zero before and after the sweep: the state above
    // its top, the source above its own, and straggling lifts the result at
    // most one group.  Source values above the source's top are not read.
    const int q_top = SRC ? source_top(tops, tops.xa, Ng) : -1;
    const int G0 = min(Ng - 1, max(state_top(tops, Ng), q_top) + (STRAG ? 1 : 0));
    int top = -1;  // highest group with a nonzero result in this thread's lanes
    double acc_dose = 0.0, acc_proxy = 0.0;
    if (lane < lanes) {
        Pack<T, LPT> rF[RING], rf[RING], rQ[RING];
        // Loads are unconditional (groups below 0 re-read group 0 and are
        // never consumed) and full chunks run without branches, so the
        // compiler can count the loads in flight instead of draining them.
        // Row bases are wave-uniform (scalar), the lane a 32-bit offset.
        auto fetch = [&](int k, int g) {
            const long long base = static_cast<long long>(max(g, 0)) * lanes;
            rF[k] = load_pack<T, LPT>(F + base + lane);
            rf[k] = load_pack<T, LPT>(f + base + lane);
            if (SRC) rQ[k] = load_pack<T, LPT>(Q1 + source_row(g, q_top) * lanes + lane);
        };
#pragma unroll
        for (int k = 0; k < D; ++k) fetch(k, G0 - k);
        T P_hi[LPT], R_hi[LPT];
        double hi_delta[LPT], dose[LPT];
#pragma unroll
        for (int j = 0; j < LPT; ++j) {
            P_hi[j] = R_hi[j] = T(0);
            hi_delta[j] = dose[j] = 0.0;
        }
        // The linear forms run one group ahead through the scalar cache:
        // group g-1's are requested before group g's arithmetic (the
        // scheduling barrier keeps the request there), so their latency is
        // covered.  (Dose weights are read at use: two sets of forms plus
        // them would not fit the scalar registers.)
        Forms cn = load_forms(coef, max(G0, 0));
        auto step = [&](auto slot, int g) {  // group g sits in ring slot `slot`
            constexpr int k = decltype(slot)::value;
            const Forms c = cn;
            cn = load_forms(coef, max(g - 1, 0));
            __builtin_amdgcn_sched_barrier(0);
            fetch((k + D) % RING, g - D);
            const Pack<T, LPT> cF = rF[k], cf = rf[k], cQ = rQ[k];
            const Pack<T, LPT> lo = rF[(k + 1) % RING];  // old F at g-1
            const bool q_live = g <= q_top;
            double Fv[LPT], fv[LPT];
#pragma unroll
            for (int j = 0; j < LPT; ++j)
                recur<SRC, STRAG>(c, cF.v[j], cf.v[j], g > 0 ? static_cast<double>(lo.v[j]) : 0.0,
                                  SRC && q_live ? static_cast<double>(cQ.v[j]) : 0.0, P_hi[j],
                                  R_hi[j], hi_delta[j], fv[j], Fv[j]);
            const long long base = static_cast<long long>(g) * lanes;
            store_pack<T, LPT>(F + base + lane, Fv);
            store_pack<T, LPT>(f + base + lane, fv);
            bool nz = false;
#pragma unroll
            for (int j = 0; j < LPT; ++j)
                nz |= (static_cast<T>(Fv[j]) != T(0)) | (static_cast<T>(fv[j]) != T(0));
            top = max(top, nz ? g : -1);
            if (DOSE) {  // the lanes' transverse weights are applied after the sweep
                const double w1 = coef[g].w1, w2 = coef[g].w2;
#pragma unroll
                for (int j = 0; j < LPT; ++j) {
                    dose[j] = add_dose(dose[j], Fv[j], fv[j], w1, w2);
                    acc_proxy += fv[j];
                }
            }
        };
        int g0 = G0;
        for (; g0 >= RING - 1; g0 -= RING)
            unroll<RING>([&](auto k) { step(k, g0 - decltype(k)::value); });
        unroll<RING>([&](auto k) {  // tail: groups g0 .. 0 (fewer than RING)
            if (decltype(k)::value <= g0) step(k, g0 - decltype(k)::value);
        });
        // (loaded only now: a load issued before the ring would hold up its
        // first consumer behind every state load in flight)
        if (DOSE)
#pragma unroll
            for (int j = 0; j < LPT; ++j) acc_dose = fma(dose[j], yzw[(lane + j) / nang], acc_dose);
    }
    if (DOSE) {
        const double d = block_sum(acc_dose, lds);
        if (threadIdx.x == 0) partials[blockIdx.x] = d;
        if (proxy) {
            const double p = block_sum(acc_proxy, lds);
            if (threadIdx.x == 0) partials[gridDim.x + blockIdx.x] = p;
        }
    }
    if (tops.out) publish_top(top, tops.out, tops.out_x, ldi);
}

// Two consecutive half steps in one sweep: the final E-half of depth step n
// (source Qa, with the dose and proxy of step n) and the first E-half of step
// n+1 (source Qb), i.e. E(h) o E(h) over the same coefficients, reading and
// writing the state once instead of twice.  The second recurrence runs one
// group behind the first: at group g it needs the first's outputs at g+1 and
// g+2 and, for straggling, at g, which the first has just produced.  The
// first's outputs are rounded to the state type before the second uses them,
// exactly as if stored and reloaded, so the result is bit-identical to two
// launches.  XOUT also stores them (the state at the end of step n, which the
// secondary source of step n reads).
template <typename T, int LPT, bool SRC>
constexpr int pair_depth() {
    return LPT == 4 ? (SRC ? 4 : 6) : (sizeof(T) == 4 ? (SRC ? 10 : 14) : (SRC ? 4 : 6));
}

template <typename T, int LPT, bool SRC, bool STRAG, bool XOUT>
__global__ __launch_bounds__(kBlock) void energy_pair_kernel(
    T* __restrict__ F, T* __restrict__ f, const EnergyCoef* __restrict__ coef,
    const T* __restrict__ Qa, const T* __restrict__ Qb, T* __restrict__ XF, T* __restrict__ Xf,
    const unsigned* __restrict__ xmask, int Ng, int lanes, const double* __restrict__ yzw,
    int nang, double* __restrict__ partials, int proxy, SweepTops tops) {
    constexpr int D = pair_depth<T, LPT, SRC>(), RING = D + 1;
    __shared__ double lds[kBlock / 64];
    __shared__ int ldi[kBlock / 64];
    const int lane = (blockIdx.x * kBlock + threadIdx.x) * LPT;
    reset_tops(tops);
    // The first half's result is zero above t1, the second's above G0 (see
    // energy_half_kernel); both recurrences start at G0.
    const int qa_top = SRC ? source_top(tops, tops.xa, Ng) : -1;
    const int qb_top = SRC ? source_top(tops, tops.xb, Ng) : -1;
    const int t1 = max(state_top(tops, Ng), qa_top) + (STRAG ? 1 : 0);
    const int G0 = min(Ng - 1, max(t1, qb_top) + (STRAG ? 1 : 0));
    int top_a = -1, top_b = -1;  // highest nonzero group of each half's result
    double acc_dose = 0.0, acc_proxy = 0.0;
    if (lane < lanes && G0 >= 0) {
        Pack<T, LPT> rF[RING], rf[RING], rQa[RING], rQb[RING];
        // Qb (the second half's source) is refilled separately, at the end of
        // a step: the second half reads slot k - 1's Qb in the step that
        // refills that slot.
        auto fetch = [&](int k, int g) {
            const long long base = static_cast<long long>(max(g, 0)) * lanes;
            rF[k] = load_pack<T, LPT>(F + base + lane);
            rf[k] = load_pack<T, LPT>(f + base + lane);
            if (SRC) rQa[k] = load_pack<T, LPT>(Qa + source_row(g, qa_top) * lanes + lane);
        };
        auto fetch_qb = [&](int k, int g) {
            if (SRC) rQb[k] = load_pack<T, LPT>(Qb + source_row(g, qb_top) * lanes + lane);
        };
#pragma unroll
        for (int k = 0; k < D; ++k) {
            fetch(k, G0 - k);
            fetch_qb(k, G0 - k);
        }
        // first half: carried input at g+1, output difference; dose sums
        T P_hi[LPT], R_hi[LPT];
        double hd[LPT], dose[LPT];
        // second half, one group behind: its input (the first's output,
        // rounded to the state type) at g+1 and g+2, its output difference
        T P2[LPT], R2[LPT], P2_hi[LPT], R2_hi[LPT];
        double hd2[LPT];
#pragma unroll
        for (int j = 0; j < LPT; ++j) {
            P_hi[j] = R_hi[j] = P2[j] = R2[j] = P2_hi[j] = R2_hi[j] = T(0);
            hd[j] = dose[j] = hd2[j] = 0.0;
        }
        // second half at group g2, whose lower neighbour's input is P_lo2 and
        // whose source is q
        auto second = [&](int g2, const T (&P_lo2)[LPT], const Pack<T, LPT>& q) {
            // (requested here, not hoisted: three sets of forms live at once
            // would not fit the scalar registers)
            __builtin_amdgcn_sched_barrier(0);
            const Forms c2 = load_forms(coef, g2);
            const bool q_live = g2 <= qb_top;
            double Fv[LPT], fv[LPT];
#pragma unroll
            for (int j = 0; j < LPT; ++j)
                recur<SRC, STRAG>(c2, P2[j], R2[j], static_cast<double>(P_lo2[j]),
                                  SRC && q_live ? static_cast<double>(q.v[j]) : 0.0, P2_hi[j],
                                  R2_hi[j], hd2[j], fv[j], Fv[j]);
            const long long base = static_cast<long long>(g2) * lanes;
            store_pack<T, LPT>(F + base + lane, Fv);
            store_pack<T, LPT>(f + base + lane, fv);
            bool nz = false;
#pragma unroll
            for (int j = 0; j < LPT; ++j)
                nz |= (static_cast<T>(Fv[j]) != T(0)) | (static_cast<T>(fv[j]) != T(0));
            top_b = max(top_b, nz ? g2 : -1);
        };
        Forms cn = load_forms(coef, G0);
        // group g in ring slot `slot`; FIRST: g = Ng - 1, no second half behind it
        auto step = [&](auto slot, int g, auto first) {
            constexpr int k = decltype(slot)::value;
            const Forms c = cn;
            cn = load_forms(coef, max(g - 1, 0));
            __builtin_amdgcn_sched_barrier(0);
            fetch((k + D) % RING, g - D);
            const Pack<T, LPT> cF = rF[k], cf = rf[k], cQa = rQa[k];
            const Pack<T, LPT> lo = rF[(k + 1) % RING];
            const bool q_live = g <= qa_top;
            double Fv[LPT], fv[LPT];
            T tF[LPT];
#pragma unroll
            for (int j = 0; j < LPT; ++j)
                recur<SRC, STRAG>(c, cF.v[j], cf.v[j], g > 0 ? static_cast<double>(lo.v[j]) : 0.0,
                                  SRC && q_live ? static_cast<double>(cQa.v[j]) : 0.0, P_hi[j],
                                  R_hi[j], hd[j], fv[j], Fv[j]);
            {  // dose and proxy of step n from the first half's outputs
                const double w1 = coef[g].w1, w2 = coef[g].w2;
#pragma unroll
                for (int j = 0; j < LPT; ++j) {
                    dose[j] = add_dose(dose[j], Fv[j], fv[j], w1, w2);
                    acc_proxy += fv[j];
                }
            }
            // (only the groups the source reads, when xmask is given)
            if (XOUT && (!xmask || ((xmask[g >> 5] >> (g & 31)) & 1u))) {
                const long long base = static_cast<long long>(g) * lanes;
                store_pack<T, LPT>(XF + base + lane, Fv);
                store_pack<T, LPT>(Xf + base + lane, fv);
            }
            bool nz = false;
#pragma unroll
            for (int j = 0; j < LPT; ++j) {
                tF[j] = static_cast<T>(Fv[j]);
                nz |= (tF[j] != T(0)) | (static_cast<T>(fv[j]) != T(0));
            }
            top_a = max(top_a, nz ? g : -1);
            if (!decltype(first)::value) second(g + 1, tF, rQb[(k + D) % RING]);  // Qb at g+1
            fetch_qb((k + D) % RING, g - D);
#pragma unroll
            for (int j = 0; j < LPT; ++j) {  // the first's output at g: the second's next input
                P2[j] = tF[j];
                R2[j] = static_cast<T>(fv[j]);
            }
        };
        // group G0 (slot 0) on its own, so the loop body has no branch
        step(std::integral_constant<int, 0>{}, G0, std::true_type{});
        int g0 = G0 - 1;  // in slot 1
        for (; g0 >= RING - 1; g0 -= RING)
            unroll<RING>([&](auto i) {
                step(std::integral_constant<int, (decltype(i)::value + 1) % RING>{},
                     g0 - decltype(i)::value, std::false_type{});
            });
        unroll<RING>([&](auto i) {
            if (decltype(i)::value <= g0)
                step(std::integral_constant<int, (decltype(i)::value + 1) % RING>{},
                     g0 - decltype(i)::value, std::false_type{});
        });
        const T none[LPT] = {};
        Pack<T, LPT> q0{};
        if (SRC) q0 = load_pack<T, LPT>(Qb + lane);
        second(0, none, q0);  // group 0 has no lower neighbour
#pragma unroll
        for (int j = 0; j < LPT; ++j) acc_dose = fma(dose[j], yzw[(lane + j) / nang], acc_dose);
    }
    const double d = block_sum(acc_dose, lds);
    if (threadIdx.x == 0) partials[blockIdx.x] = d;
    if (proxy) {
        const double p = block_sum(acc_proxy, lds);
        if (threadIdx.x == 0) partials[gridDim.x + blockIdx.x] = p;
    }
    if (tops.out) publish_top(top_b, tops.out, nullptr, ldi);
    if (tops.out_x) publish_top(top_a, tops.out_x, nullptr, ldi);
}

// ------------------------------------------------------ few lanes: split ---
// The sweeps on grids of few lanes (energy_split).  There the time is the
// serial walk over the groups of a wave that has a SIMD to itself: the
// instructions it issues per group and every latency it exposes.  One thread
// per lane left most SIMDs idle and waited at every group for coefficients
// (scalar loads return out of order, so the wait for the second half's set
// also drained the prefetch of the next).  Here
//  * two adjacent threads share a lane and evaluate one linear form each
//    (role 0: f, role 1: F), exchanging results by a DPP swap: half the
//    arithmetic per wave and twice the waves, one per work-group, so they
//    spread over the CUs;
//  * the coefficients of 16 groups at a time are staged in LDS in the order
//    the roles read them; a group's are read one group ahead, and the second
//    half's are the registers the first half used one group before;
//  * rows are addressed through buffer resources by one running scalar offset,
//    and the highest nonzero group is looked for only until it is found.
// The operations on each value are those of recur(), in its order, so states
// are bit-identical to the kernels above.  Loads and stores are temporal: at
// these sizes the state stays in the caches between operators.
constexpr int kSplitRing = 16;  // groups per LDS chunk, the unroll
// Slots of the register ring (a divisor of kSplitRing).
template <typename T, bool FOUR>
constexpr int split_ring() { return FOUR || sizeof(T) == 8 ? 8 : 16; }

// Lanes of one array from which one thread per lane is the better sweep.  32,768
// lanes are one wave here for every SIMD; beyond that some SIMDs run two, which a
// paired sweep's registers allow in FP32 only, and one thread per lane starts to
// fill the chip.  Sweeps with dose sums, most of them paired (eight steps of a
// march x 250 groups, split against not): FP32 38,416 lanes 2.35 against 2.52 ms,
// 43,264 2.55 against 2.76, 44,100 2.84 against 2.82, 56,644 3.80 against 3.31;
// FP64 23,716 4.68 against 5.02, 28,561 5.51 against 5.56, 33,124 6.33 against
// 6.08, 56,644 11.2 against 10.2.  A single sweep without them has the registers
// for two waves (one sweep x 250 groups): FP32 44,100 lanes 66 against 72 us,
// 48,841 76 against 73, but where every row starts on a 64-byte boundary 50,176
// 48 against 72 and 63,504 68 against 76; FP64 43,264 83 against 92, 44,100 107
// against 100, 50,176 109 against 97.
inline bool energy_split(long long lanes, int Ng, size_t elem, bool sums = true) {
    const long long limit = sums ? (elem == 4 ? 44000 : 30000)
                            : elem == 8      ? 43500
                            : lanes % 16 == 0 ? (1LL << 16)
                                              : 47000;
    return lanes < limit && lanes * Ng * static_cast<long long>(elem) < (1LL << 31);
}

__device__ inline double swap_pair(double v) {
    const unsigned long long u = __builtin_bit_cast(unsigned long long, v);
    const unsigned lo = __builtin_amdgcn_mov_dpp(static_cast<int>(u), 0xB1, 0xF, 0xF, false);
    const unsigned hi = __builtin_amdgcn_mov_dpp(static_cast<int>(u >> 32), 0xB1, 0xF, 0xF, false);
    return __builtin_bit_cast(double, (static_cast<unsigned long long>(hi) << 32) | lo);
}
__device__ inline float swap_pair(float v) {
    return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0xB1, 0xF, 0xF, false));
}

// One role's coefficients of a group: the form's seven (the output
// difference's negated for role 0, whose difference is) and its dose weight.
struct RoleForm {
    double c[8];
};

// One half's carried values in a thread: inputs at g + 1, and own - other of
// its outputs there (b - a for role 1, the negation for role 0).
template <typename T>
struct SplitHalf {
    double P_hi = 0.0, R_hi = 0.0, diff = 0.0;
    // The thread's output at g: recur()'s `a` (role 0) or `b` (role 1).
    template <bool SRC, bool STRAG>
    __device__ inline double step(const RoleForm& k, double P, double R, double P_lo, double src) {
        double v = fma(k.c[3], R, fma(k.c[2], P, fma(k.c[1], R_hi, k.c[0] * P_hi)));
        if (STRAG) v = fma(k.c[4], P_lo, v);
        if (SRC) v = fma(k.c[5], src, v);
        v = flush_tiny<T>(fma(k.c[6], diff, v));
        P_hi = P;
        R_hi = R;
        diff = v - swap_pair(v);
        return v;
    }
};

// PAIR: the two half steps of energy_pair_kernel (DOSE is always on then);
// otherwise energy_half_kernel.  One wave per work-group, 32 lanes.  XOUT
// writes every group up to the top: a branch per group costs more here than
// the rows nobody reads.
template <typename T, bool PAIR, bool SRC, bool STRAG, bool DOSE, bool XOUT>
__global__ __launch_bounds__(64) void energy_split_kernel(
    T* __restrict__ F, T* __restrict__ f, const EnergyCoef* __restrict__ coef,
    const T* __restrict__ Qa, const T* __restrict__ Qb, T* __restrict__ XF, T* __restrict__ Xf,
    int Ng, int lanes, const double* __restrict__ yzw, int nang, double* __restrict__ partials,
    int proxy, SweepTops tops) {
    typedef double f64x2 __attribute__((ext_vector_type(2)));
    constexpr int R = kSplitRing;
    constexpr int RING = split_ring<T, PAIR && SRC>(), D = RING - 1;
    __shared__ __attribute__((aligned(16))) double forms[2][R][2][8];  // [chunk][group][role]
    reset_tops(tops);
    const int role = threadIdx.x & 1;
    const int own_lane = blockIdx.x * 32 + (threadIdx.x >> 1);
    // Threads past the last lane repeat it: they sit in the wave that owns it,
    // so they load and store the same values in the same instructions.
    const bool live = own_lane < lanes;
    const int lane = min(own_lane, lanes - 1);
    const int qa_top = SRC ? source_top(tops, tops.xa, Ng) : -1;
    const int qb_top = SRC && PAIR ? source_top(tops, tops.xb, Ng) : -1;
    const int t1 = max(state_top(tops, Ng), qa_top) + (STRAG ? 1 : 0);
    const int G0 = min(Ng - 1, PAIR ? max(t1, qb_top) + (STRAG ? 1 : 0) : t1);
    int top_a = -1, top_b = -1;
    double dose = 0.0, psum = 0.0;
    if (G0 >= 0) {
        const int row = lanes * static_cast<int>(sizeof(T));  // bytes of one group's row
        const unsigned bytes = static_cast<unsigned>(row) * static_cast<unsigned>(Ng);
        const __amdgpu_buffer_rsrc_t bF = make_rsrc(F, bytes), bf = make_rsrc(f, bytes);
        const __amdgpu_buffer_rsrc_t ba = make_rsrc(const_cast<T*>(SRC ? Qa : F), bytes);
        const __amdgpu_buffer_rsrc_t bb = make_rsrc(const_cast<T*>(SRC && PAIR ? Qb : F), bytes);
        const unsigned voff = static_cast<unsigned>(lane) * sizeof(T);
        const int qa_row = max(qa_top, 0) * row, qb_row = max(qb_top, 0) * row;
        T rF[RING], rf[RING], rQa[RING], rQb[RING];
        auto fetch = [&](int k, int at) {  // the row at byte offset `at` into slot k
            rF[k] = bload<T>(bF, voff, at);
            rf[k] = bload<T>(bf, voff, at);
            if (SRC) rQa[k] = bload<T>(ba, voff, min(at, qa_row));
        };
        auto fetch_qb = [&](int k, int at) {
            if (SRC && PAIR) rQb[k] = bload<T>(bb, voff, min(at, qb_row));
        };
        // Chunk staging: thread t holds four values of group g0 - t / 4: role
        // (t / 2) % 2, values 4 (t % 2) .. + 3 of that role's RoleForm.
        const int ck = threadIdx.x >> 2, cr = (threadIdx.x >> 1) & 1, ch = threadIdx.x & 1;
        double st[4];
        auto stage_load = [&](int g0) {
            const double* c = reinterpret_cast<const double*>(coef + max(g0 - ck, 0)) + 7 * cr + 4 * ch;
#pragma unroll
            for (int e = 0; e < 3; ++e) st[e] = c[e];
            st[3] = c[ch && !cr ? 11 : 3];  // the weights: w1 follows aF, w2 closes the record
        };
        auto stage_store = [&](int buf) {
            f64x2* dst = reinterpret_cast<f64x2*>(&forms[buf][ck][cr][4 * ch]);
            dst[0] = f64x2{st[0], st[1]};
            dst[1] = f64x2{ch && !cr ? -st[2] : st[2], st[3]};
        };
        auto read_form = [&](int buf, int k) {
            RoleForm r;
            const f64x2* src = reinterpret_cast<const f64x2*>(&forms[buf][k][role][0]);
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const f64x2 v = src[e];
                r.c[2 * e] = v[0];
                r.c[2 * e + 1] = v[1];
            }
            return r;
        };
        // (both before the ring's first loads, as in the steady state: the wait
        // for a chunk's coefficients must not be a wait for the ring)
        stage_load(G0);
        stage_store(0);
        stage_load(G0 - R);
        int ld = G0 * row;  // row of the next load, clamped at group 0
        int sto = ld;       // row of the step's group
#pragma unroll
        for (int k = 0; k < D; ++k) {
            fetch(k, ld);
            fetch_qb(k, ld);
            ld = max(ld - row, 0);
        }
        wave_lds_sync();
        SplitHalf<T> one, two;
        double P2 = 0.0, R2 = 0.0;  // the first half's outputs at g + 1, rounded to the state type
        char* const out = reinterpret_cast<char*>((role ? F : f) + lane);
        char* const xout = XOUT ? reinterpret_cast<char*>((role ? XF : Xf) + lane) : nullptr;
        RoleForm cn = read_form(0, 0), c2 = {};
        auto put = [](char* p, int at, T v) { *reinterpret_cast<T*>(p + static_cast<unsigned>(at)) = v; };
        // The source of a group, zero above its top (where the row is not its own).
        auto source = [](T q, bool on) { return on ? static_cast<double>(q) : 0.0; };
        // The second half at g2 (row at, coefficients c2).
        auto second = [&](int g2, int at, double P_lo, T q, auto track) {
            const double v = two.template step<SRC, STRAG>(c2, P2, R2, P_lo,
                                                           SRC ? source(q, g2 <= qb_top) : 0.0);
            const T s = static_cast<T>(v);
            put(out, at, s);
            if (decltype(track)::value && __builtin_amdgcn_ballot_w64(s != T(0)) != 0)
                top_b = max(top_b, g2);
        };
        int sto2 = sto;  // row of the second half's group
        // Above G0 (the first step's second half) the zero coefficients give
        // zeros, stored at G0's row and overwritten by the next step.
        auto step = [&](auto slot, int g, int buf, auto track) {
            constexpr int k = decltype(slot)::value;
            const RoleForm c = cn;
            cn = read_form(k + 1 < R ? buf : buf ^ 1, (k + 1) % R);
            const int at = ld;
            fetch((k + D) % RING, at);
            ld = max(at - row, 0);
            // each step's loads stay in its own issue slots, so the ring keeps
            // its depth (and its registers)
            __builtin_amdgcn_sched_barrier(0);
            const double v = one.template step<SRC, STRAG>(
                c, rF[k % RING], rf[k % RING],
                STRAG && g > 0 ? static_cast<double>(rF[(k + 1) % RING]) : 0.0,
                SRC ? source(rQa[k % RING], g <= qa_top) : 0.0);
            const T s = static_cast<T>(v);
            if (DOSE) {
                dose = fma(v, c.c[7], dose);
                psum += v;
            }
            if (decltype(track)::value && __builtin_amdgcn_ballot_w64(s != T(0)) != 0)
                top_a = max(top_a, g);
            if (XOUT) put(xout, sto, s);
            if (!PAIR) {
                put(out, sto, s);
            } else {
                const T o = swap_pair(s);
                const double Pn = role ? s : o, Rn = role ? o : s;
                second(g + 1, sto2, Pn, rQb[(k + D) % RING], track);
                fetch_qb((k + D) % RING, at);
                P2 = Pn;
                R2 = Rn;
                c2 = c;
            }
            sto2 = sto;
            sto -= row;
        };
        // at the top of a chunk (group g0 in slot 0): the next chunk's
        // coefficients into the other buffer, those after it into registers
        auto chunk = [&](int g0, int buf) {
            stage_store(buf ^ 1);
            stage_load(g0 - 2 * R);
            wave_lds_sync();
        };
        using Yes = std::true_type;
        int g0 = G0, buf = 0;
        for (; g0 >= R - 1 && (top_a < 0 || (PAIR && top_b < 0)); g0 -= R, buf ^= 1) {
            chunk(g0, buf);
            unroll<R>([&](auto k) { step(k, g0 - decltype(k)::value, buf, Yes{}); });
        }
        for (; g0 >= R - 1; g0 -= R, buf ^= 1) {
            chunk(g0, buf);
            unroll<R>([&](auto k) { step(k, g0 - decltype(k)::value, buf, std::false_type{}); });
        }
        if (g0 >= 0) {
            chunk(g0, buf);
            unroll<R>([&](auto k) {  // tail: groups g0 .. 0 (fewer than R)
                if (decltype(k)::value <= g0) step(k, g0 - decltype(k)::value, buf, Yes{});
            });
        }
        if (PAIR)  // group 0 has no lower neighbour
            second(0, 0, 0.0, SRC ? bload<T>(bb, voff, 0) : T(0), Yes{});
    }
    if (DOSE) {  // partials: dose (both roles), proxy (role 0)
        double d = live ? dose * yzw[lane / nang] : 0.0, p = live && !role ? psum : 0.0;
        for (int off = 32; off > 0; off >>= 1) {
            d += __shfl_xor(d, off);
            p += __shfl_xor(p, off);
        }
        if (threadIdx.x == 0) {
            partials[blockIdx.x] = d;
            if (proxy) partials[gridDim.x + blockIdx.x] = p;
        }
    }
    if (threadIdx.x == 0) {
        const int t = PAIR ? top_b : top_a;
        if (tops.out && t >= 0) atomicMax(tops.out, t);
        if (tops.out_x && top_a >= 0) atomicMax(tops.out_x, top_a);
    }
}

// First-order implicit upwind energy step: the reference's legacy energy
// model (energyDgCnKernel, use_legacy branch, src/energy_solver.cu:88-106)
// and its lite-memory primary step (litePrimaryEnergyStepKernel,
// src/bfpm_solver.cu:600-622, psi^1 only: f == null).  One thread per lane,
// high to low energy, in place: the old psi^1 of g+1 (straggling) is carried
// in a register and the old psi^1 of g-1 is read before it is overwritten.
// Divisions as in the reference; results flushed like the eq15 sweeps.
template <typename T, bool SRC, bool DOSE>
__global__ __launch_bounds__(kBlock) void energy_upwind_kernel(
    T* __restrict__ F, T* __restrict__ f, const UpwindCoef* __restrict__ uc,
    const EnergyCoef* __restrict__ coef, const T* __restrict__ Q1, int Ng, int lanes,
    const double* __restrict__ yzw, int nang, double* __restrict__ partials, int proxy,
    int straggling, SweepTops tops) {
    __shared__ double lds[kBlock / 64];
    __shared__ int ldi[kBlock / 64];
    const int lane = blockIdx.x * kBlock + threadIdx.x;
    reset_tops(tops);
    const int q_top = SRC ? source_top(tops, tops.xa, Ng) : -1;
    const int G0 = min(Ng - 1, max(state_top(tops, Ng), q_top) + (straggling ? 1 : 0));
    int top = -1;
    double acc_dose = 0.0, acc_proxy = 0.0;
    if (lane < lanes && G0 >= 0) {
        double next_F = 0.0, next_f = 0.0, dose = 0.0;
        double F_hi = 0.0;  // old psi^1 at g+1 (zero above G0)
        double Fg = static_cast<double>(F[static_cast<long long>(G0) * lanes + lane]);
        for (int g = G0; g >= 0; --g) {
            const long long idx = static_cast<long long>(g) * lanes + lane;
            const double F_lo = g > 0 ? static_cast<double>(F[idx - lanes]) : 0.0;
            const double fg = f ? static_cast<double>(f[idx]) : 0.0;
            const UpwindCoef c = uc[g];
            const double src = (SRC && g <= q_top) ? static_cast<double>(Q1[idx]) : 0.0;
            double Fv = (fmax(Fg, 0.0) / c.h + c.c_hi * next_F + src) / c.denom;
            double fv = (fg / c.h + c.c_hi * next_f) / c.denom;
            if (c.strag > 0.0) {
                const double lap = fmax(F_hi, 0.0) - 2.0 * fmax(Fg, 0.0) + fmax(F_lo, 0.0);
                Fv += c.strag * lap;
            }
            const T sF = static_cast<T>(flush_tiny<T>(fmax(Fv, 0.0)));
            const T sf = static_cast<T>(flush_tiny<T>(fmax(fv, 0.0)));
            F[idx] = sF;
            if (f) f[idx] = sf;
            next_F = static_cast<double>(sF);
            next_f = static_cast<double>(sf);
            top = max(top, (sF != T(0) || sf != T(0)) ? g : -1);
            if (DOSE) {
                dose = add_dose(dose, next_F, next_f, coef[g].w1, coef[g].w2);
                acc_proxy += next_f;
            }
            F_hi = Fg;
            Fg = F_lo;
        }
        if (DOSE) acc_dose = dose * yzw[lane / nang];
    }
    if (DOSE) {
        const double d = block_sum(acc_dose, lds);
        if (threadIdx.x == 0) partials[blockIdx.x] = d;
        if (proxy) {
            const double p = block_sum(acc_proxy, lds);
            if (threadIdx.x == 0) partials[gridDim.x + blockIdx.x] = p;
        }
    }
    if (tops.out) publish_top(top, tops.out, tops.out_x, ldi);
}

template <typename T, int LPT, bool SRC, bool STRAG>
void dispatch_pair(T* F, T* f, const EnergyCoef* coef, const T* Qa, const T* Qb, T* XF, T* Xf,
                   const unsigned* xmask, int Ng, long long lanes, const double* yzw, int nang,
                   double* partials, bool proxy, hipStream_t s, const SweepTops& tops) {
    const int blocks = energy_blocks(lanes, Ng, sizeof(T));
    BFPN_REQUIRE(lanes < (1LL << 31), "energy sweep indexes lanes with 32-bit offsets");
    if (XF)
        hipLaunchKernelGGL((energy_pair_kernel<T, LPT, SRC, STRAG, true>), dim3(blocks),
                           dim3(kBlock), 0, s, F, f, coef, Qa, Qb, XF, Xf, xmask, Ng,
                           static_cast<int>(lanes), yzw, nang, partials, proxy ? 1 : 0, tops);
    else
        hipLaunchKernelGGL((energy_pair_kernel<T, LPT, SRC, STRAG, false>), dim3(blocks),
                           dim3(kBlock), 0, s, F, f, coef, Qa, Qb, XF, Xf, xmask, Ng,
                           static_cast<int>(lanes), yzw, nang, partials, proxy ? 1 : 0, tops);
}

template <typename T, bool SRC, bool STRAG>
void dispatch_pair_lpt(T* F, T* f, const EnergyCoef* coef, const T* Qa, const T* Qb, T* XF,
                       T* Xf, const unsigned* xmask, int Ng, long long lanes, const double* yzw,
                       int nang, double* partials, bool proxy, hipStream_t s,
                       const SweepTops& tops) {
    if (energy_split(lanes, Ng, sizeof(T))) {
        const dim3 grid(energy_blocks(lanes, Ng, sizeof(T)));
        if (XF)
            hipLaunchKernelGGL((energy_split_kernel<T, true, SRC, STRAG, true, true>), grid,
                               dim3(64), 0, s, F, f, coef, Qa, Qb, XF, Xf, Ng,
                               static_cast<int>(lanes), yzw, nang, partials, proxy ? 1 : 0, tops);
        else
            hipLaunchKernelGGL((energy_split_kernel<T, true, SRC, STRAG, true, false>), grid,
                               dim3(64), 0, s, F, f, coef, Qa, Qb, XF, Xf, Ng,
                               static_cast<int>(lanes), yzw, nang, partials, proxy ? 1 : 0, tops);
        return;
    }
    if constexpr (sizeof(T) == 4) {
        const int lpt = lanes_per_thread(lanes, sizeof(T));
        if (lpt == 4)
            return dispatch_pair<T, 4, SRC, STRAG>(F, f, coef, Qa, Qb, XF, Xf, xmask, Ng, lanes,
                                                   yzw, nang, partials, proxy, s, tops);
    }
    dispatch_pair<T, 1, SRC, STRAG>(F, f, coef, Qa, Qb, XF, Xf, xmask, Ng, lanes, yzw, nang,
                                    partials, proxy, s, tops);
}

template <typename T, int LPT, bool SRC, bool STRAG>
void dispatch_dose(T* F, T* f, const EnergyCoef* coef, const T* Q1, int Ng, long long lanes,
                   const double* yzw, int nang, double* partials, bool proxy, hipStream_t s,
                   const SweepTops& tops) {
    const int blocks = energy_blocks(lanes, Ng, sizeof(T));
    BFPN_REQUIRE(lanes < (1LL << 31), "energy sweep indexes lanes with 32-bit offsets");
    if (partials)
        hipLaunchKernelGGL((energy_half_kernel<T, LPT, SRC, STRAG, true>), dim3(blocks),
                           dim3(kBlock), 0, s, F, f, coef, Q1, Ng, static_cast<int>(lanes), yzw,
                           nang, partials, proxy ? 1 : 0, tops);
    else
        hipLaunchKernelGGL((energy_half_kernel<T, LPT, SRC, STRAG, false>), dim3(blocks),
                           dim3(kBlock), 0, s, F, f, coef, Q1, Ng, static_cast<int>(lanes), yzw,
                           nang, partials, 0, tops);
}

template <typename T, bool SRC, bool STRAG>
void dispatch_lpt(T* F, T* f, const EnergyCoef* coef, const T* Q1, int Ng, long long lanes,
                  const double* yzw, int nang, double* partials, bool proxy, hipStream_t s,
                  const SweepTops& tops) {
    if (energy_split(lanes, Ng, sizeof(T), partials != nullptr)) {
        const dim3 grid(static_cast<unsigned>((lanes + 31) / 32));
        T* const none = nullptr;
        if (partials)
            hipLaunchKernelGGL((energy_split_kernel<T, false, SRC, STRAG, true, false>), grid,
                               dim3(64), 0, s, F, f, coef, Q1, none, none, none, Ng,
                               static_cast<int>(lanes), yzw, nang, partials, proxy ? 1 : 0, tops);
        else
            hipLaunchKernelGGL((energy_split_kernel<T, false, SRC, STRAG, false, false>), grid,
                               dim3(64), 0, s, F, f, coef, Q1, none, none, none, Ng,
                               static_cast<int>(lanes), yzw, nang, partials, 0, tops);
        return;
    }
    if constexpr (sizeof(T) == 4) {
        const int lpt = lanes_per_thread(lanes, sizeof(T));
        if (lpt == 4)
            return dispatch_dose<T, 4, SRC, STRAG>(F, f, coef, Q1, Ng, lanes, yzw, nang, partials,
                                                   proxy, s, tops);
    }
    dispatch_dose<T, 1, SRC, STRAG>(F, f, coef, Q1, Ng, lanes, yzw, nang, partials, proxy, s, tops);
}

}  // namespace

int energy_blocks(long long lanes, int Ng, size_t elem) {
    if (energy_split(lanes, Ng, elem)) return static_cast<int>((lanes + 31) / 32);
    const long long per_block = static_cast<long long>(kBlock) * lanes_per_thread(lanes, elem);
    return static_cast<int>((lanes + per_block - 1) / per_block);
}

template <typename T>
void launch_energy_half(T* F, T* f, const EnergyCoef* coef, const T* Q1, int Ng, long long lanes,
                        bool straggling, const double* yz_weight, int nang, double* dose_partials,
                        bool proxy, hipStream_t s, const SweepTops& tops) {
    if (lanes <= 0 || Ng <= 0) return;
    if (Q1) {
        if (straggling)
            dispatch_lpt<T, true, true>(F, f, coef, Q1, Ng, lanes, yz_weight, nang, dose_partials,
                                         proxy, s, tops);
        else
            dispatch_lpt<T, true, false>(F, f, coef, Q1, Ng, lanes, yz_weight, nang, dose_partials,
                                          proxy, s, tops);
    } else {
        if (straggling)
            dispatch_lpt<T, false, true>(F, f, coef, Q1, Ng, lanes, yz_weight, nang, dose_partials,
                                          proxy, s, tops);
        else
            dispatch_lpt<T, false, false>(F, f, coef, Q1, Ng, lanes, yz_weight, nang,
                                           dose_partials, proxy, s, tops);
    }
    BFPN_HIP(hipGetLastError());
}

template <typename T>
void launch_energy_pair(T* F, T* f, const EnergyCoef* coef, const T* Qa, const T* Qb, int Ng,
                        long long lanes, bool straggling, const double* yz_weight, int nang,
                        double* dose_partials, bool proxy, T* XF, T* Xf, hipStream_t s,
                        const SweepTops& tops, const unsigned* xmask) {
    if (lanes <= 0 || Ng <= 0) return;
    BFPN_REQUIRE(dose_partials, "the paired energy sweep needs dose partials");
    BFPN_REQUIRE((Qa != nullptr) == (Qb != nullptr), "both half steps need a source, or neither");
    BFPN_REQUIRE((XF != nullptr) == (Xf != nullptr), "the intermediate state needs both arrays");
    const auto run = [&](auto src, auto strag) {
        dispatch_pair_lpt<T, decltype(src)::value, decltype(strag)::value>(
            F, f, coef, Qa, Qb, XF, Xf, xmask, Ng, lanes, yz_weight, nang, dose_partials, proxy,
            s, tops);
    };
    using Y = std::true_type;
    using N = std::false_type;
    if (Qa) {
        if (straggling) run(Y{}, Y{});
        else run(Y{}, N{});
    } else {
        if (straggling) run(N{}, Y{});
        else run(N{}, N{});
    }
    BFPN_HIP(hipGetLastError());
}

template <typename T>
void launch_energy_upwind(T* F, T* f, const UpwindCoef* uc, const EnergyCoef* coef, const T* Q1,
                          int Ng, long long lanes, bool straggling, const double* yz_weight,
                          int nang, double* dose_partials, bool proxy, hipStream_t s,
                          const SweepTops& tops) {
    if (lanes <= 0 || Ng <= 0) return;
    BFPN_REQUIRE(lanes < (1LL << 31), "energy sweep indexes lanes with 32-bit offsets");
    const int blocks = static_cast<int>((lanes + kBlock - 1) / kBlock);
    const int st = straggling ? 1 : 0, px = proxy ? 1 : 0;
    const int n = static_cast<int>(lanes);
    if (Q1 && dose_partials)
        hipLaunchKernelGGL((energy_upwind_kernel<T, true, true>), dim3(blocks), dim3(kBlock), 0, s,
                           F, f, uc, coef, Q1, Ng, n, yz_weight, nang, dose_partials, px, st, tops);
    else if (Q1)
        hipLaunchKernelGGL((energy_upwind_kernel<T, true, false>), dim3(blocks), dim3(kBlock), 0, s,
                           F, f, uc, coef, Q1, Ng, n, yz_weight, nang, dose_partials, 0, st, tops);
    else if (dose_partials)
        hipLaunchKernelGGL((energy_upwind_kernel<T, false, true>), dim3(blocks), dim3(kBlock), 0, s,
                           F, f, uc, coef, Q1, Ng, n, yz_weight, nang, dose_partials, px, st, tops);
    else
        hipLaunchKernelGGL((energy_upwind_kernel<T, false, false>), dim3(blocks), dim3(kBlock), 0,
                           s, F, f, uc, coef, Q1, Ng, n, yz_weight, nang, dose_partials, 0, st,
                           tops);
    BFPN_HIP(hipGetLastError());
}

template void launch_energy_upwind<float>(float*, float*, const UpwindCoef*, const EnergyCoef*,
                                          const float*, int, long long, bool, const double*, int,
                                          double*, bool, hipStream_t, const SweepTops&);
template void launch_energy_upwind<double>(double*, double*, const UpwindCoef*, const EnergyCoef*,
                                           const double*, int, long long, bool, const double*, int,
                                           double*, bool, hipStream_t, const SweepTops&);

template void launch_energy_pair<float>(float*, float*, const EnergyCoef*, const float*,
                                        const float*, int, long long, bool, const double*, int,
                                        double*, bool, float*, float*, hipStream_t,
                                        const SweepTops&, const unsigned*);
template void launch_energy_pair<double>(double*, double*, const EnergyCoef*, const double*,
                                         const double*, int, long long, bool, const double*, int,
                                         double*, bool, double*, double*, hipStream_t,
                                         const SweepTops&, const unsigned*);

template void launch_energy_half<float>(float*, float*, const EnergyCoef*, const float*, int,
                                        long long, bool, const double*, int, double*, bool,
                                        hipStream_t, const SweepTops&);
template void launch_energy_half<double>(double*, double*, const EnergyCoef*, const double*, int,
                                         long long, bool, const double*, int, double*, bool,
                                         hipStream_t, const SweepTops&);

}  // namespace bfpn
