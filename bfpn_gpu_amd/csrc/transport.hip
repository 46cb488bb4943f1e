// transport.hip — explicit MUSCL predictor-corrector y/z transport (Eq.18).
//
// Reference: muscl_paper_slope, spatial_flux_divergence_value and the
// flux / predictor / corrector kernels of SpatialTransportSolver::solveEq18
// (src/spatial_transport.cu:23-161, 202-262): four launches and three
// scratch arrays per call, three limited slopes per axis and cell, a division
// per slope.
//
// MI355X design: one launch, in place, each value read once and written once.
//  * A work-group owns one energy group g and MW consecutive directions m
//    (the contiguous axis) for the whole (y, z) plane, so no other work-group
//    reads or writes its data and the update can be written in place.
//  * Threads own P adjacent y columns and march along z.  The z windows of
//    psi and psi* stay in registers, and the limited z slopes are carried from
//    row to row, so each row costs one new z slope per stage.  y neighbours
//    come from LDS rings of two rows each of psi, psi* and their y slopes.  Step
//    t forms L(psi) and psi* = clip(psi - h L psi) on row t and writes row t-2:
//    clip(psi - h/2 (L psi + L psi*)).  One barrier per z step.
//  * The flow direction is fixed per lane, so only the upwind reconstruction
//    is formed: per stage one limited slope per axis and cell.
//  * The superbee slope is evaluated without a division:
//      a = R - C, b = C - L, ab > 0 and |a| >= 1e-10:
//      slope = sign(a) min(max(|a|, |b|), 2 min(|a|, |b|)),   else 0,
//    which equals forward * max(0, min(2 theta, 1), min(theta, 2)) with
//    theta = b / a, up to the rounding of that quotient; it is computed as
//    two signed medians of three (one instruction each in FP32).
//  * Rows and columns outside the plane are clamped, exactly like the
//    reference's clamped stencil taps: the slope of a boundary cell is 0 and
//    the cell outside reads the boundary value with slope 0.

#include "buffer.hpp"
#include "kernels.hpp"

#include <type_traits>

namespace bfpn {
namespace {

// Work-group size limit: 1024 threads in FP32; 768 in FP64, so that a
// thread may hold up to 168 VGPRs (its windows are twice as wide).
template <typename T>
constexpr int max_threads() { return sizeof(T) == 4 ? 1024 : 768; }

// Waves per SIMD that the registers have to allow.
template <typename T, int P>
constexpr int waves_per_simd() {
    return sizeof(T) == 4 ? (P == 1 ? 8 : P == 2 ? 5 : 4) : (P == 1 ? 4 : 3);
}

// Step t loads row t + this: rows t + 3 .. are in flight.  An XCD's work-groups
// hold that many rows of their planes in its 4 MB L2, and neighbouring chunks of
// directions share lines there: four steps of a whole 81 x 81 x 400 x 500 FP32
// march take 198.4 ms with seven rows ahead, 197.8 with six, 197.4 with five and
// 197.2 with four; FP64 planes of 33 to 48 columns 5 % less with four than with
// seven.  Seven hides the latency of short marches better (2 %) where one FP32
// column a thread leaves the lines few.
template <typename T, int P>
constexpr int rows_ahead() { return sizeof(T) == 4 && P == 1 ? 7 : 4; }

// LDS slots of MW values per y column (two rows each of psi, psi* and their
// y slopes), and the distance of
// two columns: chosen so that the P columns a thread steps over amount to MW
// values modulo the banks (P = 1, 2; an odd multiple of MW for P = 3), so the
// columns that one wave reads fall on distinct banks.
constexpr int kSlots = 8;
template <int MW, int P>
constexpr int column_pitch() { return kSlots * MW + (P == 2 ? MW / 2 : MW); }

// Superbee slope of two differences (either order), without the 1e-10 test:
//   ab > 0: sign(a) min(max(|a|, |b|), 2 min(|a|, |b|)),  else 0,
// which is the median of a, b and 2 m, with m = median(a, b, 0) the minmod
// of a and b: m = 0 when the signs differ (then the median is 0 too), and for
// a common sign the median of a, b, 2m is the expression above.  One
// median-of-three instruction each in FP32; FP64 uses
// median(x, y, z) = max(min(x, y), min(max(x, y), z)).
__device__ inline float superbee(float a, float b) {
    const float m = __builtin_amdgcn_fmed3f(a, b, 0.0f);
    return __builtin_amdgcn_fmed3f(a, b, 2.0f * m);
}
__device__ inline double superbee(double a, double b) {
    const double lo = fmin(a, b), hi = fmax(a, b);
    const double m = fmax(lo, fmin(hi, 0.0));
    return fmax(lo, fmin(hi, 2.0 * m));
}

// a: forward, b: backward difference (physical orientation); 0 when the
// forward difference is below 1e-10.
template <typename T>
__device__ inline T limited_slope(T a, T b) {
    return fabs(a) < T(1e-10) ? T(0) : superbee(a, b);
}

// Flux divergence at one cell, per axis written in the lane's upwind frame:
//   w (F(+1/2) - F(-1/2)) / d = (|w| / d) (downwind face - upwind face),
// where the downwind face is the cell's own reconstruction c + s_down/2 and
// the upwind face the upwind neighbour's, n + s_up/2.  The upwind frame's
// slopes are +-S of the physical limited slopes S (superbee is odd and
// symmetric, and the 1e-10 test goes to the physical forward difference
// either way).
//  y: (c - n) + hy (S_c - S_n), hy = +-1/2 the sign of wy; the physical slope
//     is formed once per cell and published in LDS for the downwind neighbour.
//  z: (c - n) + hz (S_c - S_n) from the row window.  For wz < 0 that is the
//     negation of the next row's value for wz >= 0, so the march forms
//     U = fma(hz, S(r) - S(r - 1), c(r) - c(r - 1)) once per row r and takes
//     U(row) or -U(row + 1).
//
// grid: (direction chunks x groups, XCD-swizzled), block: MW directions times
// the y columns, P adjacent columns y = ry P + j per thread, so that inner
// differences are shared and only the outer neighbours come from LDS.
//
// Step t commits psi row t+1 to LDS; after its one barrier it forms the y
// slopes of psi row t+1 and of psi* row t-1 (for the next step), psi* of row t
// (predictor) and the result of row t-2 (corrector).  Every ring has two rows:
// a slot is rewritten one barrier after its last reader.
//
// The z march is unrolled by 8: the psi window and the rows in flight share
// one register ring indexed by row mod 8 (row t+4 or t+7 is loaded into a slot
// that step t no longer reads), so sliding a window is a renaming
// rather than a chain of moves and a loaded row is never copied (a copy would
// wait for the load).  Rows past Nz are loaded as copies of row Nz: with them,
// and with zero slopes carried into rows 0, the clamped stencil at both ends
// needs no selects.  The first four steps (Start) and the last ones (End)
// leave out the halves that have no row to work on; those tests are uniform.
//
// A corrector adds its two axes' terms in one order in the blocks of eight steps
// that start 13 or more rows before Nz and the other way round elsewhere (at
// t = 2, 3, and from Upper on): a choice without meaning that keeps values what
// they have been.
//
// What bounds it: vector issue and HBM together (47 vector instructions, 8
// bytes per cell).  Against a march with four-row rings in LDS (12 LDS
// accesses per cell instead of 10) whose edge steps did all of their work, one
// kernel at a time, FP32: 9 x 9 nodes x 49 directions x 500 groups 9.8 -> 8.6
// us, 11 x 11 x 121 x 500 24.0 -> 17.0, 13 x 13 x 81 x 500 26.6 -> 16.8, 21 x 21
// x 400 x 500 214 -> 195 (3.6 TB/s), 81 x 81 x 400 x 500 2478 -> 2358 (4.5 TB/s);
// FP64: 21 x 21 x 400 x 250 227 -> 154, 41 x 41 x 400 x 60 185 -> 164, 81 x 41 x
// 400 x 60 929 -> 327, 97 x 41 x 400 x 60 1497 -> 749.
enum class Part { Start, Inner, Upper, EndLoad, End };

template <typename T, int MW, int P, bool CLIP>
__device__ __forceinline__ void transport_march(T* __restrict__ F, const T* __restrict__ omend,
                                                int Ny, int Nz, int nang, T inv_dy, T inv_dz, T h,
                                                int tiles, const int* __restrict__ top) {
    extern __shared__ unsigned char lds_raw[];
    const int mchunks = (nang + MW - 1) / MW;
    // Only the groups up to the state's top hold nonzero values (the others
    // stay zero); their tiles are the first `active` and the grid's later
    // blocks exit at once.  Blocks are dispatched round-robin over the 8
    // XCDs.  Direction chunks of one group share 128-byte lines (a plane row
    // is nang floats), so the chunks of a group run consecutively on one XCD
    // and share its L2: block b -> logical tile (b mod 8) * (n8 / 8) + b / 8,
    // n8 = active rounded up to a multiple of 8.
    const int active = top ? min(tiles, (min(*top, tiles / mchunks - 1) + 1) * mchunks) : tiles;
    const int n8 = (active + 7) & ~7;
    if (static_cast<int>(blockIdx.x) >= n8) return;
    const int L = (blockIdx.x & 7) * (n8 >> 3) + (blockIdx.x >> 3);
    if (L >= active) return;
    const int g = L / mchunks;
    T* ring = reinterpret_cast<T*>(lds_raw);
    constexpr int YP = column_pitch<MW, P>(), A = rows_ahead<T, P>();
    constexpr int kPsi = 0, kPred = 2, kS = 4, kSPred = 6;  // first slot of each ring

    // A thread whose columns would pass Ny takes the last P instead: the ones
    // it shares with its neighbour get the same values from both.
    const int mm = threadIdx.x % MW, first = threadIdx.x / MW * P;
    const int y0 = min(first, Ny + 1 - P);
    const int m0 = (L - g * mchunks) * MW;
    const bool live = m0 + mm < nang;
    // Lanes past the last direction compute a copy of the last one from
    // in-bounds addresses, so loads and arithmetic need no predicate; the
    // global stores of all copies go to an offset past the end of the buffer
    // resource, which the hardware's range check drops.
    const int m = live ? m0 + mm : nang - 1;
    const T wy = omend[2 * m], wz = omend[2 * m + 1];
    const bool py = wy >= T(0), pz = wz >= T(0);
    const T cy = fabs(wy) * inv_dy, cz = fabs(wz) * inv_dz;
    const T hy = py ? T(0.5) : T(-0.5), hz = pz ? T(0.5) : T(-0.5);
    const T hh = T(0.5) * h;
    const long long zstride = static_cast<long long>(Ny + 1) * nang;
    const unsigned zbytes = static_cast<unsigned>(zstride * sizeof(T));  // one z row
    // the group's block from direction m0 on, as a buffer resource: uniform
    // row offsets, 32-bit lane offsets
    const __amdgpu_buffer_rsrc_t Fg =
        make_rsrc(F + static_cast<long long>(g) * zstride * (Nz + 1) + m0,
                   static_cast<unsigned>((zstride * (Nz + 1) - m0) * sizeof(T)));

    unsigned boff[P];  // byte offset of the lane's column in a plane row
    unsigned soff[P];  // the same for stores; kOutside (dropped) for copies
    T* const own = ring + y0 * YP + mm;  // LDS: the thread's first column,
    const T *left, *right, *near[P];     // the ones beside it, the upwind ones (clamped)
    T win[P][8];    // psi rows t .. t+2, then rows t+3 .. t+A in flight (row mod 8)
    T wpred[P][4];  // psi*, rows t-2 .. t after the predictor of step t (row mod 4)
    T wbase[P][4];  // psi - h/2 L(psi), the same rows
    T sy[P][2], dn[P][2];    // y slope and c - (upwind neighbour) of psi rows t, t+1
    T syp[P][2], dnp[P][2];  // the same of psi* rows t-2, t-1
    T sz[P], szp[P];  // z slopes of psi row t and psi* row t-2 before step t
    T uz[P], uzp[P];  // U of the same rows
    {
        auto column = [&](int y) { return ring + min(max(y, 0), Ny) * YP + mm; };
        left = column(y0 - 1);
        right = column(y0 + P);
#pragma unroll
        for (int j = 0; j < P; ++j) {
            const int y = y0 + j;
            boff[j] = static_cast<unsigned>((y * nang + (m - m0)) * sizeof(T));
            soff[j] = (y >= first && live) ? boff[j] : kOutside;
            near[j] = column(py ? y - 1 : y + 1);
#pragma unroll
            for (int r = 0; r < A; ++r)
                win[j][r] = bload<T>(Fg, boff[j], static_cast<unsigned>(min(r, Nz)) * zbytes);
            sz[j] = szp[j] = uz[j] = uzp[j] = T(0);
        }
    }
    // y slopes S of a row from its values c and the outer neighbours, into
    // registers and LDS slot `slot`, and the differences D to the upwind
    // neighbours.
    auto slopes = [&](const T (&c)[P], T l, T r, T (&S)[P], T (&D)[P], int slot) {
        T d[P + 1];
        d[0] = c[0] - l;
#pragma unroll
        for (int j = 1; j < P; ++j) d[j] = c[j] - c[j - 1];
        d[P] = r - c[P - 1];
#pragma unroll
        for (int j = 0; j < P; ++j) {
            S[j] = limited_slope(d[j + 1], d[j]);
            D[j] = py ? d[j] : -d[j + 1];
            own[j * YP + slot * MW] = S[j];
        }
    };
    {
#pragma unroll
        for (int j = 0; j < P; ++j) own[j * YP + kPsi * MW] = win[j][0];
        __syncthreads();
        T c[P], S[P], D[P];
#pragma unroll
        for (int j = 0; j < P; ++j) c[j] = win[j][0];
        slopes(c, left[kPsi * MW], right[kPsi * MW], S, D, kS);
#pragma unroll
        for (int j = 0; j < P; ++j) {
            sy[j][0] = S[j];
            dn[j][0] = D[j];
        }
    }

    auto step = [&](int t, auto phase, auto part) {
        constexpr int k8 = decltype(phase)::value;  // t mod 8
        constexpr int k2 = k8 & 1, k4 = k8 & 3;
        constexpr Part S = decltype(part)::value;
        constexpr bool E = S == Part::End || S == Part::EndLoad;
        if (E && t > Nz + 2) return;
        const bool do_slope = !E || t + 1 <= Nz;
        const bool do_pred = !E || t <= Nz;
        const bool do_slopep = S == Part::Start ? k8 >= 1 : !E || t <= Nz + 1;
        const bool do_corr = S != Part::Start || k8 >= 2;
        if (do_slope)
#pragma unroll
            for (int j = 0; j < P; ++j) own[j * YP + (kPsi + (k2 ^ 1)) * MW] = win[j][(k8 + 1) & 7];
        __syncthreads();
        // Keep each step's arithmetic after its barrier: moved earlier, the z
        // differences of later rows would wait for rows still in flight.
        __builtin_amdgcn_sched_barrier(0);
        if (S != Part::End) {  // row t + A into a free register slot
            const unsigned so = static_cast<unsigned>(min(t + A, Nz)) * zbytes;
#pragma unroll
            for (int j = 0; j < P; ++j) win[j][(k8 + A) & 7] = bload<T>(Fg, boff[j], so);
        }
        // LDS reads of the step, issued together
        T al = T(0), ar = T(0), bl = T(0), br = T(0), en[P], cn[P];
        if (do_slope) {
            al = left[(kPsi + (k2 ^ 1)) * MW];
            ar = right[(kPsi + (k2 ^ 1)) * MW];
        }
        if (do_slopep) {
            bl = left[(kPred + (k2 ^ 1)) * MW];
            br = right[(kPred + (k2 ^ 1)) * MW];
        }
#pragma unroll
        for (int j = 0; j < P; ++j) {
            en[j] = do_pred ? near[j][(kS + k2) * MW] : T(0);
            cn[j] = do_corr ? near[j][(kSPred + k2) * MW] : T(0);
        }
        if (do_slope) {  // y slopes of psi row t+1
            T c[P], S[P], D[P];
#pragma unroll
            for (int j = 0; j < P; ++j) c[j] = win[j][(k8 + 1) & 7];
            slopes(c, al, ar, S, D, kS + (k2 ^ 1));
#pragma unroll
            for (int j = 0; j < P; ++j) {
                sy[j][k2 ^ 1] = S[j];
                dn[j][k2 ^ 1] = D[j];
            }
        }
        if (do_slopep) {  // y slopes of psi* row t-1
            T c[P], S[P], D[P];
#pragma unroll
            for (int j = 0; j < P; ++j) c[j] = wpred[j][(k4 + 3) & 3];
            slopes(c, bl, br, S, D, kSPred + (k2 ^ 1));
#pragma unroll
            for (int j = 0; j < P; ++j) {
                syp[j][k2 ^ 1] = S[j];
                dnp[j][k2 ^ 1] = D[j];
            }
        }
        if (do_pred) {  // predictor on row t
#pragma unroll
            for (int j = 0; j < P; ++j) {
                const T c = win[j][k8], up = win[j][(k8 + 1) & 7];
                const T dz = up - c;
                const T s = limited_slope(win[j][(k8 + 2) & 7] - up, dz);
                const T un = fma(hz, s - sz[j], dz);  // U of row t+1
                const T fy = fma(hy, sy[j][k2] - en[j], dn[j][k2]), fz = pz ? uz[j] : -un;
                const T L0 = fma(cy, fy, cz * fz);
                sz[j] = s;
                uz[j] = un;
                T v = c - h * L0;
                if (CLIP) v = fmax(v, T(0));
                wbase[j][k4] = c - hh * L0;
                // rows past Nz: copies of row Nz
                wpred[j][k4] = S == Part::Start && k8 >= 2 && t > Nz ? wpred[j][(k4 + 3) & 3] : v;
                own[j * YP + (kPred + k2) * MW] = v;
            }
        } else {
#pragma unroll
            for (int j = 0; j < P; ++j) wpred[j][k4] = wpred[j][(k4 + 3) & 3];  // past Nz: row Nz
        }
        if (do_corr) {  // corrector on row t-2, written in place
            const unsigned so = static_cast<unsigned>(t - 2) * zbytes;
#pragma unroll
            for (int j = 0; j < P; ++j) {
                const T c = wpred[j][(k4 + 2) & 3], up = wpred[j][(k4 + 3) & 3];
                const T dz = up - c;
                const T s = limited_slope(wpred[j][k4] - up, dz);
                const T un = fma(hz, s - szp[j], dz);  // U of row t-1
                const T fy = fma(hy, syp[j][k2] - cn[j], dnp[j][k2]), fz = pz ? uzp[j] : -un;
                const T L1 = S == Part::Inner ? fma(cy, fy, cz * fz) : fma(cz, fz, cy * fy);
                szp[j] = s;
                uzp[j] = un;
                T v = wbase[j][(k4 + 2) & 3] - hh * L1;
                if (CLIP) v = fmax(v, T(0));
                bstore(v, Fg, soff[j], so);
            }
        }
    };
    // four steps from t0, t0 mod 8 = B
    auto block = [&](int t0, auto base, auto part) {
        constexpr int B = decltype(base)::value;
        step(t0, std::integral_constant<int, B>{}, part);
        step(t0 + 1, std::integral_constant<int, B + 1>{}, part);
        step(t0 + 2, std::integral_constant<int, B + 2>{}, part);
        step(t0 + 3, std::integral_constant<int, B + 3>{}, part);
    };
    using I0 = std::integral_constant<int, 0>;
    using I4 = std::integral_constant<int, 4>;
    using Start = std::integral_constant<Part, Part::Start>;
    using Inner = std::integral_constant<Part, Part::Inner>;
    using Upper = std::integral_constant<Part, Part::Upper>;
    using EndLoad = std::integral_constant<Part, Part::EndLoad>;
    using End = std::integral_constant<Part, Part::End>;
    // One straight path: alternatives for the last blocks that join again cost
    // 20 to 40 registers.
    block(0, I0{}, Start{});
    int t0 = 4;
    for (; t0 + 13 <= Nz; t0 += 8) {
        block(t0, I4{}, Inner{});
        block(t0 + 4, I0{}, Inner{});
    }
    for (; t0 + 8 <= Nz; t0 += 8) {  // (at most once)
        block(t0, I4{}, Upper{});
        block(t0 + 4, I0{}, Upper{});
    }
    // at most 10 steps are left, and rows up to Nz + 2 <= t0 + 9 to load
    block(t0, I4{}, EndLoad{});
    block(t0 + 4, I0{}, std::conditional_t<(A < 6), EndLoad, End>{});
    step(t0 + 8, I4{}, End{});
    step(t0 + 9, std::integral_constant<int, 5>{}, End{});
}

// Which arrays a launch marches and how: one with or without the clip, or a
// species' two in one launch (blockIdx.y): psi^1 with or without, psi^2 without.
enum class Arrays { Clipped, Signed, ClippedSigned, SignedSigned };

template <typename T, int MW, int P, Arrays A>
__global__ __launch_bounds__(max_threads<T>())
__attribute__((amdgpu_waves_per_eu(waves_per_simd<T, P>()))) void transport_march_kernel(
    T* __restrict__ F, T* __restrict__ f, const T* __restrict__ omend, int Ny, int Nz, int nang,
    T inv_dy, T inv_dz, T h, int tiles, const int* __restrict__ top) {
    if constexpr (A == Arrays::Clipped) {
        transport_march<T, MW, P, true>(F, omend, Ny, Nz, nang, inv_dy, inv_dz, h, tiles, top);
    } else if constexpr (A == Arrays::ClippedSigned) {
        if (blockIdx.y == 0)
            transport_march<T, MW, P, true>(F, omend, Ny, Nz, nang, inv_dy, inv_dz, h, tiles, top);
        else
            transport_march<T, MW, P, false>(f, omend, Ny, Nz, nang, inv_dy, inv_dz, h, tiles, top);
    } else {
        T* const X = A == Arrays::SignedSigned && blockIdx.y ? f : F;
        transport_march<T, MW, P, false>(X, omend, Ny, Nz, nang, inv_dy, inv_dz, h, tiles, top);
    }
}

struct MarchShape {
    int MW, P, threads;
};

// Launch shape of `Ng` planes of Ny1 columns and nang directions.
//
// FP32: 16 directions (64-byte row segments) and one column per thread up to 64
// columns.  From there on to 96 columns 32 directions, whole cache lines, and
// three columns: four steps of a whole march at 81 x 81 nodes x 400 directions x
// 500 groups 197.2 ms against 198.9 with (16, 2), and 203.4 with that and seven
// rows ahead, where the clipped kernel's two work-groups per CU read 7.4 GB a
// launch for a state of 5.2, 5.6 here; alone, 81 x 21 x 121 x 500 203 against 261
// us, 65 x 41 x 400 x 300 572 against 685.  A CU holds one such
// work-group, so where their last round would leave much of the chip idle (81 x
// 81 x 400 x 60, 780 of them: 327 against 300 us; 81 x 81 x 81 x 120, 360: 144
// against 113) the smaller ones of (16, 2) are kept.  More columns per thread
// than needed share more differences but leave fewer waves per SIMD: two cost
// 18.8 against 17.0 us at 13 x 13 x 81 x 500.  8 directions are 32-byte segments
// (254 against 195 us at 21 x 21 x 400 x 500): for the widest planes.
//
// FP64: a thread's windows allow four waves per SIMD, so what counts is how
// many work-groups that leaves per CU: 16 / waves up to four waves, beyond that
// 4 / (waves on its fullest SIMD).  24 directions at 21 columns (two work-groups
// of 8 waves), 158 us for 400 x 250, against 200 with 16 (two of 6) and 170 with
// 8; but at 13 columns (two of 5 waves against four of 4) 162 against 128 us
// x 500.  8 directions, half lines, need the other half's work-group near: up to
// 28 columns, or 36 where a group has few chunks (31 x 31 x 81 x 500 190 against
// 162 us with 16, but 49 directions 84 against 101), and 49 columns and more,
// where 16 do not fit.  Their cost counts 6 % more.  Planes above 96 columns take
// two columns per thread.
MarchShape march_shape(int Ny1, int nang, int Ng, size_t elem) {
    auto threads_of = [&](int MW, int P) { return (MW * ((Ny1 + P - 1) / P) + 63) / 64 * 64; };
    auto tiles_of = [&](int MW) { return static_cast<long long>((nang + MW - 1) / MW) * Ng; };
    MarchShape best{0, 0, 0};
    if (elem == 8) {
        double least = 0.0;
        for (const int MW : {16, 24, 8}) {
            const int threads = threads_of(MW, 1), waves = threads / 64;
            if (threads > max_threads<double>()) continue;
            if (MW == 8 && best.MW && Ny1 > (nang <= 64 ? 36 : 28)) continue;
            const int resident = waves <= 4 ? 16 / waves : 4 / ((waves + 3) / 4);
            const double cost = (MW == 8 ? 1.06 : 1.0) * ((nang + MW - 1) / MW) / resident;
            if (best.MW && cost >= least) continue;
            least = cost;
            best = MarchShape{MW, 1, threads};
        }
        // (two columns per thread reach 192 columns; the limit is 170)
        return best.MW ? best : MarchShape{8, 2, threads_of(8, 2)};
    }
    constexpr int cand[][2] = {{16, 1}, {32, 3}, {16, 2}, {8, 2}, {8, 3}};
    for (const auto& c : cand) {
        const int MW = c[0], P = c[1], threads = threads_of(MW, P);
        if (MW == 32 && tiles_of(MW) * 5 < (tiles_of(MW) + 255) / 256 * 256 * 4) continue;  // 256 CUs, 80 %
        if (threads <= max_threads<float>()) return MarchShape{MW, P, threads};
    }
    return best;
}

template <typename T, int MW, int P>
void launch_march(T* F, T* f, const T* omend, int Ny, int Nz, int Ng, int nang, int threads, double dy,
                  double dz, double h, bool preserve_sign, hipStream_t s, const int* top) {
    BFPN_REQUIRE(Ny + 1 >= P, "a transport thread needs its P columns");
    const size_t lds = sizeof(T) * column_pitch<MW, P>() * (Ny + 1);
    BFPN_REQUIRE(lds <= 160 * 1024, "transport plane too wide for the LDS rings");
    const long long tiles = static_cast<long long>((nang + MW - 1) / MW) * Ng;
    BFPN_REQUIRE(tiles < (1LL << 31) - 8, "transport grid too large");
    const dim3 grid(static_cast<unsigned>((tiles + 7) / 8 * 8), f ? 2 : 1);
    auto go = [&](auto kernel) {
        allow_dynamic_lds(reinterpret_cast<const void*>(kernel), lds);
        hipLaunchKernelGGL(kernel, grid, dim3(threads), lds, s, F, f, omend, Ny, Nz, nang,
                           static_cast<T>(1.0 / dy), static_cast<T>(1.0 / dz), static_cast<T>(h),
                           static_cast<int>(tiles), top);
    };
    if (f && preserve_sign)
        go(&transport_march_kernel<T, MW, P, Arrays::SignedSigned>);
    else if (f)
        go(&transport_march_kernel<T, MW, P, Arrays::ClippedSigned>);
    else if (preserve_sign)
        go(&transport_march_kernel<T, MW, P, Arrays::Signed>);
    else
        go(&transport_march_kernel<T, MW, P, Arrays::Clipped>);
    BFPN_HIP(hipGetLastError());
}

}  // namespace

template <typename T>
void launch_transport_half(T* F, const T* omend, int Ny, int Nz, int Ng, int nang, double dy,
                           double dz, double h, bool preserve_sign, hipStream_t s,
                           const int* top, T* f) {
    if (Ng <= 0 || nang <= 0) return;
    BFPN_REQUIRE(Ny >= 1 && Nz >= 1, "transport needs Ny, Nz >= 1");
    BFPN_REQUIRE(Ny + 1 <= (sizeof(T) == 4 ? 341 : 170),
                 sizeof(T) == 4 ? "transport supports at most 341 y nodes in FP32"
                                : "transport supports at most 170 y nodes in FP64");
    // one group's block is addressed with 32-bit byte offsets
    BFPN_REQUIRE(static_cast<long long>(Ny + 1) * (Nz + 1) * nang * sizeof(T) < (1LL << 31),
                 "transport needs (Ny+1)(Nz+1)*Nmu*Nom values of one energy group below 2 GiB");
    const MarchShape sh = march_shape(Ny + 1, nang, Ng, sizeof(T));
#define BFPN_MARCH(MW_, P_)                                                                   \
    if (sh.MW == MW_ && sh.P == P_)                                                           \
        return launch_march<T, MW_, P_>(F, f, omend, Ny, Nz, Ng, nang, sh.threads, dy, dz, h,     \
                                        preserve_sign, s, top)
    BFPN_MARCH(16, 1);
    BFPN_MARCH(8, 2);
    if constexpr (sizeof(T) == 4) {
        BFPN_MARCH(32, 3);
        BFPN_MARCH(16, 2);
        BFPN_MARCH(8, 3);
    } else {
        BFPN_MARCH(24, 1);
        BFPN_MARCH(8, 1);
    }
#undef BFPN_MARCH
    throw Error(BFPN_E_INVALID, "no transport launch shape for this plane");
}

template void launch_transport_half<float>(float*, const float*, int, int, int, int, double, double,
                                           double, bool, hipStream_t, const int*, float*);
template void launch_transport_half<double>(double*, const double*, int, int, int, int, double,
                                            double, double, bool, hipStream_t, const int*, double*);

}  // namespace bfpn
