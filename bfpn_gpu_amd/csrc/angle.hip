// angle.hip — Crank-Nicolson angular diffusion on the zero-boundary DST-I basis.
//
// Reference: AngleDiffusionSolver::solveEq19 (src/angle_diffusion.cu:420-483):
// factor build, scale, and four separable kernels (FwdU, FwdV*factor, InvV,
// InvU; src/angle_diffusion.cu:254-362), each a full pass over HBM with two
// scratch arrays.
//
// MI355X design: one launch, one read and one write of the state per call.
// The whole sandwich
//     Y = Psi Su^T,  Z = coeff_g (.) (Sv Y),  W = Sv^T Z,  Psi' = W Su
// runs per (g, s) plane of Nmu x Nom values, in place.  The CN factors
// (ratio * DST normalisation) are built once on the host per (g, direction).
// FP32 state: matrix cores, stages chained in registers (below).  FP64 state:
// vector kernel, a thread per row or column of a plane.  Planes wider than 32,
// and thin ones in FP64 (angle_by_lines): vector kernel, a thread per value,
// with the plane and bases in LDS.

#include "angle_operands.hpp"
#include "buffer.hpp"
#include "kernels.hpp"
#include "mfma.hpp"

#include <type_traits>

namespace bfpn {
namespace {

// ---------------------------------------------------------- FP32 / MFMA ----
// One wave per (g, s) plane (each wave walks a contiguous run of planes), the
// plane zero padded to 32 x 32, every stage a 32x32x32 product on the matrix
// cores in split FP16 with FP32 accumulation (MT / NT = 16-row tiles along v
// and a): the state and the constant bases in two FP16 terms each, three
// products kept.  The DST runs every depth step on the same beam, so its
// error compounds: with two-term BF16 splits the FP32 IDD drifts ~1 % above
// the FP64 one over 1600 steps; two FP16 terms carry 22 significand bits,
// and the operator is about as exact as FP32 arithmetic.  FP16 needs a range: each
// plane is scaled by a power of two s so that max|X s| lies in [16, 32),
// the bases are stored times 16, so every intermediate stays below 2^14
// (|Y|, |W| <= 21 max|X| for the sine bases, |Z| <= 1.6 max|X| with the CN
// normalisation) and small values stay clear of the FP16 subnormals; the
// CN factors absorb 1/256 and the result is multiplied by 1/(256 s), all
// exact.
// The stages chain in registers, with no LDS: a stage's output tile, lane
// holding D[4q+r][i], is the next stage's K operand when the K axis is taken
// in the order  slot 8q + 4u + r  <->  index 16u + 4q + r  (chain_index), and
// the constant sine bases on the other side are stored with their columns in
// that order.  The sandwich is evaluated as
//     Y  = X Su^T            (A = X from HBM,   B = Su)
//     Z  = C (.) (Sv Y)      (A = Sv chained,   B = Y)
//     W^T = Z^T Sv           (A = Z^T,          B = Sv chained)
//     X'^T = Su^T W^T        (A = Su chained,   B = W)
// using the symmetry of the DST-I bases; X'^T leaves the last stage with 4
// consecutive elements of a plane row per lane and is stored straight back.
// V4 (Nom >= 4): rows are read and written as 16-byte vectors, columns 4k .. of
// a row per vector.  Where Nom is no multiple of 4 the row's last vector holds
// its last four columns instead and overlaps the one before: the plan stores
// the bases' columns (stage 1, the repeated ones as zeros) and rows (stage 4,
// where both lanes compute the same value) in that order, angle_column().
template <int MT, int NT, bool V4>
__global__ __launch_bounds__(256) void angle_mfma_kernel(float* __restrict__ F_, float* __restrict__ f_,
                                                         const float* __restrict__ factors,
                                                         AnglePlan plan, int planes, int per_wave,
                                                         int nyz, int Nmu, int Nom, float one,
                                                         const int* __restrict__ top) {
    float* const F = blockIdx.y ? f_ : F_;  // the second array of a launch over two
    // Only the planes of groups up to the state's top are nonzero (the
    // others stay zero): the first `active` planes, shared out evenly over
    // the grid's waves; blocks without any exit before touching LDS.
    const int active = top ? min(planes, (min(*top, planes / nyz - 1) + 1) * nyz) : planes;
    const int pw = top ? (active + gridDim.x * 4 - 1) / (gridDim.x * 4) : per_wave;
    if (static_cast<int>(blockIdx.x) * 4 * pw >= active) return;
    // The six constant basis arrays (Su, Su chained, Sv chained; hi, lo)
    // live in LDS, shared by the work-group's four waves and read per stage:
    // held in registers they would cost 48 VGPRs and one of the four waves
    // per SIMD.  Rows padded to 40 values (80 bytes) against bank conflicts.
    __shared__ __attribute__((aligned(16))) _Float16 cst[6][32][40];
    {
        const _Float16* src[6] = {plan.su_h, plan.su_l, plan.sup_h, plan.sup_l, plan.svp_h,
                                  plan.svp_l};
        for (int e = threadIdx.x; e < 6 * 32 * 4; e += blockDim.x) {  // 16-byte chunks
            const int a = e >> 7, r = (e >> 2) & 31, c = (e & 3) * 8;
            *reinterpret_cast<f16x8*>(&cst[a][r][c]) =
                *reinterpret_cast<const f16x8*>(src[a] + r * 32 + c);
        }
    }
    __syncthreads();
    const int lane = threadIdx.x & 63, i = lane & 15, q = lane >> 4;
    // (the wave's first plane, made visibly wave-uniform for the compiler)
    int p = __builtin_amdgcn_readfirstlane((blockIdx.x * 4 + (threadIdx.x >> 6)) * pw);
    const int p_end = min(active, p + pw);
    if (p >= p_end) return;
    const int na = Nmu * Nom;
    // The wave's run of planes as a buffer resource: a plane is a uniform
    // offset, the lane's elements fixed 32-bit offsets (V4: two 16-byte loads
    // per row tile, and one 16-byte store per output tile, kOutside where
    // the tile lies outside the plane).
    const int p0 = p;
    const __amdgpu_buffer_rsrc_t Fw =
        make_rsrc(F + static_cast<long long>(p0) * na,
                  static_cast<unsigned>(static_cast<long long>(p_end - p0) * na * sizeof(float)));
    unsigned ld_off[MT][2], st_off[MT][NT];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
#pragma unroll
        for (int h = 0; h < 2; ++h)
            ld_off[mt][h] = static_cast<unsigned>(
                (min(mt * 16 + i, Nmu - 1) * Nom +
                 (V4 ? min(8 * q + 4 * h, max(Nom - 4, 0)) : min(8 * q, Nom - 1))) * sizeof(float));
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) {
            const int v = mt * 16 + i, a0 = nt * 16 + 4 * q;
            const int first = V4 ? min(a0, Nom - 4) : a0;
            st_off[mt][nt] = (v < Nmu && a0 < Nom)
                                 ? static_cast<unsigned>((v * Nom + first) * sizeof(float))
                                 : kOutside;
        }
    }
    // Rows of fewer than 4 columns: a lane's columns are clamped to the row's
    // last, and its 4-column output groups are cut there.
    const int e_max = max(Nom - 1 - 8 * q, 0);
    // Fragment of constant `a` (0 Su, 1 Su chained, 2 Sv chained), tile t,
    // at compile-time offsets from the lane's base (row i, columns 8q..).
    auto frag = [&](const _Float16* base, int a, int t) {
        constexpr int kArr = 32 * 40, kTile = 16 * 40;
        return HalfFrag2{*reinterpret_cast<const f16x8*>(base + (2 * a) * kArr + t * kTile),
                         *reinterpret_cast<const f16x8*>(base + (2 * a + 1) * kArr + t * kTile)};
    };

    int g_cur = -1;
    float cf[MT][NT][4];
    int g = p / nyz, s_in = p - g * nyz;  // group and node of plane p (uniform)
    for (; p < p_end; ++p, (++s_in == nyz) ? (s_in = 0, ++g) : 0) {
        // an opaque zero per plane keeps the constant reads inside the loop
        // (`one`, a kernel argument equal to 1, keeps the residuals of the
        // splits in stages 2-4 single FMAs)
        int oz;
        asm volatile("v_mov_b32 %0, 0" : "=v"(oz));
        const _Float16* cb = &cst[0][i][8 * q] + oz;
        const unsigned so = static_cast<unsigned>((p - p0) * na * static_cast<int>(sizeof(float)));
        if (g != g_cur) {  // CN factors of this group, in the D layout, / 256
            g_cur = g;
            const float* C = factors + static_cast<long long>(g) * na;
            constexpr float kUnscale = 1.0f / (kAngleBasisScale * kAngleBasisScale);
#pragma unroll
            for (int mt = 0; mt < MT; ++mt)
#pragma unroll
                for (int nt = 0; nt < NT; ++nt)
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        const int nu = mt * 16 + 4 * q + r, mu = nt * 16 + i;
                        cf[mt][nt][r] = (nu < Nmu && mu < Nom) ? C[nu * Nom + mu] * kUnscale : 0.f;
                    }
        }
        // stage 1: Y[v][mu] = sum_a X[v][a] Su[mu][a].  The padding rows and
        // columns of the 32 x 32 tile load clamped copies of plane values:
        // the bases' zero padding multiplies them by exact zeros (columns
        // a >= Nom here, rows v >= Nmu in stage 2), so no lane is masked.
        float x[MT][8];
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
            if (V4) {
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    const float4 t = bload4(Fw, ld_off[mt][h], so);
                    x[mt][4 * h] = t.x;
                    x[mt][4 * h + 1] = t.y;
                    x[mt][4 * h + 2] = t.z;
                    x[mt][4 * h + 3] = t.w;
                }
            } else {
#pragma unroll
                for (int e = 0; e < 8; ++e)
                    x[mt][e] = bload<float>(Fw, ld_off[mt][0] + 4u * min(e, e_max), so);
            }
        }
        // the plane's scale s = 2^(4 - floor(log2 max|X|)) (biased exponent
        // clamped so that s and 1/s are normal numbers), uniform over the wave
        float mx = 0.f;
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
#pragma unroll
            for (int e = 0; e < 8; ++e) mx = fmaxf(mx, fabsf(x[mt][e]));
        const int ebits = __float_as_int(wave_max_nonneg(mx)) >> 23;
        const int sb = min(max(258 - ebits, 1), 253);
        const float sc = __int_as_float(sb << 23);
        const float unscale = __int_as_float((254 - sb) << 23) / (kAngleBasisScale * kAngleBasisScale);
        HalfFrag2 xa[MT];
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) xa[mt] = split8_h<true>(x[mt], sc);
        f32x4 d1[MT][NT];
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
#pragma unroll
            for (int nt = 0; nt < NT; ++nt) d1[mt][nt] = mma_sc(xa[mt], frag(cb, 0, nt), zero4());
        // stage 2: Z[nu][mu] = C[nu][mu] sum_v Sv[nu][v] Y[v][mu]
        f32x4 d2[MT][NT];
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) {
            float y[8];
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                y[r] = d1[0][nt][r];
                y[4 + r] = MT > 1 ? d1[MT - 1][nt][r] : 0.f;
            }
            const HalfFrag2 b = split8_h<false>(y, one);
#pragma unroll
            for (int mt = 0; mt < MT; ++mt) {
                d2[mt][nt] = mma_cs(frag(cb, 2, mt), b, zero4());
#pragma unroll
                for (int r = 0; r < 4; ++r) d2[mt][nt][r] *= cf[mt][nt][r];
            }
        }
        // stage 3: W^T[mu][v] = sum_nu Z[nu][mu] Sv[nu][v]
        f32x4 d3[NT][MT];
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) {
            float z[8];
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                z[r] = d2[0][nt][r];
                z[4 + r] = MT > 1 ? d2[MT - 1][nt][r] : 0.f;
            }
            const HalfFrag2 a = split8_h<false>(z, one);
#pragma unroll
            for (int mt = 0; mt < MT; ++mt) d3[nt][mt] = mma_sc(a, frag(cb, 2, mt), zero4());
        }
        // stage 4, transposed: X'^T[a][v] = sum_mu Su[mu][a] W[v][mu] (operands
        // swapped), so each lane holds 4 consecutive a of one row v; in place
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
            float w[8];
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                w[r] = d3[0][mt][r];
                w[4 + r] = NT > 1 ? d3[NT - 1][mt][r] : 0.f;
            }
            const HalfFrag2 b = split8_h<false>(w, one);
#pragma unroll
            for (int nt = 0; nt < NT; ++nt) {
                f32x4 d = mma_cs(frag(cb, 1, nt), b, zero4());
#pragma unroll
                for (int r = 0; r < 4; ++r) d[r] *= unscale;
                const int a0 = nt * 16 + 4 * q;
                if (V4) {
                    bstore4(make_float4(d[0], d[1], d[2], d[3]), Fw, st_off[mt][nt], so);
                } else {
#pragma unroll
                    for (int r = 0; r < 4; ++r)
                        bstore(d[r], Fw, a0 + r < Nom ? st_off[mt][nt] + 4u * r : kOutside, so);
                }
            }
        }
    }
}

// Planes of at most 16 x 16 directions: one 16 x 16 tile per stage, the same
// split FP16 arithmetic and stage chaining as above (a stage's D tile is the
// next one's operand as it is), with the constant fragments in registers and
// no LDS.  Run beside the kernel above on a beam's planes, 1 x 1 to 16 x 16
// directions, the results were the same bits; that was measured and rests on the
// order in which the hardware accumulates (mfma.hpp), it is no promise.  A plane's
// result does not depend on its place in a tile.
// Planes of at most 8 rows (PM2) or columns (PN2) share a tile, two along that
// axis at stride 8, with block-diagonal bases: up to four planes for the issue
// of one; each keeps its own scale, and a tile with a value that is not finite
// runs plane by plane, so that it spoils its own plane only.  A lane holds 4
// columns 4q .. of row i, read through a buffer resource at fixed offsets
// (outside the plane: past the resource, which reads 0 and drops stores), one
// tile ahead of the arithmetic.  VEC: Nom >= 4, one 16-byte vector per lane,
// the row's last one overlapping as above.
// What bounds it: HBM and issue about equally (80 vector operations and 2
// accesses per tile).  The general kernel padded these planes to K = 32, read
// 8 clamped values per lane and stored under branches.  Measured, per call with
// the general kernel and with this one: 13 x 13 directions (29.8 M cells, HBM
// floor 42 us) 104 -> 44 us, 11 x 11 (26.7 M) 114 -> 47, 10 x 10 (12.8 M)
// 61 -> 33, 7 x 7 (2 M, launch included) 23 -> 13.
template <bool PM2, bool PN2, bool VEC>
__global__ __launch_bounds__(256) void angle_small_kernel(float* __restrict__ F_, float* __restrict__ f_,
                                                          const float* __restrict__ factors,
                                                          AnglePlan plan, int planes, int per_wave,
                                                          int nyz, int Nmu, int Nom, float one,
                                                          const int* __restrict__ top) {
    float* const F = blockIdx.y ? f_ : F_;  // the second array of a launch over two
    constexpr int NPN = PN2 ? 2 : 1, P = (PM2 ? 2 : 1) * NPN;  // planes per tile
    const int Ng = planes / nyz;
    const int active = top ? min(planes, (min(*top, Ng - 1) + 1) * nyz) : planes;
    const int waves = gridDim.x * 4;
    const int pw = top ? ((active + waves - 1) / waves + P - 1) / P * P : per_wave;
    const int lane = threadIdx.x & 63, i = lane & 15, q = lane >> 4;
    int p = __builtin_amdgcn_readfirstlane((blockIdx.x * 4 + (threadIdx.x >> 6)) * pw);
    const int p_end = min(active, p + pw);
    if (p >= p_end) return;
    const int na = Nmu * Nom;
    const int p0 = p;
    const __amdgpu_buffer_rsrc_t Fw =
        make_rsrc(F + static_cast<long long>(p0) * na,
                  static_cast<unsigned>(static_cast<long long>(p_end - p0) * na * sizeof(float)));
    // Coordinates of a tile index x (0 .. 15) along an axis packed or not:
    // block and index inside it.
    auto blk = [](bool two, int x) { return two ? x >> 3 : 0; };
    auto idx = [](bool two, int x) { return two ? x & 7 : x; };
    // load / store layout: row i, columns 4q ..; the lane's plane in the tile
    const int v = idx(PM2, i), a0 = idx(PN2, 4 * q), lp = blk(PM2, i) * NPN + blk(PN2, 4 * q);
    unsigned off[VEC ? 1 : 4];
#pragma unroll
    for (int r = 0; r < (VEC ? 1 : 4); ++r) {
        const int c = VEC ? min(a0, Nom - 4) : a0 + r;
        off[r] = v < Nmu && a0 + r < Nom
                     ? static_cast<unsigned>((lp * na + v * Nom + c) * sizeof(float))
                     : kOutside;
    }
    // constant fragments: element (i, 4q + r) of the block-diagonal bases, Su's
    // columns (stage 1) and rows (stage 4) in vector order (Su for stage 4 and
    // Sv are stored with their columns chained: index 4k + r in slot 8k + r)
    auto constant = [](const _Float16* h, const _Float16* l, int at, bool diagonal) {
        Const16 f;
        f.hi = *reinterpret_cast<const f16x4*>(h + at);
        f.lo = *reinterpret_cast<const f16x4*>(l + at);
        if (!diagonal) f.hi = f.lo = f16x4{};
        return f;
    };
    auto wide = [](const Const16& f) {
        const f16x4 z{};
        return Const32{__builtin_shufflevector(f.lo, z, 0, 1, 2, 3, 4, 5, 6, 7),
                       __builtin_shufflevector(z, f.hi, 0, 1, 2, 3, 4, 5, 6, 7),
                       __builtin_shufflevector(f.hi, z, 0, 1, 2, 3, 4, 5, 6, 7)};
    };
    const bool du = blk(PN2, i) == blk(PN2, 4 * q), dv = blk(PM2, i) == blk(PM2, 4 * q);
    const Const16 su = constant(plan.su_h, plan.su_l, idx(PN2, i) * 32 + idx(PN2, 4 * q), du);
    const Const32 sup =
        wide(constant(plan.sup_h, plan.sup_l, idx(PN2, i) * 32 + 2 * idx(PN2, 4 * q), du));
    const Const32 sv =
        wide(constant(plan.svp_h, plan.svp_l, idx(PM2, i) * 32 + 2 * idx(PM2, 4 * q), dv));
    // CN factors in the layout of stage 2's result: nu = 4q + r, mu = i
    const int nu0 = idx(PM2, 4 * q), mu = idx(PN2, i), lpd = blk(PM2, 4 * q) * NPN + blk(PN2, i);
    f32x4 cf = zero4();
    int g_cur = -1;
    int g = p / nyz, s_in = p - g * nyz;  // group and node of the tile's first plane (uniform)

    auto load = [&](int at) {
        const unsigned so = static_cast<unsigned>((at - p0) * na * static_cast<int>(sizeof(float)));
        const bool mine = P == 1 || at + lp < p_end;  // (a run's last tile may be part full)
        f32x4 x;
        if constexpr (VEC) {
            const float4 t = bload4(Fw, mine ? off[0] : kOutside, so);
            x = f32x4{t.x, t.y, t.z, t.w};
        } else {
#pragma unroll
            for (int r = 0; r < 4; ++r) x[r] = bload<float>(Fw, mine ? off[r] : kOutside, so);
        }
        return x;
    };
    f32x4 next = load(p);
    for (; p < p_end; p += P) {
        const f32x4 x = next;
        next = load(p + P < p_end ? p + P : p);
        const bool straddles = P > 1 && s_in + P > nyz;  // planes of more than one group
        if (g != g_cur || straddles) {
            constexpr float kUnscale = 1.0f / (kAngleBasisScale * kAngleBasisScale);
            const int gl = straddles ? min(g + (s_in + lpd) / nyz, Ng - 1) : g;
            const float* C = factors + static_cast<long long>(gl) * na;
#pragma unroll
            for (int r = 0; r < 4; ++r)
                cf[r] = nu0 + r < Nmu && mu < Nom ? C[(nu0 + r) * Nom + mu] * kUnscale : 0.f;
            g_cur = straddles ? -1 : g;
        }
        for (s_in += P; s_in >= nyz; s_in -= nyz) ++g;
        const unsigned so = static_cast<unsigned>((p - p0) * na * static_cast<int>(sizeof(float)));
        // the planes of `x` (a lane of another plane: zeros, and not `mine`)
        auto sandwich = [&](f32x4 x, float mx, bool mine) {
            // each plane's scale, as in angle_mfma_kernel
            const int sb = min(max(258 - (__float_as_int(mx) >> 23), 1), 253);
            const float sc = __int_as_float(sb << 23);
            const float unscale =
                __int_as_float((254 - sb) << 23) / (kAngleBasisScale * kAngleBasisScale);
            f16x4 xh, xl;
            split4_h<true>(x, sc, xh, xl);
            const f32x4 y = mma16_sc(xh, xl, su);                    // Y  = X Su^T
            const f32x4 z = mma32_cs(sv, split44_h(y, one)) * cf;    // Z  = C (.) (Sv Y)
            const f32x4 w = mma32_sc(split44_h(z, one), sv);         // W^T = Z^T Sv
            const f32x4 d = mma32_cs(sup, split44_h(w, one)) * unscale;  // X'^T = Su^T W^T
            if constexpr (VEC) {
                bstore4(make_float4(d[0], d[1], d[2], d[3]), Fw, mine ? off[0] : kOutside, so);
            } else {
#pragma unroll
                for (int r = 0; r < 4; ++r) bstore(d[r], Fw, mine ? off[r] : kOutside, so);
            }
        };
        if constexpr (P == 1) {
            float mx = fmaxf(fmaxf(fabsf(x[0]), fabsf(x[1])), fmaxf(fabsf(x[2]), fabsf(x[3])));
            sandwich(x, wave_max_nonneg(mx), true);
        } else {
            unsigned u = 0;  // the plane's largest |value| as bits (above infinity's: NaN)
#pragma unroll
            for (int r = 0; r < 4; ++r) u = max(u, __float_as_uint(x[r]) & 0x7fffffffu);
            u = block_max_bits<PM2, PN2>(u);
            const bool mine = p + lp < p_end;
            if (__builtin_amdgcn_ballot_w64(u >= 0x7f800000u) == 0) {
                sandwich(x, __uint_as_float(u), mine);
            } else {
                for (int k = 0; k < P; ++k)
                    sandwich(lp == k ? x : zero4(), __uint_as_float(min(u, 0x7f800000u)),
                             mine && lp == k);
            }
        }
    }
}

// ------------------------------------------------------- FP64, vector ------
// FP64 planes of at most 32 x 32, not thin: one thread per row, then per column, then per
// row of a plane, its line in registers, the bases through the scalar cache
// (they are uniform, so a multiply-add reads its basis value from an SGPR and
// needs one operand of the line).  The column pass does both inner stages and
// the CN factors.  Planes pass through LDS between
// the passes (rows padded to an odd pitch); HBM accesses are coalesced copies
// of a work-group's run of planes.  Sizes are padded to those of dst_pitch(),
// the bases with zeros.
// The vector ALUs have the matrix cores' FP64 rate on this GPU, and 20 x 20
// planes would pad to 32 x 32 tiles there (2.6 times the work).  Bound: HBM and
// vector FP64 issue about equally (64 multiply-adds and 16 bytes per value at
// 20 x 20).  The kernel below, one thread per value with both operands from
// LDS: 1691 us for 21 x 21 nodes x 20 x 20 directions x 500 groups (1.4 GB;
// HBM floor 248 us), this one 497 us; 18 x 18 x 12 x 12 x 400 216 -> 91 us,
// 21 x 21 x 13 x 13 x 400 325 -> 235 us.
constexpr int kRowThreads = 256;

// y[j] = sum_k x[k] S[k][j], four sums at a time; done(j, y[j]) for each j.
// S: blocked [j / 4][k][j % 4], 64 bytes per two k, requested two such chunks
// ahead (the scheduling barrier keeps the request there; left to itself the
// compiler loads all of S and spills scalar registers by the thousand).
template <int N, typename Done>
__device__ inline void dst_line(const double* __restrict__ S, const double (&x)[N], Done&& done) {
    typedef double f64x8 __attribute__((ext_vector_type(8)));
#pragma unroll 1
    for (int j = 0; j < N; j += 4) {
        const f64x8* c = reinterpret_cast<const f64x8*>(S + j * N);
        f64x8 a = c[0], b = c[1];
        double acc[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
        for (int k = 0; k < N; k += 2) {
            const f64x8 now = a;
            a = b;
            if (k + 4 < N) b = c[k / 2 + 2];
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                acc[e] = fma(x[k], now[e], acc[e]);
                acc[e] = fma(x[k + 1], now[4 + e], acc[e]);
            }
        }
#pragma unroll
        for (int e = 0; e < 4; ++e) done(j + e, acc[e]);
    }
}

// su, sv: the bases padded to NU x NU and NV x NV, blocked as dst_line reads
// them.  EXACT: the plane is NV x NU and nothing is padded.
template <int NU, int NV, bool EXACT>
__global__ __launch_bounds__(kRowThreads) void angle_rows_kernel(
    double* __restrict__ F, const double* __restrict__ factors, const double* __restrict__ su,
    const double* __restrict__ sv, long long planes, int nyz, int Nmu, int Nom, int per_block,
    const int* __restrict__ top) {
    extern __shared__ unsigned char lds_raw[];
    const long long active =
        top ? min(planes, static_cast<long long>(min(*top, static_cast<int>(planes / nyz) - 1) + 1) * nyz)
            : planes;
    const long long p0 = static_cast<long long>(blockIdx.x) * per_block;
    if (p0 >= active) return;
    // A plane holds NV rows of pitch values, at most three rows past Nmu and
    // columns past Nom.  Those are read as zeros whatever they hold: the padded
    // bases make NaNs of them where the plane holds an infinity, which would
    // spread to all of it.  (Kept out at the stores instead, by a select 3 %, by
    // a branch, which spills scalar registers, up to four times as slow.)
    constexpr int pitch = NU | 1, plane = NV * pitch;
    double* X = reinterpret_cast<double*>(lds_raw);
    const int na = Nmu * Nom;
    const int np = static_cast<int>(min(static_cast<long long>(per_block), active - p0));
    const int rows = np * Nmu, cols = np * Nom, n = np * na;
    double* base = F + p0 * na;
    // coalesced copy of the run: value e sits at column c of row v of a plane;
    // a step of kRowThreads values is dp planes, dv rows and dc columns
    const int dr = kRowThreads / Nom, dc = kRowThreads - dr * Nom, dp = dr / Nmu, dv = dr - dp * Nmu;
    auto each = [&](auto&& f) {
        const int r = threadIdx.x / Nom;
        int c = threadIdx.x - r * Nom, p = r / Nmu, v = r - p * Nmu;
        for (int e = threadIdx.x; e < n; e += kRowThreads) {
            f(e, p * plane + v * pitch + c);
            c += dc;
            v += dv;
            p += dp;
            if (c >= Nom) {
                c -= Nom;
                ++v;
            }
            if (v >= Nmu) {
                v -= Nmu;
                ++p;
            }
        }
    };
    each([&](int e, int at) { X[at] = base[e]; });
    __syncthreads();
    auto row_pass = [&] {
        for (int r = threadIdx.x; r < rows; r += kRowThreads) {
            const int p = r / Nmu;
            double* line = X + p * plane + (r - p * Nmu) * pitch;
            double x[NU];
#pragma unroll
            for (int a = 0; a < NU; ++a) x[a] = EXACT || a < NU - 3 || a < Nom ? line[a] : 0.0;
            dst_line<NU>(su, x, [&](int j, double y) { line[j] = y; });
        }
    };
    row_pass();  // Y[v][mu] = sum_a X[v][a] Su[mu][a]
    __syncthreads();
    for (int t = threadIdx.x; t < cols; t += kRowThreads) {
        const int p = t / Nom, mu = t - p * Nom;
        const double* C = factors + (p0 + p) / nyz * na + mu;
        double* line = X + p * plane + mu;
        double x[NV];
        auto read = [&] {
#pragma unroll
            for (int v = 0; v < NV; ++v) x[v] = EXACT || v < NV - 3 || v < Nmu ? line[v * pitch] : 0.0;
        };
        // Z[nu][mu] = C[nu][mu] sum_v Sv[nu][v] Y[v][mu], in the column's place
        read();
        dst_line<NV>(sv, x, [&](int j, double y) { line[j * pitch] = y * C[min(j, Nmu - 1) * Nom]; });
        // W[v][mu] = sum_nu Sv[nu][v] Z[nu][mu]
        read();
        dst_line<NV>(sv, x, [&](int j, double y) { line[j * pitch] = y; });
    }
    __syncthreads();
    row_pass();  // X'[v][a] = sum_mu W[v][mu] Su[mu][a]
    __syncthreads();
    each([&](int e, int at) { base[e] = X[at]; });
}

// --------------------------------------------------------- vector, wide ---

constexpr int kThreads = 256;
constexpr int kMaxAngles = 1024;  // Nmu*Nom per plane held in LDS

template <typename T>
__global__ __launch_bounds__(kThreads) void angle_kernel(T* __restrict__ F,
                                                         const T* __restrict__ factors,
                                                         const T* __restrict__ su,
                                                         const T* __restrict__ sv, long long planes,
                                                         int nyz, int Nmu, int Nom, int per_block,
                                                         const int* __restrict__ top) {
    extern __shared__ unsigned char lds_raw[];
    // planes of groups above the state's top are zero and stay zero
    const long long active =
        top ? min(planes, static_cast<long long>(min(*top, static_cast<int>(planes / nyz) - 1) + 1) * nyz)
            : planes;
    const long long p0 = static_cast<long long>(blockIdx.x) * per_block;
    if (p0 >= active) return;
    T* lds = reinterpret_cast<T*>(lds_raw);
    const int na = Nmu * Nom;
    T* Su = lds;                    // Nom*Nom, Su[mu][a]
    T* Sv = Su + Nom * Nom;         // Nmu*Nmu, Sv[nu][v]
    T* X = Sv + Nmu * Nmu;          // per_block * na
    T* Y = X + per_block * na;      // per_block * na
    for (int e = threadIdx.x; e < Nom * Nom; e += kThreads) Su[e] = su[e];
    for (int e = threadIdx.x; e < Nmu * Nmu; e += kThreads) Sv[e] = sv[e];
    const int np = static_cast<int>(min(static_cast<long long>(per_block), active - p0));
    const int n = np * na;
    T* base = F + p0 * na;
    for (int e = threadIdx.x; e < n; e += kThreads) X[e] = base[e];
    __syncthreads();
    // Y[p][v][mu] = sum_a X[p][v][a] Su[mu][a]
    for (int e = threadIdx.x; e < n; e += kThreads) {
        const int p = e / na, r = e - p * na, v = r / Nom, mu = r - v * Nom;
        const T* x = X + p * na + v * Nom;
        const T* s = Su + mu * Nom;
        T acc = T(0);
        for (int a = 0; a < Nom; ++a) acc += x[a] * s[a];
        Y[e] = acc;
    }
    __syncthreads();
    // X[p][nu][mu] = coeff[g][nu][mu] * sum_v Sv[nu][v] Y[p][v][mu]
    for (int e = threadIdx.x; e < n; e += kThreads) {
        const int p = e / na, r = e - p * na, nu = r / Nom, mu = r - nu * Nom;
        const T* y = Y + p * na + mu;
        const T* s = Sv + nu * Nmu;
        T acc = T(0);
        for (int v = 0; v < Nmu; ++v) acc += s[v] * y[v * Nom];
        const long long g = (p0 + p) / nyz;
        X[e] = acc * factors[g * na + r];
    }
    __syncthreads();
    // Y[p][v][mu] = sum_nu Sv[nu][v] X[p][nu][mu]
    for (int e = threadIdx.x; e < n; e += kThreads) {
        const int p = e / na, r = e - p * na, v = r / Nom, mu = r - v * Nom;
        const T* z = X + p * na + mu;
        T acc = T(0);
        for (int nu = 0; nu < Nmu; ++nu) acc += Sv[nu * Nmu + v] * z[nu * Nom];
        Y[e] = acc;
    }
    __syncthreads();
    // F[p][v][a] = sum_mu Y[p][v][mu] Su[mu][a]
    for (int e = threadIdx.x; e < n; e += kThreads) {
        const int p = e / na, r = e - p * na, v = r / Nom, a = r - v * Nom;
        const T* w = Y + p * na + v * Nom;
        T acc = T(0);
        for (int mu = 0; mu < Nom; ++mu) acc += w[mu] * Su[mu * Nom + a];
        base[e] = acc;
    }
}

}  // namespace

void launch_angle_mfma(float* F, const float* factors, const AnglePlan& plan, int Ng, int nyz,
                       int Nmu, int Nom, hipStream_t s, const int* top, float* f) {
    BFPN_REQUIRE(Nmu >= 1 && Nom >= 1 && Nmu <= 32 && Nom <= 32, "MFMA DST needs Nmu, Nom <= 32");
    const long long planes = static_cast<long long>(Ng) * nyz;
    if (planes == 0) return;
    BFPN_REQUIRE(planes * Nmu * Nom < (1LL << 31) && planes < (1LL << 30),
                 "MFMA DST indexes planes with 32-bit offsets");
    // 8192 waves (32 per CU) walking contiguous runs of planes, in tiles of
    // planes_per_tile
    auto shape = [&](int planes_per_tile, int& per_wave) {
        const long long tiles = (planes + planes_per_tile - 1) / planes_per_tile;
        const long long waves = std::min<long long>(tiles, 8192);
        per_wave = static_cast<int>((tiles + waves - 1) / waves) * planes_per_tile;
        return (static_cast<int>((planes + per_wave - 1) / per_wave) + 3) / 4;
    };
    int per_wave = 0;
    auto go = [&](auto kernel, int planes_per_tile) {
        const int blocks = shape(planes_per_tile, per_wave);
        hipLaunchKernelGGL(kernel, dim3(blocks, f ? 2 : 1), dim3(256), 0, s, F, f, factors, plan,
                           static_cast<int>(planes), per_wave, nyz, Nmu, Nom, 1.0f, top);
    };
    const bool vec = Nom >= 4;
    if (Nmu <= 16 && Nom <= 16) {
        if (Nmu <= 8 && Nom <= 8) {
            if (vec) go(&angle_small_kernel<true, true, true>, 4);
            else go(&angle_small_kernel<true, true, false>, 4);
        } else if (Nmu <= 8) {
            go(&angle_small_kernel<true, false, true>, 2);
        } else if (Nom <= 8) {
            if (vec) go(&angle_small_kernel<false, true, true>, 2);
            else go(&angle_small_kernel<false, true, false>, 2);
        } else {
            go(&angle_small_kernel<false, false, true>, 1);
        }
    } else if (Nom > 16) {
        if (Nmu > 16) go(&angle_mfma_kernel<2, 2, true>, 1);
        else go(&angle_mfma_kernel<1, 2, true>, 1);
    } else {
        if (vec) go(&angle_mfma_kernel<2, 1, true>, 1);
        else go(&angle_mfma_kernel<2, 1, false>, 1);
    }
    BFPN_HIP(hipGetLastError());
}

template <typename T>
void launch_angle_full(T* F, const T* factors, const T* su, const T* sv, int Ng, int nyz, int Nmu,
                       int Nom, hipStream_t s, const int* top) {
    const int na = Nmu * Nom;
    BFPN_REQUIRE(na > 0 && na <= kMaxAngles, "Nmu*Nom must be in [1, 1024]");
    const long long planes = static_cast<long long>(Ng) * nyz;
    if (planes == 0) return;
    if constexpr (sizeof(T) == 8) {
        if (angle_by_lines(Nmu, Nom)) {
            const int widest = std::max(Nmu, Nom);
            const int nu = dst_pitch(Nom), nv = dst_pitch(Nmu);
            // one line per thread in the passes over the longer axis
            const int per_block = std::max(1, kRowThreads / widest);
            const size_t lds = sizeof(double) * static_cast<size_t>(per_block) * nv * (nu | 1);
            const long long blocks = (planes + per_block - 1) / per_block;
            BFPN_REQUIRE(blocks < (1LL << 31), "too many angular planes");
            auto go = [&](auto kernel) {
                allow_dynamic_lds(reinterpret_cast<const void*>(kernel), lds);
                hipLaunchKernelGGL(kernel, dim3(static_cast<unsigned>(blocks)), dim3(kRowThreads),
                                   lds, s, F, factors, su, sv, planes, nyz, Nmu, Nom, per_block, top);
            };
            auto with_nu = [&](auto u) {
                constexpr int NU = decltype(u)::value;
                auto with_nv = [&](auto v) {
                    constexpr int NV = decltype(v)::value;
                    if (Nom == NU && Nmu == NV)
                        go(&angle_rows_kernel<NU, NV, true>);
                    else
                        go(&angle_rows_kernel<NU, NV, false>);
                };
                switch (nv) {
                    case 4: with_nv(std::integral_constant<int, 4>{}); break;
                    case 8: with_nv(std::integral_constant<int, 8>{}); break;
                    case 12: with_nv(std::integral_constant<int, 12>{}); break;
                    case 16: with_nv(std::integral_constant<int, 16>{}); break;
                    case 20: with_nv(std::integral_constant<int, 20>{}); break;
                    case 24: with_nv(std::integral_constant<int, 24>{}); break;
                    case 28: with_nv(std::integral_constant<int, 28>{}); break;
                    default: with_nv(std::integral_constant<int, 32>{}); break;
                }
            };
            switch (nu) {
                case 4: with_nu(std::integral_constant<int, 4>{}); break;
                case 8: with_nu(std::integral_constant<int, 8>{}); break;
                case 12: with_nu(std::integral_constant<int, 12>{}); break;
                case 16: with_nu(std::integral_constant<int, 16>{}); break;
                case 20: with_nu(std::integral_constant<int, 20>{}); break;
                case 24: with_nu(std::integral_constant<int, 24>{}); break;
                case 28: with_nu(std::integral_constant<int, 28>{}); break;
                default: with_nu(std::integral_constant<int, 32>{}); break;
            }
            BFPN_HIP(hipGetLastError());
            return;
        }
    }
    const int per_block = std::max(1, 1024 / na);
    const size_t lds = sizeof(T) * (static_cast<size_t>(Nom) * Nom + static_cast<size_t>(Nmu) * Nmu +
                                    2 * static_cast<size_t>(per_block) * na);
    const long long blocks = (planes + per_block - 1) / per_block;
    BFPN_REQUIRE(blocks < (1LL << 31), "too many angular planes");
    hipLaunchKernelGGL(angle_kernel<T>, dim3(static_cast<unsigned>(blocks)), dim3(kThreads), lds, s,
                       F, factors, su, sv, planes, nyz, Nmu, Nom, per_block, top);
    BFPN_HIP(hipGetLastError());
}

template void launch_angle_full<float>(float*, const float*, const float*, const float*, int, int,
                                       int, int, hipStream_t, const int*);
template void launch_angle_full<double>(double*, const double*, const double*, const double*, int,
                                        int, int, int, hipStream_t, const int*);

}  // namespace bfpn
