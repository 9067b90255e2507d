// wave_sweep.hpp -- passes over register tiles, one wave per tile
// (k_wave_sweep, instantiated in kernels_reduce.hip).
//
// A pass is defined by 6 + G tile qubits: six are spelled by the lane id (the
// low ones, so that each access covers whole 128-byte lines), G by a thread's
// register slots.  A wave holds the 2^(6+G) amplitudes whose other bits agree,
// of phi and (REV) of lambda, applies every op of the pass to them and writes
// them back: no LDS traffic for the amplitudes and no barriers, so the waves
// of a SIMD drift apart and one's loads and stores hide behind another's
// arithmetic.  Ops mix amplitudes along one register bit (arithmetic only) or
// one of lane bits 0-3 (partners by DPP moves); a qubit on lane bit 4 or 5
// first changes places with one on a register bit (one instruction per word of
// a pair of slots), so the tile may be stored in another layout than it was
// loaded in.  Diagonal ops need no tile qubit.
// Controls and Z factors may sit anywhere: their parity splits into a part of
// the lane, a part of the slot (one bit per slot, prepared by the host) and a
// part fixed for the tile.
//
// REV is the adjoint's reverse sweep: in front of undoing gadget exp(i theta P)
// on both states, the op adds Im <lambda| i^{#Y} P |phi> to a per-thread FP64
// accumulator in LDS.  The factors of a gadget are real (c) and either purely
// imaginary or purely real (g), so an amplitude costs four multiply-adds.
#pragma once

#include "launch.hpp"

namespace fsa {
namespace sweep {

__device__ __forceinline__ double flip(double v, uint32_t signBit) {
    return __builtin_bit_cast(double, __builtin_bit_cast(uint64_t, v) ^ ((uint64_t)signBit << 32));
}
__device__ __forceinline__ float flip(float v, uint32_t signBit) {
    return __builtin_bit_cast(float, __builtin_bit_cast(uint32_t, v) ^ signBit);
}
// sign bit of slot i
__device__ __forceinline__ uint32_t slot_sign(uint32_t sw, int i) { return (sw << (31 - i)) & 0x80000000u; }

// An empty constraint that differs between the forms of an op.  Without it the
// compiler moves what the forms share (c * x of every amplitude) in front of
// the branch between them, which takes more registers than there are.
template <int ID, typename R>
__device__ __forceinline__ void pin(R& v) { asm volatile("" : "+v"(v) : "n"(ID)); }

// v' = c v + (i g or g) w: IMAG picks the imaginary factor (lane bits, diagonal groups)
template <bool IMAG, typename R>
__device__ __forceinline__ void rot(R& x, R& y, R wx, R wy, R c, R g) {
    const R ox = x, oy = y;
    if constexpr (IMAG) {
        x = c * ox - g * wy;
        y = c * oy + g * wx;
    } else {
        x = c * ox + g * wx;
        y = c * oy + g * wy;
    }
}

// The rotation (x, y) -> (cos a x - sin a y, sin a x + cos a y) as three shears,
// T = -tan(a / 2) and g = sin a: three multiply-adds in place instead of two
// and two products, and |T| <= 1 because the host takes a from (-pi/2, pi/2].
template <typename R>
__device__ __forceinline__ void shear(R& x, R& y, R T, R g) {
    x += T * y;
    y += g * x;
    x += T * y;
}

// Im or Re of conj(l) p in FP64
template <bool IMAG, typename R>
__device__ __forceinline__ double term(R lx, R ly, R px, R py) {
    if constexpr (IMAG) return (double)lx * (double)py - (double)ly * (double)px;
    else return (double)lx * (double)px + (double)ly * (double)py;
}

// Forward passes in FP32 rotate with the rounded cosine and sine instead.  Their
// norm is not quite 1, which <H> = <phi|H|phi> / <phi|phi> cancels; rounded shears
// keep the determinant but not the circle, and leave <H> of 6 layers on 13 qubits
// 1.4 times as far off (gradients are as good either way).  It costs FP32
// gradients 1%.
template <typename R, bool REV> constexpr bool sweep_shears() { return REV || sizeof(R) == 8; }
// c: the shear coefficient T (SHEAR) or the cosine
template <bool SHEAR, typename R>
__device__ __forceinline__ void turn(R& x, R& y, R c, R g) {
    if constexpr (SHEAR) {
        shear(x, y, c, g);
    } else {
        const R ox = x, oy = y;
        x = c * ox - g * oy;
        y = c * oy + g * ox;
    }
}

template <typename R, int S>
struct Tile {
    R px[S], py[S], lx[S], ly[S];
};

// the value of lane l ^ (1 << BIT): DPP moves on the vector unit (quad_perm,
// row_half_mirror after quad_perm, row_ror:8), so the exchange does not go
// through the LDS crossbar
template <int BIT>
__device__ __forceinline__ uint32_t lane_xor32(uint32_t v) {
#if defined(__AMDGCN__)
    if constexpr (BIT == 0) return __builtin_amdgcn_update_dpp(v, v, 0xB1, 0xf, 0xf, true);
    if constexpr (BIT == 1) return __builtin_amdgcn_update_dpp(v, v, 0x4E, 0xf, 0xf, true);
    if constexpr (BIT == 2) {
        v = __builtin_amdgcn_update_dpp(v, v, 0x1B, 0xf, 0xf, true);
        return __builtin_amdgcn_update_dpp(v, v, 0x141, 0xf, 0xf, true);
    }
    return __builtin_amdgcn_update_dpp(v, v, 0x128, 0xf, 0xf, true);
#else
    return (uint32_t)__shfl_xor(v, 1 << BIT, 64);
#endif
}
template <int BIT>
__device__ __forceinline__ float lane_xor(float v) {
    return __builtin_bit_cast(float, lane_xor32<BIT>(__builtin_bit_cast(uint32_t, v)));
}
template <int BIT>
__device__ __forceinline__ double lane_xor(double v) {
    const uint64_t u = __builtin_bit_cast(uint64_t, v);
    return __builtin_bit_cast(double, (uint64_t)lane_xor32<BIT>((uint32_t)u) |
                                          ((uint64_t)lane_xor32<BIT>((uint32_t)(u >> 32)) << 32));
}

// lane bit L (4 or 5) and the register bit that tells a from b change places:
// a's upper half goes to b's lower one and back, one instruction per word
template <int L>
__device__ __forceinline__ void exchange32(uint32_t& a, uint32_t& b) {
#if defined(__AMDGCN__)
    if constexpr (L == 5) {
        const auto r = __builtin_amdgcn_permlane32_swap(a, b, false, false);
        a = r[0]; b = r[1];
    } else {
        const auto r = __builtin_amdgcn_permlane16_swap(a, b, false, false);
        a = r[0]; b = r[1];
    }
#else
    const bool up = (threadIdx.x >> L) & 1u;
    const uint32_t x = (uint32_t)__shfl_xor(up ? a : b, 1 << L, 64);
    if (up) a = x;
    else b = x;
#endif
}
template <int L>
__device__ __forceinline__ void exchange(float& a, float& b) {
    uint32_t x = __builtin_bit_cast(uint32_t, a), y = __builtin_bit_cast(uint32_t, b);
    exchange32<L>(x, y);
    a = __builtin_bit_cast(float, x);
    b = __builtin_bit_cast(float, y);
}
template <int L>
__device__ __forceinline__ void exchange(double& a, double& b) {
    const uint64_t x = __builtin_bit_cast(uint64_t, a), y = __builtin_bit_cast(uint64_t, b);
    uint32_t xl = (uint32_t)x, xh = (uint32_t)(x >> 32), yl = (uint32_t)y, yh = (uint32_t)(y >> 32);
    exchange32<L>(xl, yl);
    exchange32<L>(xh, yh);
    a = __builtin_bit_cast(double, (uint64_t)xl | ((uint64_t)xh << 32));
    b = __builtin_bit_cast(double, (uint64_t)yl | ((uint64_t)yh << 32));
}

// the tile's sum of Im conj(lambda) phi, slots signed by sw
template <typename R, int S, bool SS>
__device__ __forceinline__ double diag_sum(Tile<R, S>& t, uint32_t sw) {
    double s[2] = {0, 0};
#pragma unroll
    for (int i = 0; i < S; i++) {
        pin<SS>(t.lx[i]);
        pin<SS>(t.ly[i]);
        const double w = term<true>(t.lx[i], t.ly[i], t.px[i], t.py[i]);
        s[i & 1] += SS ? flip(w, slot_sign(sw, i)) : w;
    }
    return s[0] + s[1];
}

// diagonal factors: v' = v (c + i g s), s the slot's sign
// (ONE: c is turn()'s, of a single gadget)
template <typename R, int S, bool REV, bool ONE, bool SS>
__device__ __forceinline__ void op_diag(Tile<R, S>& t, R c, R g, uint32_t sw) {
    pin<2 + 2 * ONE + SS>(c);
    pin<2 + 2 * ONE + SS>(g);
#pragma unroll
    for (int i = 0; i < S; i++) {
        const R gi = SS ? flip(g, slot_sign(sw, i)) : g;
        if constexpr (ONE) {
            constexpr bool SH = sweep_shears<R, REV>();
            const R Ti = SS && SH ? flip(c, slot_sign(sw, i)) : c;
            if constexpr (REV) shear(t.lx[i], t.ly[i], Ti, gi);
            turn<SH>(t.px[i], t.py[i], Ti, gi);
        } else {
            if constexpr (REV) rot<true>(t.lx[i], t.ly[i], t.lx[i], t.ly[i], c, gi);
            rot<true>(t.px[i], t.py[i], t.px[i], t.py[i], c, gi);
        }
    }
}

// The X/Y qubit on register bit B: pairs (i, j = i | 1 << B), each two plane
// rotations.  IMAG (X): v_i' = c v_i + i g v_j and back mix (x_i, y_j) and
// (x_j, y_i); the two amplitudes have the same sign.  Otherwise (Y)
// v_i' = c v_i - g v_j, v_j' = c v_j + g v_i mix (x_i, x_j) and (y_i, y_j); the
// signs are opposite, and g is taken with that of i, the second's partner.
template <typename R, int S, bool REV, int B, bool IMAG, bool SS>
__device__ __forceinline__ void op_reg(Tile<R, S>& t, R T, R g, uint32_t sw, double& sum) {
    constexpr int ID = 8 + 4 * B + 2 * IMAG + SS;
    pin<ID>(T);
    pin<ID>(g);
    double s[2] = {0, 0};
#pragma unroll
    for (int i = 0; i < S; i++) {
        if (i & (1 << B)) continue;
        const int j = i | (1 << B);
        constexpr bool SH = sweep_shears<R, REV>();
        const R gi = SS ? flip(g, slot_sign(sw, i)) : g, Ti = SS && SH ? flip(T, slot_sign(sw, i)) : T;
        if constexpr (REV) {
            pin<ID>(t.lx[i]);
            pin<ID>(t.ly[i]);
            pin<ID>(t.lx[j]);
            pin<ID>(t.ly[j]);
            // an amplitude takes its partner's sign
            const double wi = term<IMAG>(t.lx[i], t.ly[i], t.px[j], t.py[j]);
            const double wj = term<IMAG>(t.lx[j], t.ly[j], t.px[i], t.py[i]);
            s[0] += SS ? flip(wi, slot_sign(sw, j)) : wi;
            s[1] += SS ? flip(wj, slot_sign(sw, i)) : wj;
            if constexpr (IMAG) {
                shear(t.lx[i], t.ly[j], Ti, gi);
                shear(t.lx[j], t.ly[i], Ti, gi);
            } else {
                shear(t.lx[i], t.lx[j], Ti, gi);
                shear(t.ly[i], t.ly[j], Ti, gi);
            }
        }
        if constexpr (IMAG) {
            turn<SH>(t.px[i], t.py[j], Ti, gi);
            turn<SH>(t.px[j], t.py[i], Ti, gi);
        } else {
            turn<SH>(t.px[i], t.px[j], Ti, gi);
            turn<SH>(t.py[i], t.py[j], Ti, gi);
        }
    }
    sum = s[0] + s[1];
}

// the X/Y qubit on lane bit B: partners from lane l ^ (1 << B) (g carries the partner lane's sign)
template <typename R, int S, bool REV, int B, bool IMAG, bool SS>
__device__ __forceinline__ void op_lane(Tile<R, S>& t, R c, R g, uint32_t sw, double& sum) {
    pin<100 + 4 * B + 2 * IMAG + SS>(c);
    pin<100 + 4 * B + 2 * IMAG + SS>(g);
    double s[2] = {0, 0};
#pragma unroll
    for (int i = 0; i < S; i++) {
        const R gi = SS ? flip(g, slot_sign(sw, i)) : g;
        const R wx = lane_xor<B>(t.px[i]), wy = lane_xor<B>(t.py[i]);
        if constexpr (REV) {
            const double w = term<IMAG>(t.lx[i], t.ly[i], wx, wy);
            s[i & 1] += SS ? flip(w, slot_sign(sw, i)) : w;
            const R ux = lane_xor<B>(t.lx[i]), uy = lane_xor<B>(t.ly[i]);
            rot<IMAG>(t.lx[i], t.ly[i], ux, uy, c, gi);
        }
        rot<IMAG>(t.px[i], t.py[i], wx, wy, c, gi);
    }
    sum = s[0] + s[1];
}

// lane bit L and register bit B change places
template <typename R, int S, bool REV, int L, int B>
__device__ __forceinline__ void op_swap(Tile<R, S>& t) {
#pragma unroll
    for (int i = 0; i < S; i++) {
        if (i & (1 << B)) continue;
        const int j = i | (1 << B);
        exchange<L>(t.px[i], t.px[j]);
        exchange<L>(t.py[i], t.py[j]);
        if constexpr (REV) {
            exchange<L>(t.lx[i], t.lx[j]);
            exchange<L>(t.ly[i], t.ly[j]);
        }
    }
}

template <typename R>
__device__ __forceinline__ void mat_pair(R& ax, R& ay, R& bx, R& by, const R* f) {
    const cx<R> a = mk<R>(ax, ay), b = mk<R>(bx, by);
    const cx<R> u = cfma(cmul(mk<R>(f[0], f[1]), a), mk<R>(f[2], f[3]), b);
    const cx<R> v = cfma(cmul(mk<R>(f[4], f[5]), a), mk<R>(f[6], f[7]), b);
    ax = u.x; ay = u.y; bx = v.x; by = v.y;
}

// 2x2 matrix on register bit B, on the pairs whose slot bit is set in sw (on: this lane's controls are set)
template <typename R, int S, bool REV, int B>
__device__ __forceinline__ void op_mat_reg(Tile<R, S>& t, const R* fu, uint32_t sw, bool on) {
    if (!on) return;
    R f[8];
#pragma unroll
    for (int k = 0; k < 8; k++) { f[k] = fu[k]; pin<40 + B>(f[k]); }
#pragma unroll
    for (int i = 0; i < S; i++) {
        if ((i & (1 << B)) || !((sw >> i) & 1u)) continue;
        const int j = i | (1 << B);
        mat_pair(t.px[i], t.py[i], t.px[j], t.py[j], f);
        if constexpr (REV) mat_pair(t.lx[i], t.ly[i], t.lx[j], t.ly[j], f);
    }
}

// 2x2 matrix on a lane bit; set: this lane holds the pair's second amplitude
template <typename R, int S, bool REV>
__device__ __forceinline__ void op_mat_lane(Tile<R, S>& t, int m, bool set, const R* f, uint32_t sw, bool on) {
    const cx<R> own = set ? mk<R>(f[6], f[7]) : mk<R>(f[0], f[1]);
    const cx<R> off = set ? mk<R>(f[4], f[5]) : mk<R>(f[2], f[3]);
#pragma unroll
    for (int i = 0; i < S; i++) {
        if (!((sw >> i) & 1u)) continue;                     // the same for every lane
        const cx<R> w = mk<R>(__shfl_xor(t.px[i], m, 64), __shfl_xor(t.py[i], m, 64));
        const cx<R> p = cfma(cmul(own, mk<R>(t.px[i], t.py[i])), off, w);
        if (on) { t.px[i] = p.x; t.py[i] = p.y; }
        if constexpr (REV) {
            const cx<R> u = mk<R>(__shfl_xor(t.lx[i], m, 64), __shfl_xor(t.ly[i], m, 64));
            const cx<R> l = cfma(cmul(own, mk<R>(t.lx[i], t.ly[i])), off, u);
            if (on) { t.lx[i] = l.x; t.ly[i] = l.y; }
        }
    }
}

// Applies an op other than a diagonal gadget to the tile (hdr: its fields up to
// g, already loaded; sb: sign bit of its lane and tile part) and returns the
// lane's part of its gradient term.
template <typename R, int G, bool REV>
__device__ __forceinline__ double apply(Tile<R, 1 << G>& t, const SweepOp& hdr, const SweepOp* __restrict__ op,
                                        uint32_t lane, uint64_t base, uint32_t sb) {
    constexpr int S = 1 << G;
    const uint32_t sw = hdr.sw;
    if (hdr.code >= SWEEP_MAT_LANE) {
        if ((base & hdr.oz) != hdr.oz) return 0;             // a control outside the tile is 0
        R f[8];
#pragma unroll
        for (int i = 0; i < 8; i++) f[i] = (R)op->f[i];
        const bool on = (lane & hdr.lz) == hdr.lz;
        const uint32_t bit = op->bit;
        switch (hdr.code) {
        case SWEEP_MAT_LANE: op_mat_lane<R, S, REV>(t, 1 << bit, ((lane >> bit) & 1u) != 0, f, sw, on); break;
        case SWEEP_MAT_REG + 0: if constexpr (G > 0) op_mat_reg<R, S, REV, 0>(t, f, sw, on); break;
        case SWEEP_MAT_REG + 1: if constexpr (G > 1) op_mat_reg<R, S, REV, 1>(t, f, sw, on); break;
        case SWEEP_MAT_REG + 2: if constexpr (G > 2) op_mat_reg<R, S, REV, 2>(t, f, sw, on); break;
        case SWEEP_MAT_REG + 3: if constexpr (G > 3) op_mat_reg<R, S, REV, 3>(t, f, sw, on); break;
        case SWEEP_MAT_REG + 4: if constexpr (G > 4) op_mat_reg<R, S, REV, 4>(t, f, sw, on); break;
        default: break;
        }
        return 0;
    }
    // a shear coefficient (register bits) changes sign with g, a cosine does not
    const R g = flip((R)hdr.g, sb), c = sweep_shears<R, REV>() && hdr.code >= SWEEP_REG ? flip((R)hdr.c, sb) : (R)hdr.c;
    double sum = 0;
    switch (hdr.code) {
#define FSA_SWEEP_FORMS(OP, BASE, BV)                                             \
    case BASE + 4 * BV: OP<R, S, REV, BV, false, false>(t, c, g, sw, sum); break; \
    case BASE + 4 * BV + 1: OP<R, S, REV, BV, false, true>(t, c, g, sw, sum); break; \
    case BASE + 4 * BV + 2: OP<R, S, REV, BV, true, false>(t, c, g, sw, sum); break; \
    case BASE + 4 * BV + 3: OP<R, S, REV, BV, true, true>(t, c, g, sw, sum); break;
    FSA_SWEEP_FORMS(op_lane, SWEEP_LANE, 0) FSA_SWEEP_FORMS(op_lane, SWEEP_LANE, 1)
    FSA_SWEEP_FORMS(op_lane, SWEEP_LANE, 2) FSA_SWEEP_FORMS(op_lane, SWEEP_LANE, 3)
    FSA_SWEEP_FORMS(op_reg, SWEEP_REG, 0) FSA_SWEEP_FORMS(op_reg, SWEEP_REG, 1) FSA_SWEEP_FORMS(op_reg, SWEEP_REG, 2)
#undef FSA_SWEEP_FORMS
    // register bits that not every tile has
#define FSA_SWEEP_FORMS(BV)                                                                                      \
    case SWEEP_REG + 4 * BV: if constexpr (G > BV) op_reg<R, S, REV, BV, false, false>(t, c, g, sw, sum); break; \
    case SWEEP_REG + 4 * BV + 1: if constexpr (G > BV) op_reg<R, S, REV, BV, false, true>(t, c, g, sw, sum); break; \
    case SWEEP_REG + 4 * BV + 2: if constexpr (G > BV) op_reg<R, S, REV, BV, true, false>(t, c, g, sw, sum); break; \
    case SWEEP_REG + 4 * BV + 3: if constexpr (G > BV) op_reg<R, S, REV, BV, true, true>(t, c, g, sw, sum); break;
    FSA_SWEEP_FORMS(3) FSA_SWEEP_FORMS(4)
#undef FSA_SWEEP_FORMS
#define FSA_SWEEP_SWAP(LV, BV) \
    case SWEEP_SWAP + 5 * (LV - 4) + BV: if constexpr (G > BV) op_swap<R, S, REV, LV, BV>(t); break;
    FSA_SWEEP_SWAP(4, 0) FSA_SWEEP_SWAP(4, 1) FSA_SWEEP_SWAP(4, 2) FSA_SWEEP_SWAP(4, 3) FSA_SWEEP_SWAP(4, 4)
    FSA_SWEEP_SWAP(5, 0) FSA_SWEEP_SWAP(5, 1) FSA_SWEEP_SWAP(5, 2) FSA_SWEEP_SWAP(5, 3) FSA_SWEEP_SWAP(5, 4)
#undef FSA_SWEEP_SWAP
    default: break;
    }
    return flip(sum, sb);
}

}  // namespace sweep
}  // namespace fsa
