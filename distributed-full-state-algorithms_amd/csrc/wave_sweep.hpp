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
// one lane bit (partners from lane l ^ bit); diagonal ops need no tile qubit.
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

// v' = c v + (i g or g) w: IMAG picks the imaginary factor
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

// Im or Re of conj(l) p in FP64
template <bool IMAG, typename R>
__device__ __forceinline__ double term(R lx, R ly, R px, R py) {
    if constexpr (IMAG) return (double)lx * (double)py - (double)ly * (double)px;
    else return (double)lx * (double)px + (double)ly * (double)py;
}

template <typename R, int S>
struct Tile {
    R px[S], py[S], lx[S], ly[S];
};

// e^{-i theta Z..Z}: v' = v (c + i g s), s = +-1 by parity (g carries the lane's sign)
template <typename R, int S, bool REV, bool SS>
__device__ __forceinline__ void op_diag(Tile<R, S>& t, R c, R g, uint32_t sw, double& sum) {
    pin<SS>(c);
    pin<SS>(g);
    double s[2] = {0, 0};
#pragma unroll
    for (int i = 0; i < S; i++) {
        const R gi = SS ? flip(g, slot_sign(sw, i)) : g;
        if constexpr (REV) {
            pin<SS>(t.lx[i]);
            pin<SS>(t.ly[i]);
            const double w = term<true>(t.lx[i], t.ly[i], t.px[i], t.py[i]);
            s[i & 1] += SS ? flip(w, slot_sign(sw, i)) : w;
            rot<true>(t.lx[i], t.ly[i], t.lx[i], t.ly[i], c, gi);
        }
        rot<true>(t.px[i], t.py[i], t.px[i], t.py[i], c, gi);
    }
    sum = s[0] + s[1];
}

// the X/Y qubit on register bit B: pairs (i, j = i | 1 << B)
template <typename R, int S, bool REV, int B, bool IMAG, bool SS>
__device__ __forceinline__ void op_reg(Tile<R, S>& t, R c, R g, uint32_t sw, double& sum) {
    pin<8 + 4 * B + 2 * IMAG + SS>(c);
    pin<8 + 4 * B + 2 * IMAG + SS>(g);
    double s[2] = {0, 0};
#pragma unroll
    for (int i = 0; i < S; i++) {
        if (i & (1 << B)) continue;
        const int j = i | (1 << B);
        // an amplitude takes its partner's sign
        const R gi = SS ? flip(g, slot_sign(sw, i)) : g, gj = SS ? flip(g, slot_sign(sw, j)) : g;
        if constexpr (REV) {
            pin<8 + 4 * B + 2 * IMAG + SS>(t.lx[i]);
            pin<8 + 4 * B + 2 * IMAG + SS>(t.ly[i]);
            pin<8 + 4 * B + 2 * IMAG + SS>(t.lx[j]);
            pin<8 + 4 * B + 2 * IMAG + SS>(t.ly[j]);
            const double wi = term<IMAG>(t.lx[i], t.ly[i], t.px[j], t.py[j]);
            const double wj = term<IMAG>(t.lx[j], t.ly[j], t.px[i], t.py[i]);
            s[0] += SS ? flip(wi, slot_sign(sw, j)) : wi;
            s[1] += SS ? flip(wj, slot_sign(sw, i)) : wj;
            const R ax = t.lx[i], ay = t.ly[i];
            rot<IMAG>(t.lx[i], t.ly[i], t.lx[j], t.ly[j], c, gj);
            rot<IMAG>(t.lx[j], t.ly[j], ax, ay, c, gi);
        }
        const R ax = t.px[i], ay = t.py[i];
        rot<IMAG>(t.px[i], t.py[i], t.px[j], t.py[j], c, gj);
        rot<IMAG>(t.px[j], t.py[j], ax, ay, c, gi);
    }
    sum = s[0] + s[1];
}

// the X/Y qubit on a lane bit: partners from lane l ^ m (g carries the partner lane's sign)
template <typename R, int S, bool REV, bool IMAG, bool SS>
__device__ __forceinline__ void op_lane(Tile<R, S>& t, int m, R c, R g, uint32_t sw, double& sum) {
    pin<4 + 2 * IMAG + SS>(c);
    pin<4 + 2 * IMAG + SS>(g);
    double s[2] = {0, 0};
#pragma unroll
    for (int i = 0; i < S; i++) {
        const R gi = SS ? flip(g, slot_sign(sw, i)) : g;
        const R wx = __shfl_xor(t.px[i], m, 64), wy = __shfl_xor(t.py[i], m, 64);
        if constexpr (REV) {
            const double w = term<IMAG>(t.lx[i], t.ly[i], wx, wy);
            s[i & 1] += SS ? flip(w, slot_sign(sw, i)) : w;
            const R ux = __shfl_xor(t.lx[i], m, 64), uy = __shfl_xor(t.ly[i], m, 64);
            rot<IMAG>(t.lx[i], t.ly[i], ux, uy, c, gi);
        }
        rot<IMAG>(t.px[i], t.py[i], wx, wy, c, gi);
    }
    sum = s[0] + s[1];
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

// Applies op to the tile (hdr: its fields up to g, already loaded) and returns
// the lane's part of its gradient term.
template <typename R, int G, bool REV>
__device__ __forceinline__ double apply(Tile<R, 1 << G>& t, const SweepOp& hdr, const SweepOp* __restrict__ op,
                                        uint32_t lane, uint64_t base) {
    constexpr int S = 1 << G;
    if (hdr.code >= SWEEP_MAT_LANE) {
        if ((base & hdr.oz) != hdr.oz) return 0;             // a control outside the tile is 0
        R f[8];
#pragma unroll
        for (int i = 0; i < 8; i++) f[i] = (R)op->f[i];
        const bool on = (lane & hdr.lz) == hdr.lz;
        const uint32_t bit = op->bit;
        switch (hdr.code) {
        case SWEEP_MAT_LANE: op_mat_lane<R, S, REV>(t, 1 << bit, ((lane >> bit) & 1u) != 0, f, hdr.sw, on); break;
        case SWEEP_MAT_REG + 0: if constexpr (G > 0) op_mat_reg<R, S, REV, 0>(t, f, hdr.sw, on); break;
        case SWEEP_MAT_REG + 1: if constexpr (G > 1) op_mat_reg<R, S, REV, 1>(t, f, hdr.sw, on); break;
        case SWEEP_MAT_REG + 2: if constexpr (G > 2) op_mat_reg<R, S, REV, 2>(t, f, hdr.sw, on); break;
        case SWEEP_MAT_REG + 3: if constexpr (G > 3) op_mat_reg<R, S, REV, 3>(t, f, hdr.sw, on); break;
        case SWEEP_MAT_REG + 4: if constexpr (G > 4) op_mat_reg<R, S, REV, 4>(t, f, hdr.sw, on); break;
        default: break;
        }
        return 0;
    }
    const R c = (R)hdr.c;
    // lane and tile part of the sign
    const uint32_t sb = (par32((lane | SWEEP_CONST_SIGN) & hdr.lz) ^ par64(base & hdr.oz)) << 31;
    const R g = flip((R)hdr.g, sb);
    const uint32_t sw = hdr.sw;
    double sum = 0;
    switch (hdr.code) {
    case SWEEP_DIAG: op_diag<R, S, REV, false>(t, c, g, sw, sum); break;
    case SWEEP_DIAG + 1: op_diag<R, S, REV, true>(t, c, g, sw, sum); break;
    case SWEEP_LANE: op_lane<R, S, REV, false, false>(t, 1 << op->bit, c, g, sw, sum); break;
    case SWEEP_LANE + 1: op_lane<R, S, REV, false, true>(t, 1 << op->bit, c, g, sw, sum); break;
    case SWEEP_LANE + 2: op_lane<R, S, REV, true, false>(t, 1 << op->bit, c, g, sw, sum); break;
    case SWEEP_LANE + 3: op_lane<R, S, REV, true, true>(t, 1 << op->bit, c, g, sw, sum); break;
#define FSA_SWEEP_B(BV)                                                                                          \
    case SWEEP_REG + 4 * BV: if constexpr (G > BV) op_reg<R, S, REV, BV, false, false>(t, c, g, sw, sum); break; \
    case SWEEP_REG + 4 * BV + 1: if constexpr (G > BV) op_reg<R, S, REV, BV, false, true>(t, c, g, sw, sum); break; \
    case SWEEP_REG + 4 * BV + 2: if constexpr (G > BV) op_reg<R, S, REV, BV, true, false>(t, c, g, sw, sum); break; \
    case SWEEP_REG + 4 * BV + 3: if constexpr (G > BV) op_reg<R, S, REV, BV, true, true>(t, c, g, sw, sum); break;
    FSA_SWEEP_B(0) FSA_SWEEP_B(1) FSA_SWEEP_B(2) FSA_SWEEP_B(3) FSA_SWEEP_B(4)
#undef FSA_SWEEP_B
    default: break;
    }
    return flip(sum, sb);
}

}  // namespace sweep
}  // namespace fsa
