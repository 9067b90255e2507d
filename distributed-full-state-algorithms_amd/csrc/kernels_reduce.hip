// kernels_reduce.hip -- reductions (FP64 accumulation, fixed order), partial
// trace, Pauli-sum application, state initialisation and precision conversion.
//
// Reductions are two-level and deterministic: a fixed grid writes one partial
// per workgroup (wavefront shuffle, then LDS across the 4 waves), and a single
// workgroup sums the partials in index order.  Results never depend on timing.
#include "engine.hpp"

#include <cstring>
#include "launch.hpp"
#include "wave_sweep.hpp"

namespace fsa {

namespace {

constexpr int RED_ITEMS = 8;
// grid cap of the grid-stride reductions and adjoint sweep kernels: four
// 256-thread blocks per CU.  The 24-qubit adjoint ran 1.3-1.4% faster than with
// 2048 (FP64 diagonal passes 4% faster) and 4096 was slower (same box).
constexpr unsigned RED_MAX_BLOCKS = 1024;

__device__ __forceinline__ double wave_sum(double v) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v += __shfl_down(v, off, 64);
    return v;
}

// sum of (vr, vi) over the workgroup into lane 0 of wave 0
__device__ __forceinline__ void block_sum2(double& vr, double& vi) {
    __shared__ double sr[BLOCK / 64], si[BLOCK / 64];
    vr = wave_sum(vr);
    vi = wave_sum(vi);
    const unsigned lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
    if (lane == 0) { sr[wave] = vr; si[wave] = vi; }
    __syncthreads();
    if (threadIdx.x == 0) {
        double a = 0, b = 0;
        for (int w = 0; w < BLOCK / 64; w++) { a += sr[w]; b += si[w]; }
        vr = a; vi = b;
    }
}

unsigned red_blocks(uint64_t num) {
    uint64_t per = (uint64_t)BLOCK * RED_ITEMS;
    uint64_t b = (num + per - 1) / per;
    if (b < 1) b = 1;
    if (b > RED_MAX_BLOCKS) b = RED_MAX_BLOCKS;
    return (unsigned)b;
}

__global__ __launch_bounds__(BLOCK) void k_final_sum(const double* __restrict__ part, unsigned numParts,
                                                     double* __restrict__ out) {
    double vr = 0, vi = 0;
    for (unsigned i = threadIdx.x; i < numParts; i += BLOCK) { vr += part[2 * i]; vi += part[2 * i + 1]; }
    block_sum2(vr, vi);
    if (threadIdx.x == 0) { out[0] = vr; out[1] = vi; }
}

// per-slot sums of the adjoint sweep's partial rows: block p adds the first
// nb[p] rows of slot p in row order (the order k_final_sum uses)
__global__ __launch_bounds__(BLOCK) void k_grad_sums(const double* __restrict__ rows, uint64_t stride,
                                                     const uint32_t* __restrict__ nb, double* __restrict__ res) {
    const double* r = rows + stride * blockIdx.x;
    const unsigned n = nb[blockIdx.x];
    double vr = 0, vi = 0;
    for (unsigned i = threadIdx.x; i < n; i += BLOCK) { vr += r[2 * i]; vi += r[2 * i + 1]; }
    block_sum2(vr, vi);
    if (threadIdx.x == 0) { res[2 * blockIdx.x] = vr; res[2 * blockIdx.x + 1] = vi; }
}

template <typename R>
__global__ __launch_bounds__(BLOCK) void k_norm2(const cx<R>* __restrict__ a, uint64_t num,
                                                 double* __restrict__ part) {
    double acc = 0;
    for (uint64_t j = (uint64_t)blockIdx.x * BLOCK + threadIdx.x; j < num; j += (uint64_t)gridDim.x * BLOCK) {
        cx<R> v = a[j];
        acc += (double)v.x * (double)v.x + (double)v.y * (double)v.y;
    }
    double dummy = 0;
    block_sum2(acc, dummy);
    if (threadIdx.x == 0) { part[2 * blockIdx.x] = acc; part[2 * blockIdx.x + 1] = 0; }
}

template <typename R>
__global__ __launch_bounds__(BLOCK) void k_inner(const cx<R>* __restrict__ a, const cx<R>* __restrict__ b,
                                                 uint64_t num, double* __restrict__ part) {
    double vr = 0, vi = 0;
    for (uint64_t j = (uint64_t)blockIdx.x * BLOCK + threadIdx.x; j < num; j += (uint64_t)gridDim.x * BLOCK) {
        cx<R> x = a[j], y = b[j];
        // conj(x) * y
        vr += (double)x.x * (double)y.x + (double)x.y * (double)y.y;
        vi += (double)x.x * (double)y.y - (double)x.y * (double)y.x;
    }
    block_sum2(vr, vi);
    if (threadIdx.x == 0) { part[2 * blockIdx.x] = vr; part[2 * blockIdx.x + 1] = vi; }
}

// Pauli-string sums.  Workgroup (t, c) handles term t over chunk c of 2^N (DM)
// or 2^n (SV) indices and writes f_t * (its partial sum).
//  DM (reference distributed_densitymatrix.hpp:322-344 / misc.hpp:16-38): only
//  entries with column c = r ^ mxy are nonzero, each sigma product equals
//  (-i)^{#Y} (-1)^{par(c & myz)}, so Tr(P rho) = (-i)^{#Y} sum_r (-1)^{..} rho[r + 2^N c].
//  SV: <psi|P|psi> = i^{#Y} sum_j conj(psi_j) (-1)^{par(j1 & myz)} psi_{j1}, j1 = j ^ mxy;
//  real, so the imaginary part is 0 (NaN where the real part is no number).
constexpr uint64_t EXP_CHUNK = (uint64_t)BLOCK * 16;

template <typename R, bool DM>
__global__ __launch_bounds__(BLOCK) void k_pauli_expec(const cx<R>* __restrict__ a, unsigned nbits,
                                                       const PauliTermDev* __restrict__ terms,
                                                       unsigned chunks, double* __restrict__ part) {
    const unsigned t = blockIdx.x / chunks, c = blockIdx.x % chunks;
    const PauliTermDev term = terms[t];
    const uint64_t num = 1ULL << nbits;
    const uint64_t start = (uint64_t)c * EXP_CHUNK;
    const uint64_t end = start + EXP_CHUNK < num ? start + EXP_CHUNK : num;
    double vr = 0, vi = 0;
    for (uint64_t r = start + threadIdx.x; r < end; r += BLOCK) {
        uint64_t r1 = r ^ term.mxy;
        double sg = par64(r1 & term.myz) ? -1.0 : 1.0;
        if (DM) {
            cx<R> v = a[r + (r1 << nbits)];
            vr += sg * (double)v.x;
            vi += sg * (double)v.y;
        } else {
            cx<R> x = a[r], y = a[r1];
            vr += sg * ((double)x.x * (double)y.x + (double)x.y * (double)y.y);
            vi += sg * ((double)x.x * (double)y.y - (double)x.y * (double)y.x);
        }
    }
    block_sum2(vr, vi);
    if (threadIdx.x == 0) {
        const double re = term.fr * vr - term.fi * vi;
        part[2 * blockIdx.x] = re;
        part[2 * blockIdx.x + 1] = DM ? term.fr * vi + term.fi * vr : re - re;
    }
}

// One step of the adjoint reverse sweep for a parametrised gadget, in one pass
// over phi and lambda: the term <lambda| f P |phi>, then
// U^dag on both states with the arithmetic of k_pauli / k_pauli_diag / k_phase.
// Each pair (j, j ^ mxy) of both states is read once and written once.
// NT: streaming state access (ld_stream / st_stream) when every 128-byte line
// a wave touches is written whole by one store instruction (no X/Y bit inside
// a line)
template <typename R, bool NT>
__device__ __forceinline__ cx<R> adj_ld(const cx<R>* p) {
    if constexpr (NT) return ld_stream(p);
    else return *p;
}
template <typename R, bool NT>
__device__ __forceinline__ void adj_st(cx<R>* p, cx<R> v) {
    if constexpr (NT) st_stream(p, v);
    else *p = v;
}

// First block of a sweep kernel's grid-stride loop.  FP32 sweeps run 4-5%
// faster with each XCD on a contiguous eighth of the blocks (stream_block);
// FP64 ones 4-9% slower (24-qubit adjoint, same box), so they keep the
// round-robin order.
template <typename R>
__device__ __forceinline__ uint64_t adjoint_block() {
    if constexpr (sizeof(R) == 4) return stream_block();
    return blockIdx.x;
}

template <typename R, bool NT>
__global__ __launch_bounds__(BLOCK) void k_adjoint_step(cx<R>* __restrict__ phi, cx<R>* __restrict__ lam,
                                                        uint64_t numIts, unsigned hb, AdjointStepDev st,
                                                        double* __restrict__ rows, uint64_t stride) {
    const cx<R> th = mk<R>((R)st.thr, (R)st.thi), fe = mk<R>((R)st.fer, (R)st.fei);
    const cx<R> fo = mk<R>(-fe.x, -fe.y);
    const cx<R> e0 = mk<R>((R)st.e0r, (R)st.e0i), e1 = mk<R>((R)st.e1r, (R)st.e1i);
    double vr = 0, vi = 0;
    for (uint64_t k = adjoint_block<R>() * BLOCK + threadIdx.x; k < numIts; k += (uint64_t)gridDim.x * BLOCK) {
        if (st.mxy) {
            const uint64_t j0 = ins0(k, hb), j1 = j0 ^ st.mxy;
            const cx<R> p0 = adj_ld<R, NT>(phi + j0), p1 = adj_ld<R, NT>(phi + j1);
            const cx<R> l0 = adj_ld<R, NT>(lam + j0), l1 = adj_ld<R, NT>(lam + j1);
            const bool o0 = par64(j0 & st.myz) != 0, o1 = par64(j1 & st.myz) != 0;
            const double s0 = o0 ? -1.0 : 1.0, s1 = o1 ? -1.0 : 1.0;
            // conj(lambda_j) (-1)^{par(j' & myz)} phi_j' for j = j0 and j = j1
            vr += s1 * ((double)l0.x * (double)p1.x + (double)l0.y * (double)p1.y) +
                  s0 * ((double)l1.x * (double)p0.x + (double)l1.y * (double)p0.y);
            vi += s1 * ((double)l0.x * (double)p1.y - (double)l0.y * (double)p1.x) +
                  s0 * ((double)l1.x * (double)p0.y - (double)l1.y * (double)p0.x);
            const cx<R> f0 = o0 ? fo : fe, f1 = o1 ? fo : fe;
            adj_st<R, NT>(phi + j0, cfma(cmul(th, p0), f1, p1));
            adj_st<R, NT>(phi + j1, cfma(cmul(th, p1), f0, p0));
            adj_st<R, NT>(lam + j0, cfma(cmul(th, l0), f1, l1));
            adj_st<R, NT>(lam + j1, cfma(cmul(th, l1), f0, l0));
        } else {
            const cx<R> p = adj_ld<R, NT>(phi + k), l = adj_ld<R, NT>(lam + k);
            const bool odd = par64(k & st.myz) != 0;
            const double sg = odd ? -1.0 : 1.0;
            vr += sg * ((double)l.x * (double)p.x + (double)l.y * (double)p.y);
            vi += sg * ((double)l.x * (double)p.y - (double)l.y * (double)p.x);
            if (st.phase) {
                const cx<R> f = odd ? e1 : e0;
                adj_st<R, NT>(phi + k, cmul(p, f));
                adj_st<R, NT>(lam + k, cmul(l, f));
            } else {
                const cx<R> f = odd ? fo : fe;
                adj_st<R, NT>(phi + k, cfma(cmul(th, p), f, p));
                adj_st<R, NT>(lam + k, cfma(cmul(th, l), f, l));
            }
        }
    }
    block_sum2(vr, vi);
    if (threadIdx.x == 0) {
        double* row = rows + stride * st.slot + 2 * blockIdx.x;
        row[0] = st.fr * vr - st.fi * vi;
        row[1] = st.fr * vi + st.fi * vr;
    }
}

// A run of diagonal gadgets (AdjointDiagDev): conj(lambda_k) phi_k is formed
// once per amplitude and added, with gadget g's parity sign, to g's FP64
// accumulators; both states are multiplied by the product of the gadgets'
// U^dag factors, looked up by the amplitude's parity pattern (bit g = parity
// of gadget g) in a table each block builds in LDS.  Each accumulator then
// takes the same two-level reduction as k_adjoint_step: block sums here (one
// row per workgroup in the gadget's slot), then k_grad_sums.  This kernel and
// the two below serve the states too small for register-tile passes
// (sweep_min_qubits), where a launch is what counts.
template <typename R>
__global__ __launch_bounds__(BLOCK) void k_adjoint_diag(cx<R>* __restrict__ phi, cx<R>* __restrict__ lam,
                                                        uint64_t num, AdjointDiagDev st, double* __restrict__ rows,
                                                        uint64_t stride) {
    __shared__ cx<R> tab[1u << ADJ_DIAG_MAX];
    const unsigned cnt = st.count;
    for (unsigned t = threadIdx.x; t < (1u << cnt); t += BLOCK) {
        cx<R> f = mk<R>((R)1, (R)0);
        for (unsigned g = 0; g < cnt; g++)
            f = cmul(f, ((t >> g) & 1u) ? mk<R>((R)st.e1r[g], (R)st.e1i[g]) : mk<R>((R)st.e0r[g], (R)st.e0i[g]));
        tab[t] = f;
    }
    __syncthreads();
    double vr[ADJ_DIAG_MAX], vi[ADJ_DIAG_MAX];
#pragma unroll
    for (unsigned g = 0; g < ADJ_DIAG_MAX; g++) { vr[g] = 0; vi[g] = 0; }
    for (uint64_t k = (uint64_t)blockIdx.x * BLOCK + threadIdx.x; k < num; k += (uint64_t)gridDim.x * BLOCK) {
        const cx<R> p = phi[k], l = lam[k];
        const double wr = (double)l.x * (double)p.x + (double)l.y * (double)p.y;
        const double wi = (double)l.x * (double)p.y - (double)l.y * (double)p.x;
        unsigned pat = 0;
#pragma unroll
        for (unsigned g = 0; g < ADJ_DIAG_MAX; g++) {
            if (g < cnt) {
                const unsigned odd = par32((uint32_t)k & (uint32_t)st.myz[g]);
                pat |= odd << g;
                vr[g] += odd ? -wr : wr;
                vi[g] += odd ? -wi : wi;
            }
        }
        const cx<R> f = tab[pat];
        phi[k] = cmul(p, f);
        lam[k] = cmul(l, f);
    }
#pragma unroll
    for (unsigned g = 0; g < ADJ_DIAG_MAX; g++) {
        if (g < cnt) {
            double a = vr[g], b = vi[g];
            block_sum2(a, b);
            if (threadIdx.x == 0) {
                double* row = rows + stride * st.slot[g] + 2 * blockIdx.x;
                row[0] = st.fr[g] * a - st.fi[g] * b;
                row[1] = st.fr[g] * b + st.fi[g] * a;
            }
            __syncthreads();    // block_sum2's wave partials are reused by the next gadget
        }
    }
}

// A run of G one-qubit X/Y gadgets on distinct qubits (AdjointQubitRunDev):
// each thread takes groups of 2^G amplitudes of phi and lambda (bit g of the
// group index = gadget g's qubit), adds every gadget's term from the loaded
// values (conj(lambda_j) s(j') phi_j' over its pairs j' = j ^ bit, as in
// k_adjoint_step), then applies every gadget's U^dag to its pairs and writes
// the group back.  Reduction as in k_adjoint_diag.
template <typename R, int G>
__global__ __launch_bounds__(BLOCK) void k_adjoint_qrun(cx<R>* __restrict__ phi, cx<R>* __restrict__ lam,
                                                        uint64_t numGroups, AdjointQubitRunDev st,
                                                        double* __restrict__ rows, uint64_t stride) {
    constexpr unsigned E = 1u << G;
    double vr[G], vi[G];
#pragma unroll
    for (int g = 0; g < G; g++) { vr[g] = 0; vi[g] = 0; }
    uint64_t off[E];
#pragma unroll
    for (unsigned e = 0; e < E; e++) {
        off[e] = 0;
#pragma unroll
        for (int g = 0; g < G; g++) if ((e >> g) & 1u) off[e] |= 1ULL << st.q[g];
    }
    for (uint64_t t = (uint64_t)blockIdx.x * BLOCK + threadIdx.x; t < numGroups; t += (uint64_t)gridDim.x * BLOCK) {
        uint64_t x = t;
#pragma unroll
        for (int i = 0; i < G; i++) x = ins0(x, st.sorted[i]);
        cx<R> p[E], l[E];
#pragma unroll
        for (unsigned e = 0; e < E; e++) { p[e] = phi[x | off[e]]; l[e] = lam[x | off[e]]; }
#pragma unroll
        for (int g = 0; g < G; g++) {
            // s(j) = -1 where the gadget is Y and j has its qubit set (the pair's second element)
            const double s1 = st.y[g] ? -1.0 : 1.0;
#pragma unroll
            for (unsigned e = 0; e < E; e++) {
                if ((e >> g) & 1u) continue;
                const unsigned e1 = e | (1u << g);
                vr[g] += s1 * ((double)l[e].x * (double)p[e1].x + (double)l[e].y * (double)p[e1].y) +
                         ((double)l[e1].x * (double)p[e].x + (double)l[e1].y * (double)p[e].y);
                vi[g] += s1 * ((double)l[e].x * (double)p[e1].y - (double)l[e].y * (double)p[e1].x) +
                         ((double)l[e1].x * (double)p[e].y - (double)l[e1].y * (double)p[e].x);
            }
        }
#pragma unroll
        for (int g = 0; g < G; g++) {
            const cx<R> th = mk<R>((R)st.thr[g], (R)st.thi[g]), fe = mk<R>((R)st.fer[g], (R)st.fei[g]);
            const cx<R> f1 = st.y[g] ? mk<R>(-fe.x, -fe.y) : fe;    // factor of the element with the qubit set
#pragma unroll
            for (unsigned e = 0; e < E; e++) {
                if ((e >> g) & 1u) continue;
                const unsigned e1 = e | (1u << g);
                const cx<R> p0 = p[e], p1 = p[e1], l0 = l[e], l1 = l[e1];
                p[e] = cfma(cmul(th, p0), f1, p1);
                p[e1] = cfma(cmul(th, p1), fe, p0);
                l[e] = cfma(cmul(th, l0), f1, l1);
                l[e1] = cfma(cmul(th, l1), fe, l0);
            }
        }
#pragma unroll
        for (unsigned e = 0; e < E; e++) { phi[x | off[e]] = p[e]; lam[x | off[e]] = l[e]; }
    }
#pragma unroll
    for (int g = 0; g < G; g++) {
        double a = vr[g], b = vi[g];
        block_sum2(a, b);
        if (threadIdx.x == 0) {
            double* row = rows + stride * st.slot[g] + 2 * blockIdx.x;
            row[0] = st.fr[g] * a - st.fi[g] * b;
            row[1] = st.fr[g] * b + st.fi[g] * a;
        }
        __syncthreads();    // block_sum2's wave partials are reused by the next gadget
    }
}

template <typename R>
__device__ __forceinline__ cx<R> shfl_xor_cx(cx<R> v, int m) {
    return mk<R>(__shfl_xor(v.x, m, 64), __shfl_xor(v.y, m, 64));
}

// The same run when every qubit of it is below 6: lane l of a wave holds
// amplitude base + l of phi and lambda (whole 64-amplitude blocks, so every
// line is read whole), and the partner j ^ bit comes from lane l ^ bit.  Each
// element adds conj(lambda_j) s(j') phi_j' (j' = j ^ bit, s(j') = -1 for a Y
// gadget when j' has the bit set), which over a pair is k_adjoint_step's
// term; then each gadget in turn maps v_j <- th v_j + s(j') fe v_j'.
// DG: the diagonal run that follows in the sweep (dg, 1..ADJ_DIAG_MAX gadgets)
// is applied in the same pass, after the run, as k_adjoint_diag does it: its
// terms from the updated amplitudes, then its factors from an LDS table.
template <typename R, int G, bool DG>
__global__ __launch_bounds__(BLOCK) void k_adjoint_qrun_lane(cx<R>* __restrict__ phi, cx<R>* __restrict__ lam,
                                                             uint64_t num, AdjointQubitRunDev st, AdjointDiagDev dg,
                                                             double* __restrict__ rows, uint64_t stride) {
    __shared__ cx<R> tab[DG ? 1u << ADJ_DIAG_MAX : 1u];
    const unsigned cnt = DG ? dg.count : 0u;
    if constexpr (DG) {
        for (unsigned t = threadIdx.x; t < (1u << cnt); t += BLOCK) {
            cx<R> f = mk<R>((R)1, (R)0);
            for (unsigned g = 0; g < cnt; g++)
                f = cmul(f, ((t >> g) & 1u) ? mk<R>((R)dg.e1r[g], (R)dg.e1i[g]) : mk<R>((R)dg.e0r[g], (R)dg.e0i[g]));
            tab[t] = f;
        }
        __syncthreads();
    }
    constexpr int DM = DG ? (int)ADJ_DIAG_MAX : 1;
    double vr[G], vi[G], dr[DM], di[DM];
#pragma unroll
    for (int g = 0; g < G; g++) { vr[g] = 0; vi[g] = 0; }
#pragma unroll
    for (int g = 0; g < DM; g++) { dr[g] = 0; di[g] = 0; }
    // num is a multiple of 64 and so is the stride: a wave's lanes stay together
    for (uint64_t j = (uint64_t)blockIdx.x * BLOCK + threadIdx.x; j < num; j += (uint64_t)gridDim.x * BLOCK) {
        cx<R> p = phi[j], l = lam[j];
#pragma unroll
        for (int g = 0; g < G; g++) {
            const cx<R> pp = shfl_xor_cx(p, 1 << st.q[g]);
            const bool partnerSet = ((j >> st.q[g]) & 1ULL) == 0;
            const double sg = (st.y[g] && partnerSet) ? -1.0 : 1.0;
            vr[g] += sg * ((double)l.x * (double)pp.x + (double)l.y * (double)pp.y);
            vi[g] += sg * ((double)l.x * (double)pp.y - (double)l.y * (double)pp.x);
        }
#pragma unroll
        for (int g = 0; g < G; g++) {
            const int m = 1 << st.q[g];
            const cx<R> pp = shfl_xor_cx(p, m), lp = shfl_xor_cx(l, m);
            const bool partnerSet = ((j >> st.q[g]) & 1ULL) == 0;
            const cx<R> th = mk<R>((R)st.thr[g], (R)st.thi[g]);
            const cx<R> fe = mk<R>((R)st.fer[g], (R)st.fei[g]);
            const cx<R> f = (st.y[g] && partnerSet) ? mk<R>(-fe.x, -fe.y) : fe;
            p = cfma(cmul(th, p), f, pp);
            l = cfma(cmul(th, l), f, lp);
        }
        if constexpr (DG) {
            const double wr = (double)l.x * (double)p.x + (double)l.y * (double)p.y;
            const double wi = (double)l.x * (double)p.y - (double)l.y * (double)p.x;
            unsigned pat = 0;
#pragma unroll
            for (unsigned g = 0; g < ADJ_DIAG_MAX; g++) {
                if (g < cnt) {
                    const unsigned odd = par32((uint32_t)j & (uint32_t)dg.myz[g]);
                    pat |= odd << g;
                    dr[g] += odd ? -wr : wr;
                    di[g] += odd ? -wi : wi;
                }
            }
            const cx<R> fd = tab[pat];
            p = cmul(p, fd);
            l = cmul(l, fd);
        }
        phi[j] = p;
        lam[j] = l;
    }
#pragma unroll
    for (int g = 0; g < G; g++) {
        double a = vr[g], b = vi[g];
        block_sum2(a, b);
        if (threadIdx.x == 0) {
            double* row = rows + stride * st.slot[g] + 2 * blockIdx.x;
            row[0] = st.fr[g] * a - st.fi[g] * b;
            row[1] = st.fr[g] * b + st.fi[g] * a;
        }
        __syncthreads();    // block_sum2's wave partials are reused by the next gadget
    }
    if constexpr (DG) {
#pragma unroll
        for (unsigned g = 0; g < ADJ_DIAG_MAX; g++) {
            if (g < cnt) {
                double a = dr[g], b = di[g];
                block_sum2(a, b);
                if (threadIdx.x == 0) {
                    double* row = rows + stride * dg.slot[g] + 2 * blockIdx.x;
                    row[0] = dg.fr[g] * a - dg.fi[g] * b;
                    row[1] = dg.fr[g] * b + dg.fi[g] * a;
                }
                __syncthreads();
            }
        }
    }
}

// Register-tile pass (wave_sweep.hpp): REV over phi and lambda, else over phi.
// Gradient terms accumulate per thread in LDS, two gadgets to a row: lanes
// below 32 keep the first gadget's sum of lanes l and l + 32, the others the
// second's, so one exchange folds both and a row of 256 doubles serves two.
// Three workgroups of four waves per CU (VGPRs and LDS): more waves hide more
// of the loads and of the scalar work between ops.
// 20 layers of ZZ and X gadgets, 24 qubits FP64: 35 reverse passes of 310 us (210 us of
// them the bare loads and stores, against 160 run passes of 197 us and 40
// diagonal passes of 193 us), 26 forward passes of 140 us (against 19 LDS tile
// passes of 602 us); FP32: 36 of 237 us and 23 of 89 us.  Bound by vector
// instructions (the vector unit is busy 62% and 54% of the time in FP64, 77% and
// 87% in FP32).  Exchanges through LDS instead of DPP moves and layout changes
// took 375 us a reverse pass, diagonal gadgets one by one and rotations without
// shears 336 us.
template <typename R, int G, bool REV>
__global__ __launch_bounds__(BLOCK, 3) void k_wave_sweep(cx<R>* __restrict__ phi, cx<R>* __restrict__ lam,
                                                         uint64_t numTiles, SweepGeom geom,
                                                         const SweepOp* __restrict__ ops, unsigned numOps,
                                                         unsigned numGrads, double* __restrict__ rows, uint64_t stride) {
    constexpr int S = 1 << G;
    __shared__ double acc[REV ? SWEEP_MAX_GRADS / 2 : 1][BLOCK];
    const uint32_t tid = threadIdx.x, lane = tid & 63u;
    const bool upper = lane >= 32u;
    if constexpr (REV)
        for (unsigned k = 0; k < (numGrads + 1) / 2; k++) acc[k][tid] = 0;
    // The offset of this lane's amplitudes, computed anew for the loads and the
    // stores of a tile: the empty register constraint hides that the two agree,
    // or the compiler would keep all of a tile's addresses alive through its ops.
    auto lane_offset = [&](const uint8_t* q) {
        float bits = __builtin_bit_cast(float, lane);
        asm volatile("" : "+v"(bits));
        const uint32_t l = __builtin_bit_cast(uint32_t, bits);
        uint64_t off = 0;
#pragma unroll
        for (unsigned b = 0; b < SWEEP_LANE_BITS; b++) off |= (uint64_t)((l >> b) & 1u) << q[b];
        return off;
    };
    auto at = [&](uint64_t base, const uint8_t* q, int i) {
#pragma unroll
        for (int b = 0; b < G; b++) if ((i >> b) & 1) base |= 1ULL << q[b];
        return base;
    };
    touched(touch_lines<BLOCK>(ops, (size_t)numOps * sizeof(SweepOp)));
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint64_t first = adjoint_block<R>() * (BLOCK / 64) + wave, step = (uint64_t)gridDim.x * (BLOCK / 64);
    for (uint64_t t = first; t < numTiles; t += step) {
        const uint64_t base = ins0_mask(t, geom.tileMask), in = lane_offset(geom.lane);
        sweep::Tile<R, S> v;
#pragma unroll
        for (int i = 0; i < S; i++) {
            const cx<R> p = adj_ld<R, true>(phi + at(base, geom.reg, i) + in);
            v.px[i] = p.x; v.py[i] = p.y;
            if constexpr (REV) {
                const cx<R> l = adj_ld<R, true>(lam + at(base, geom.reg, i) + in);
                v.lx[i] = l.x; v.ly[i] = l.y;
            }
        }
        auto header = [&](unsigned o) {
            SweepOp h;
            h.code = ops[o].code; h.lz = ops[o].lz; h.sw = ops[o].sw; h.flags = ops[o].flags;
            h.oz = ops[o].oz; h.c = ops[o].c; h.g = ops[o].g;
            return h;
        };
        SweepOp hdr = header(0);
        double held = 0;                                    // the even gadget's term of the current row
        double dsum = 0, dc = 1, dg = 0;                    // the current diagonal group's sum and factor
        for (unsigned o = 0; o < numOps; o++) {
            const SweepOp next = header(o + 1 < numOps ? o + 1 : o);     // loads while this op runs
            // lane and tile part of the sign
            const uint32_t sb = (par32((lane | SWEEP_CONST_SIGN) & hdr.lz) ^ par64(base & hdr.oz)) << 31;
            double w;
            if (hdr.code < SWEEP_LANE) {
                const bool ss = (hdr.code & 1u) != 0;
                const double g = sweep::flip(hdr.g, sb);
                if constexpr (REV) {
                    if (hdr.flags & SWEEP_GROUP_FIRST)
                        dsum = ss ? sweep::diag_sum<R, S, true>(v, hdr.sw) : sweep::diag_sum<R, S, false>(v, hdr.sw);
                }
                w = sweep::flip(dsum, sb);
                if (hdr.code >= SWEEP_DIAG_ONE) {
                    const R T = (R)(sweep::sweep_shears<R, REV>() ? sweep::flip(hdr.c, sb) : hdr.c);
                    if (ss) sweep::op_diag<R, S, REV, true, true>(v, T, (R)g, hdr.sw);
                    else sweep::op_diag<R, S, REV, true, false>(v, T, (R)g, hdr.sw);
                } else {
                    if (hdr.flags & SWEEP_GROUP_FIRST) { dc = 1; dg = 0; }
                    const double c = dc * hdr.c - dg * g;
                    dg = dc * g + dg * hdr.c;
                    dc = c;
                    if (hdr.flags & SWEEP_GROUP_LAST) {
                        if (ss) sweep::op_diag<R, S, REV, false, true>(v, (R)dc, (R)dg, hdr.sw);
                        else sweep::op_diag<R, S, REV, false, false>(v, (R)dc, (R)dg, hdr.sw);
                    }
                }
            } else {
                w = sweep::apply<R, G, REV>(v, hdr, ops + o, lane, base, sb);
            }
            if constexpr (REV) {
                if (hdr.flags & SWEEP_GRAD_EVEN) {
                    held = w;
                } else if (hdr.flags & SWEEP_GRAD_ODD) {
                    const double other = __shfl_xor(upper ? held : w, 32, 64);
                    acc[ops[o].row][tid] += (upper ? w : held) + other;
                }
            }
            hdr = next;
        }
        if constexpr (REV) {
            if (numGrads & 1u) {                            // a last gadget on its own
                const double other = __shfl_xor(upper ? held : 0.0, 32, 64);
                acc[numGrads / 2][tid] += (upper ? 0.0 : held) + other;
            }
        }
        const uint64_t out = lane_offset(geom.laneOut);
#pragma unroll
        for (int i = 0; i < S; i++) {
            adj_st<R, true>(phi + at(base, geom.regOut, i) + out, mk<R>(v.px[i], v.py[i]));
            if constexpr (REV) adj_st<R, true>(lam + at(base, geom.regOut, i) + out, mk<R>(v.lx[i], v.ly[i]));
        }
    }
    if constexpr (REV) {
        // workgroup sums: gadget 2 k in the lower, 2 k + 1 in the upper lanes of row k
        unsigned k = 0;
        for (unsigned o = 0; o < numOps; o++) {
            if (!(ops[o].flags & (SWEEP_GRAD_EVEN | SWEEP_GRAD_ODD))) continue;
            const double a = acc[k / 2][tid];
            double im = upper == ((k & 1u) != 0) ? a : 0.0, dummy = 0;
            block_sum2(im, dummy);
            if (tid == 0) {
                double* row = rows + stride * ops[o].slot + 2 * blockIdx.x;
                row[0] = 0;
                row[1] = im;
            }
            __syncthreads();    // block_sum2's wave partials are reused by the next gadget
            k++;
        }
    }
}

// out[j] = sum_t f_t (-1)^{par(j1 & myz_t)} in[j1], j1 = j ^ mxy_t
template <typename R>
__global__ __launch_bounds__(BLOCK) void k_apply_pauli_terms(const cx<R>* __restrict__ in, cx<R>* __restrict__ out,
                                                             uint64_t num, const PauliTermDev* __restrict__ terms,
                                                             unsigned numTerms) {
    const uint64_t j = (uint64_t)blockIdx.x * BLOCK + threadIdx.x;
    if (j >= num) return;
    double ar = 0, ai = 0;
    for (unsigned t = 0; t < numTerms; t++) {
        const PauliTermDev term = terms[t];
        uint64_t j1 = j ^ term.mxy;
        double sg = par64(j1 & term.myz) ? -1.0 : 1.0;
        cx<R> v = in[j1];
        double fr = sg * term.fr, fi = sg * term.fi;
        ar += fr * (double)v.x - fi * (double)v.y;
        ai += fr * (double)v.y + fi * (double)v.x;
    }
    out[j] = mk<R>((R)ar, (R)ai);
}

// A Pauli sum H on a statevector, grouped by X/Y mask (PauliGroupDev): either
// <psi|H|psi> (EXPEC, one partial per workgroup) or out = H psi.  A thread owns
// ITEMS amplitudes j = chunk base + 256 i + tid and walks the groups: it takes
// psi_{j ^ mxy} once per group, sums the group's coefficients with their signs,
// and multiplies once.  Signs split into a part fixed for the workgroup, a part
// of the lane and a part of i, so a term costs one lane parity however many
// amplitudes a thread owns.  Groups that agree above the chunk read the same
// other chunk, which goes to LDS once for all of them; a group that is alone
// there is loaded straight into registers.
//   EXPEC keeps psi_j in registers for all groups.  A Pauli string with a real
// coefficient is Hermitian, so the pair (j, j ^ mxy) contributes twice the real
// part of one of its two products: groups whose top X/Y qubit lies above the
// chunk are taken on half of the chunks only, which halves their loads.  The
// imaginary part is 0 (NaN where the real part is no number).
//   What bounds it: loads from the Infinity Cache and L2 (24 qubits FP64: one
// 256 MiB read per group run).  24 qubits, 100 random strings of
// weight 1-4: <H> 6.19 -> 0.65 ms, H psi 1.82 -> 1.12 ms against one pass per
// term (which left 409600 partials to one workgroup); without the LDS copy of
// shared chunks 0.82 and 1.45 ms.
template <typename R, bool EXPEC>
__global__ __launch_bounds__(BLOCK) void k_pauli_groups(const cx<R>* __restrict__ a, cx<R>* __restrict__ out,
                                                        uint64_t num, const PauliGroupDev* __restrict__ groups,
                                                        const PauliSignDev* __restrict__ terms, unsigned numGroups,
                                                        double* __restrict__ part) {
    constexpr uint64_t CHUNK = 1ULL << PAULI_CHUNK_BITS;
    constexpr int ITEMS = (int)(CHUNK / BLOCK);
    __shared__ cx<R> other[CHUNK];
    const uint32_t tid = threadIdx.x;
    double v = 0;
    for (uint64_t base = (uint64_t)blockIdx.x * CHUNK; base < num; base += (uint64_t)gridDim.x * CHUNK) {
        cx<R> x[ITEMS];
        double ar[ITEMS], ai[ITEMS];
#pragma unroll
        for (int i = 0; i < ITEMS; i++) {
            if constexpr (EXPEC) x[i] = a[base + (uint32_t)i * BLOCK + tid];
            else ar[i] = ai[i] = 0;
        }
        // amplitude of item i under group gr is element ((i ^ mi) * BLOCK + (tid ^ mxy)) of chunk base ^ mxy
        auto item_mask = [&](uint64_t m) { return ((uint32_t)m / BLOCK) & (uint32_t)(ITEMS - 1); };
        auto add_group = [&](const PauliGroupDev& gr, const cx<R> (&y)[ITEMS], double weight) {
            const uint64_t hi = base ^ (gr.mxy & ~(CHUNK - 1));
            const uint32_t mi = item_mask(gr.mxy);
            const uint32_t l = (tid ^ (uint32_t)gr.mxy) & (BLOCK - 1u);
            double c[ITEMS];
#pragma unroll
            for (int i = 0; i < ITEMS; i++) c[i] = 0;
            for (uint32_t t = gr.t0; t < gr.t1; t++) {
                const PauliSignDev term = terms[t];
                const uint32_t odd = par64(hi & term.myz) ^ par32(l & (uint32_t)term.myz & (BLOCK - 1u));
                const double cl = odd ? -term.c : term.c;
                const uint32_t mz = item_mask(term.myz);
#pragma unroll
                for (int i = 0; i < ITEMS; i++) c[i] += par32(((uint32_t)i ^ mi) & mz) ? -cl : cl;
            }
#pragma unroll
            for (int i = 0; i < ITEMS; i++) {
                const double yx = (double)y[i].x, yy = (double)y[i].y;
                if constexpr (EXPEC) {
                    // Re(conj(x) y) for a real factor, Re(i conj(x) y) for an imaginary one
                    const double xx = (double)x[i].x, xy = (double)x[i].y;
                    v += weight * c[i] * (gr.imag ? xy * yx - xx * yy : xx * yx + xy * yy);
                } else {
                    ar[i] += gr.imag ? -c[i] * yy : c[i] * yx;
                    ai[i] += gr.imag ? c[i] * yx : c[i] * yy;
                }
            }
        };
        for (unsigned g = 0; g < numGroups;) {
            const PauliGroupDev gr = groups[g];
            const unsigned run = gr.run;
            double weight = 1.0;
            if (EXPEC && gr.mxy >= CHUNK) {      // the pairs' other halves are in another chunk
                weight = 2.0;
                if ((base >> (63 - __builtin_clzll(gr.mxy))) & 1ULL) { g += run; continue; }
            }
            const cx<R>* src = a + (base ^ (gr.mxy & ~(CHUNK - 1)));
            cx<R> y[ITEMS];
            if (run == 1) {
                const uint32_t mi = item_mask(gr.mxy), l = (tid ^ (uint32_t)gr.mxy) & (BLOCK - 1u);
#pragma unroll
                for (int i = 0; i < ITEMS; i++) y[i] = src[((uint32_t)i ^ mi) * BLOCK + l];
                add_group(gr, y, weight);
                g++;
                continue;
            }
#pragma unroll
            for (int i = 0; i < ITEMS; i++) y[i] = src[(uint32_t)i * BLOCK + tid];
            __syncthreads();                     // the previous run has been read
#pragma unroll
            for (int i = 0; i < ITEMS; i++) other[(uint32_t)i * BLOCK + tid] = y[i];
            __syncthreads();
            for (const unsigned end = g + run; g < end; g++) {
                const PauliGroupDev gi = groups[g];
                const uint32_t mi = item_mask(gi.mxy), l = (tid ^ (uint32_t)gi.mxy) & (BLOCK - 1u);
#pragma unroll
                for (int i = 0; i < ITEMS; i++) y[i] = other[((uint32_t)i ^ mi) * BLOCK + l];
                add_group(gi, y, weight);
            }
        }
        if constexpr (!EXPEC) {
#pragma unroll
            for (int i = 0; i < ITEMS; i++)
                out[base + (uint32_t)i * BLOCK + tid] = mk<R>((R)ar[i], (R)ai[i]);
        }
    }
    if constexpr (EXPEC) {
        double im = 0;
        block_sum2(v, im);
        if (tid == 0) { part[2 * blockIdx.x] = v; part[2 * blockIdx.x + 1] = v - v; }
    }
}

struct TargetList { uint32_t t[32]; uint32_t k; };

// reference local_densitymatrix.hpp:134-164 (setBit defect corrected)
template <typename R>
__global__ __launch_bounds__(BLOCK) void k_partial_trace(const cx<R>* __restrict__ in, cx<R>* __restrict__ out,
                                                         uint64_t numOut, unsigned N, uint64_t allMask,
                                                         TargetList tl) {
    const uint64_t l = (uint64_t)blockIdx.x * BLOCK + threadIdx.x;
    if (l >= numOut) return;
    const uint64_t lm = ins0_mask(l, allMask);
    cx<R> acc = mk<R>(0, 0);
    const uint64_t numTraced = 1ULL << tl.k;
    for (uint64_t kk = 0; kk < numTraced; kk++) {
        uint64_t i = lm;
        for (unsigned b = 0; b < tl.k; b++)
            if ((kk >> b) & 1) i |= (1ULL << tl.t[b]) | (1ULL << (tl.t[b] + N));
        acc = cadd(acc, in[i]);
    }
    out[l] = acc;
}

// ---- initialisation ----------------------------------------------------------

__device__ __forceinline__ uint64_t mix64(uint64_t z) {
    z += 0x9E3779B97F4A7C15ULL;
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ULL;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBULL;
    return z ^ (z >> 31);
}

__device__ __forceinline__ double unit_open(uint64_t key, uint64_t c) {
    return ((double)(mix64(key + c) >> 11) + 0.5) * (1.0 / 9007199254740992.0);
}

template <typename R>
__global__ __launch_bounds__(BLOCK) void k_gaussian(cx<R>* __restrict__ a, uint64_t num, uint64_t key) {
    for (uint64_t j = (uint64_t)blockIdx.x * BLOCK + threadIdx.x; j < num; j += (uint64_t)gridDim.x * BLOCK) {
        double u1 = unit_open(key, 2 * j), u2 = unit_open(key, 2 * j + 1);
        double r = sqrt(-2.0 * log(u1));
        double ph = 6.283185307179586476925286766559 * u2;
        a[j] = mk<R>((R)(r * cos(ph)), (R)(r * sin(ph)));
    }
}

template <typename R>
__global__ __launch_bounds__(BLOCK) void k_scale_inv_sqrt(cx<R>* __restrict__ a, uint64_t num,
                                                          const double* __restrict__ norm2) {
    const double f = norm2[0] > 0 ? 1.0 / sqrt(norm2[0]) : 1.0;   // a zero vector stays zero
    for (uint64_t j = (uint64_t)blockIdx.x * BLOCK + threadIdx.x; j < num; j += (uint64_t)gridDim.x * BLOCK) {
        cx<R> v = a[j];
        a[j] = mk<R>((R)((double)v.x * f), (R)((double)v.y * f));
    }
}

template <typename R>
__global__ __launch_bounds__(BLOCK) void k_basis(cx<R>* __restrict__ a, uint64_t num, uint64_t index) {
    for (uint64_t j = (uint64_t)blockIdx.x * BLOCK + threadIdx.x; j < num; j += (uint64_t)gridDim.x * BLOCK)
        a[j] = mk<R>((R)(j == index ? 1 : 0), (R)0);
}

__global__ __launch_bounds__(BLOCK) void k_f64_to_f32(const cx<double>* __restrict__ in, cx<float>* __restrict__ out,
                                                      uint64_t num) {
    for (uint64_t j = (uint64_t)blockIdx.x * BLOCK + threadIdx.x; j < num; j += (uint64_t)gridDim.x * BLOCK)
        out[j] = mk<float>((float)in[j].x, (float)in[j].y);
}

__global__ __launch_bounds__(BLOCK) void k_f32_to_f64(const cx<float>* __restrict__ in, cx<double>* __restrict__ out,
                                                      uint64_t num) {
    for (uint64_t j = (uint64_t)blockIdx.x * BLOCK + threadIdx.x; j < num; j += (uint64_t)gridDim.x * BLOCK)
        out[j] = mk<double>((double)in[j].x, (double)in[j].y);
}

unsigned grid_stride_blocks(uint64_t num) {
    uint64_t b = (num + BLOCK - 1) / BLOCK;
    if (b > 65536) b = 65536;
    return (unsigned)(b ? b : 1);
}

}  // namespace

uint64_t reduce_workspace_doubles(uint64_t num) {
    (void)num;
    return 2ULL * RED_MAX_BLOCKS;
}

template <typename R>
void launch_norm2(hipStream_t s, const cx<R>* a, uint64_t num, double* ws, double* dout) {
    unsigned nb = red_blocks(num);
    hipLaunchKernelGGL(k_norm2<R>, dim3(nb), dim3(BLOCK), 0, s, a, num, ws);
    hipLaunchKernelGGL(k_final_sum, dim3(1), dim3(BLOCK), 0, s, ws, nb, dout);
}

template <typename R>
void launch_inner(hipStream_t s, const cx<R>* a, const cx<R>* b, uint64_t num, double* ws, double* dout) {
    unsigned nb = red_blocks(num);
    hipLaunchKernelGGL(k_inner<R>, dim3(nb), dim3(BLOCK), 0, s, a, b, num, ws);
    hipLaunchKernelGGL(k_final_sum, dim3(1), dim3(BLOCK), 0, s, ws, nb, dout);
}

uint64_t adjoint_row_stride(unsigned nq) { return 2ULL * red_blocks(1ULL << nq); }

void launch_grad_sums(hipStream_t s, const double* rows, uint64_t stride, const uint32_t* nb, unsigned numSlots,
                      double* res) {
    if (numSlots) hipLaunchKernelGGL(k_grad_sums, dim3(numSlots), dim3(BLOCK), 0, s, rows, stride, nb, res);
}

template <typename R>
unsigned launch_adjoint_step(hipStream_t s, cx<R>* phi, cx<R>* lam, unsigned nq, const AdjointStepDev& st,
                             double* rows, uint64_t stride) {
    const uint64_t numIts = st.mxy ? 1ULL << (nq - 1) : 1ULL << nq;
    const unsigned hb = st.mxy ? 63u - (unsigned)__builtin_clzll(st.mxy) : 0u;
    unsigned nb = red_blocks(numIts);
    const uint64_t lineBits = 128 / sizeof(cx<R>) - 1;
    auto* kern = (st.mxy & lineBits) ? k_adjoint_step<R, false> : k_adjoint_step<R, true>;
    hipLaunchKernelGGL(kern, dim3(nb), dim3(BLOCK), 0, s, phi, lam, numIts, hb, st, rows, stride);
    return nb;
}

template <typename R>
unsigned launch_adjoint_diag(hipStream_t s, cx<R>* phi, cx<R>* lam, unsigned nq, const AdjointDiagDev& st,
                             double* rows, uint64_t stride) {
    if (nq > 32) fail(FSA_ERR_INTERNAL, "adjoint run of diagonal gadgets on more than 32 qubits");
    const uint64_t num = 1ULL << nq;
    const unsigned nb = red_blocks(num);
    hipLaunchKernelGGL(k_adjoint_diag<R>, dim3(nb), dim3(BLOCK), 0, s, phi, lam, num, st, rows, stride);
    return nb;
}

template <typename R>
unsigned launch_adjoint_qrun(hipStream_t s, cx<R>* phi, cx<R>* lam, unsigned nq, const AdjointQubitRunDev& st,
                             double* rows, uint64_t stride, const AdjointDiagDev* tail) {
    const unsigned G = st.count;
    if (G < 2 || G > ADJ_QRUN_MAX || nq < G || nq > 32) fail(FSA_ERR_INTERNAL, "adjoint qubit run of unsupported length");
    const uint64_t numGroups = 1ULL << (nq - G);
    uint64_t bits = 0;
    for (unsigned g = 0; g < G; g++) bits |= 1ULL << st.q[g];
    if (bits < 64 && nq >= 6) {
        // every qubit of the run inside a wave's 64 consecutive amplitudes
        const uint64_t num = 1ULL << nq;
        const unsigned nbl = red_blocks(num);
        AdjointDiagDev dg;
        std::memset(&dg, 0, sizeof(dg));
        if (tail) dg = *tail;
#define FSA_QL(GV, DGV)                                                                                          \
        hipLaunchKernelGGL((k_adjoint_qrun_lane<R, GV, DGV>), dim3(nbl), dim3(BLOCK), 0, s, phi, lam, num, st, dg, \
                           rows, stride)
        if (G == 2) {
            if (tail) FSA_QL(2, true);
            else FSA_QL(2, false);
        } else {
            if (tail) FSA_QL(3, true);
            else FSA_QL(3, false);
        }
#undef FSA_QL
        return nbl;
    }
    if (tail) fail(FSA_ERR_INTERNAL, "a diagonal tail needs a qubit run below qubit 6");
    const unsigned nb = red_blocks(numGroups);
#define FSA_QR(GV)                                                                                                 \
    if (G == GV)                                                                                                   \
        hipLaunchKernelGGL((k_adjoint_qrun<R, GV>), dim3(nb), dim3(BLOCK), 0, s, phi, lam, numGroups, st, rows, stride);
    FSA_QR(2) FSA_QR(3)
#undef FSA_QR
    return nb;
}

// three (rev) or four workgroups per CU, as many as its registers allow; never more than
// red_blocks(2^nq) rows (a workgroup's four tiles hold 2^11 amplitudes or more)
template <typename R>
unsigned launch_sweep(hipStream_t s, bool rev, cx<R>* phi, cx<R>* lam, unsigned nq, const SweepGeom& geom,
                      const SweepOp* dops, unsigned numOps, unsigned numGrads, double* rows, uint64_t stride) {
    const unsigned M = SWEEP_LANE_BITS + sweep_reg_bits<R>(rev);
    if (nq < M || numOps == 0 || numGrads > (rev ? SWEEP_MAX_GRADS : 0) ||
        (unsigned)__builtin_popcountll(geom.tileMask) != M)
        fail(FSA_ERR_INTERNAL, "register-tile pass of unsupported shape");
    const uint64_t numTiles = 1ULL << (nq - M);
    const unsigned nb = (unsigned)std::min<uint64_t>((numTiles + BLOCK / 64 - 1) / (BLOCK / 64), rev ? 768 : 1024);
    auto* kern = rev ? k_wave_sweep<R, (int)sweep_reg_bits<R>(true), true> : k_wave_sweep<R, (int)sweep_reg_bits<R>(false), false>;
    hipLaunchKernelGGL(kern, dim3(nb), dim3(BLOCK), 0, s, phi, lam, numTiles, geom, dops, numOps, numGrads, rows, stride);
    return nb;
}

// ws must hold 2 * numTerms * ceil(2^nbits / EXP_CHUNK) doubles
template <typename R, bool DM>
static void launch_expec_terms(hipStream_t s, const cx<R>* a, unsigned nbits, const PauliTermDev* dterms,
                               unsigned numTerms, double* ws, double* dout) {
    unsigned chunks = (unsigned)(((1ULL << nbits) + EXP_CHUNK - 1) / EXP_CHUNK);
    unsigned nb = numTerms * chunks;
    hipLaunchKernelGGL((k_pauli_expec<R, DM>), dim3(nb), dim3(BLOCK), 0, s, a, nbits, dterms, chunks, ws);
    hipLaunchKernelGGL(k_final_sum, dim3(1), dim3(BLOCK), 0, s, ws, nb, dout);
}

template <typename R>
void launch_dm_expec(hipStream_t s, const cx<R>* rho, unsigned N, const PauliTermDev* dterms,
                     unsigned numTerms, double* ws, double* dout) {
    launch_expec_terms<R, true>(s, rho, N, dterms, numTerms, ws, dout);
}

uint64_t expec_workspace_doubles(unsigned nbits, unsigned numTerms) {
    return 2ULL * numTerms * ((((1ULL << nbits) + EXP_CHUNK - 1) / EXP_CHUNK));
}

namespace {

// workgroups of k_pauli_groups: H psi takes a chunk each, <H> leaves few partials
unsigned pauli_group_blocks(unsigned n, bool expec) {
    const uint64_t chunks = 1ULL << (n - PAULI_CHUNK_BITS);
    return (unsigned)(expec ? std::min<uint64_t>(chunks, 4096) : chunks);
}

}  // namespace

uint64_t sv_expec_workspace_doubles(unsigned n, const PauliSumDev& h) {
    return h.groups ? 2ULL * pauli_group_blocks(n, true) : expec_workspace_doubles(n, h.count);
}

template <typename R>
void launch_sv_expec(hipStream_t s, const cx<R>* psi, unsigned n, const PauliSumDev& h, double* ws, double* dout) {
    if (!h.groups) {
        launch_expec_terms<R, false>(s, psi, n, h.terms, h.count, ws, dout);
        return;
    }
    const unsigned nb = pauli_group_blocks(n, true);
    hipLaunchKernelGGL((k_pauli_groups<R, true>), dim3(nb), dim3(BLOCK), 0, s, psi, (cx<R>*)nullptr,
                       (uint64_t)(1ULL << n), h.groups, h.signs, h.count, ws);
    hipLaunchKernelGGL(k_final_sum, dim3(1), dim3(BLOCK), 0, s, ws, nb, dout);
}

template <typename R>
void launch_apply_pauli_sum(hipStream_t s, const cx<R>* in, cx<R>* out, unsigned n, const PauliSumDev& h) {
    const uint64_t num = 1ULL << n;
    if (!h.groups)
        hipLaunchKernelGGL(k_apply_pauli_terms<R>, dim3((unsigned)((num + BLOCK - 1) / BLOCK)), dim3(BLOCK), 0, s, in,
                           out, num, h.terms, h.count);
    else
        hipLaunchKernelGGL((k_pauli_groups<R, false>), dim3(pauli_group_blocks(n, false)), dim3(BLOCK), 0, s, in, out,
                           num, h.groups, h.signs, h.count, (double*)nullptr);
}

template <typename R>
void launch_partial_trace(hipStream_t s, const cx<R>* in, cx<R>* out, unsigned N, const unsigned* sortedTargets,
                          unsigned k) {
    TargetList tl{};
    uint64_t allMask = 0;
    for (unsigned i = 0; i < k; i++) {
        tl.t[i] = sortedTargets[i];
        allMask |= (1ULL << sortedTargets[i]) | (1ULL << (sortedTargets[i] + N));
    }
    tl.k = k;
    uint64_t numOut = 1ULL << (2 * (N - k));
    hipLaunchKernelGGL(k_partial_trace<R>, dim3((unsigned)((numOut + BLOCK - 1) / BLOCK)), dim3(BLOCK), 0, s, in,
                       out, numOut, N, allMask, tl);
}

template <typename R>
void launch_init_gaussian(hipStream_t s, cx<R>* a, unsigned nq, uint64_t seed) {
    // the host mixes the seed the same way the oracle does (key = mix64(seed))
    uint64_t z = seed + 0x9E3779B97F4A7C15ULL;
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ULL;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBULL;
    uint64_t key = z ^ (z >> 31);
    uint64_t num = 1ULL << nq;
    hipLaunchKernelGGL(k_gaussian<R>, dim3(grid_stride_blocks(num)), dim3(BLOCK), 0, s, a, num, key);
}

template <typename R>
void launch_scale_by_inv_sqrt(hipStream_t s, cx<R>* a, uint64_t num, const double* dnorm2) {
    hipLaunchKernelGGL(k_scale_inv_sqrt<R>, dim3(grid_stride_blocks(num)), dim3(BLOCK), 0, s, a, num, dnorm2);
}

template <typename R>
void launch_init_basis(hipStream_t s, cx<R>* a, uint64_t num, uint64_t index) {
    hipLaunchKernelGGL(k_basis<R>, dim3(grid_stride_blocks(num)), dim3(BLOCK), 0, s, a, num, index);
}

void launch_f64_to_f32(hipStream_t s, const cx<double>* in, cx<float>* out, uint64_t num) {
    hipLaunchKernelGGL(k_f64_to_f32, dim3(grid_stride_blocks(num)), dim3(BLOCK), 0, s, in, out, num);
}

void launch_f32_to_f64(hipStream_t s, const cx<float>* in, cx<double>* out, uint64_t num) {
    hipLaunchKernelGGL(k_f32_to_f64, dim3(grid_stride_blocks(num)), dim3(BLOCK), 0, s, in, out, num);
}

#define FSA_INSTANTIATE_RED(R)                                                                               \
    template void launch_norm2<R>(hipStream_t, const cx<R>*, uint64_t, double*, double*);                     \
    template void launch_inner<R>(hipStream_t, const cx<R>*, const cx<R>*, uint64_t, double*, double*);       \
    template unsigned launch_adjoint_step<R>(hipStream_t, cx<R>*, cx<R>*, unsigned, const AdjointStepDev&,       \
                                             double*, uint64_t);                                                \
    template unsigned launch_sweep<R>(hipStream_t, bool, cx<R>*, cx<R>*, unsigned, const SweepGeom&,              \
                                      const SweepOp*, unsigned, unsigned, double*, uint64_t);                   \
    template unsigned launch_adjoint_diag<R>(hipStream_t, cx<R>*, cx<R>*, unsigned, const AdjointDiagDev&,       \
                                             double*, uint64_t);                                                \
    template unsigned launch_adjoint_qrun<R>(hipStream_t, cx<R>*, cx<R>*, unsigned, const AdjointQubitRunDev&,   \
                                             double*, uint64_t, const AdjointDiagDev*);                         \
    template void launch_dm_expec<R>(hipStream_t, const cx<R>*, unsigned, const PauliTermDev*, unsigned,       \
                                     double*, double*);                                                       \
    template void launch_sv_expec<R>(hipStream_t, const cx<R>*, unsigned, const PauliSumDev&, double*, double*); \
    template void launch_apply_pauli_sum<R>(hipStream_t, const cx<R>*, cx<R>*, unsigned, const PauliSumDev&);  \
    template void launch_partial_trace<R>(hipStream_t, const cx<R>*, cx<R>*, unsigned, const unsigned*,       \
                                          unsigned);                                                          \
    template void launch_init_gaussian<R>(hipStream_t, cx<R>*, unsigned, uint64_t);                           \
    template void launch_scale_by_inv_sqrt<R>(hipStream_t, cx<R>*, uint64_t, const double*);                  \
    template void launch_init_basis<R>(hipStream_t, cx<R>*, uint64_t, uint64_t);

FSA_INSTANTIATE_RED(double)
FSA_INSTANTIATE_RED(float)

}  // namespace fsa
