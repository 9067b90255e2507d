// circuit.cpp -- recorded circuits (cached fused schedule) and the adjoint-method
// gradient (no reference counterpart).
//
// Adjoint method for U = U_K ... U_1 with gadgets U_k = exp(i theta_k P_k):
//   d<H>/d theta_k = 2 Re <psi| H U_K..U_{k+1} (i P_k) phi_k> = -2 Im <lambda_k| P_k |phi_k>,
// phi_k = U_k..U_1 psi0 and lambda_k = U_{k+1}^dag..U_K^dag H psi.  The reverse
// sweep starts from phi_K = psi and lambda_K = H psi and recomputes both by
// applying U_k^dag, so no intermediate state is stored.
#include "../../include/fsa.h"
#include "engine.hpp"

#include <algorithm>
#include <cmath>
#include <cstring>

using namespace fsa;

namespace fsa {

std::vector<PauliTermDev> pauli_terms(const double* coeffs, unsigned T, const unsigned* paulis, unsigned n, bool dm) {
    std::vector<PauliTermDev> terms(T);
    for (unsigned t = 0; t < T; t++) {
        uint64_t mxy = 0, myz = 0;
        cd ph = 1.0;
        for (unsigned q = 0; q < n; q++) {
            unsigned c = paulis[(uint64_t)t * n + q];
            if (c == 1 || c == 2) mxy |= 1ULL << q;
            if (c == 2 || c == 3) myz |= 1ULL << q;
            if (c == 2) ph *= dm ? cd(0, -1) : cd(0, 1);
        }
        cd f = coeffs[t] * ph;
        terms[t] = PauliTermDev{mxy, myz, f.real(), f.imag()};
    }
    return terms;
}

PauliGroups pauli_groups(const double* coeffs, unsigned T, const unsigned* paulis, unsigned n) {
    struct Term { uint64_t mxy, myz; double c; uint32_t imag; };
    std::vector<Term> all(T);
    for (unsigned t = 0; t < T; t++) {
        Term& v = all[t];
        v.mxy = v.myz = 0;
        for (unsigned q = 0; q < n; q++) {
            const unsigned code = paulis[(uint64_t)t * n + q];
            if (code == 1 || code == 2) v.mxy |= 1ULL << q;
            if (code == 2 || code == 3) v.myz |= 1ULL << q;
        }
        // i^{#Y}: 1, i, -1, -i
        const unsigned ny = (unsigned)__builtin_popcountll(v.mxy & v.myz) & 3u;
        v.imag = ny & 1u;
        v.c = (ny & 2u) ? -coeffs[t] : coeffs[t];
    }
    std::stable_sort(all.begin(), all.end(), [](const Term& a, const Term& b) {
        return a.mxy != b.mxy ? a.mxy < b.mxy : a.imag < b.imag;
    });
    PauliGroups h;
    h.signs.reserve(T);
    for (unsigned t = 0; t < T; t++) {
        if (h.groups.empty() || h.groups.back().mxy != all[t].mxy || h.groups.back().imag != all[t].imag)
            h.groups.push_back(PauliGroupDev{all[t].mxy, t, t, all[t].imag, 0u});
        h.groups.back().t1 = t + 1;
        h.signs.push_back(PauliSignDev{all[t].myz, all[t].c});
    }
    for (size_t g = 0, first = 0; g < h.groups.size(); g++) {
        if ((h.groups[g].mxy ^ h.groups[first].mxy) >> PAULI_CHUNK_BITS) first = g;
        if (h.groups[first].run++ == 0) h.runs++;
    }
    return h;
}

namespace {

// Which form a sum takes (expec: <H>, else H psi).  Groups save loads and leave
// <H> few partials to add up, but need states that fill the GPU with chunks
// (2^11 amplitudes), and terms that share: a run of groups reads psi once.
// Time by groups / term by term:
//   <H>, 4 or more terms: 1.0-2.6 at 18 qubits and fewer, 0.55-1.07 at 19,
// 0.27-0.99 at 20, 0.09-0.25 at 24.  One string: 1.04-1.2 if it stays in its
// chunk, 0.75-0.9 if not (half of the chunks are skipped).
//   H psi of four times as many terms as runs (Z strings, local Hamiltonians):
// 0.85-1.4 at 19 qubits, 0.54-1.09 at 20, 0.26-0.97 from 22.  Of other sums, FP64:
// 0.82-0.92 for 100 terms and more at 20 qubits and 1.0-1.17 for fewer,
// 0.96 for 64 terms at 21, 0.58-1.06 for 24 and more from 22 and 0.8-1.6 for
// fewer; FP32: 1.0-1.1 at 20, 0.79-1.07 at 21 but 1.03 for one term, 0.53-1.07
// from 22.
bool by_groups(const PauliGroups& h, unsigned n, bool fp64, bool expec) {
    const unsigned terms = (unsigned)h.signs.size();
    if (expec) return n >= 20 ? terms >= 2 || h.groups[0].mxy >> PAULI_CHUNK_BITS : terms >= 4;
    if (4 * h.runs <= terms) return true;
    return fp64 ? terms >= (n == 20 ? 100u : n == 21 ? 64u : 24u) : n >= 22 || (n == 21 && terms >= 2);
}

}  // namespace

PauliSumDev push_pauli_sum(ParamRing& ring, const double* coeffs, unsigned T, const unsigned* paulis, unsigned n,
                           int prec, bool expec) {
    PauliSumDev d;
    PauliGroups h;
    const unsigned least = expec ? 19 : 20;      // qubits
    if (n >= least) h = pauli_groups(coeffs, T, paulis, n);
    if (T == 0 || n < least || !by_groups(h, n, prec == FSA_FP64, expec)) {
        const std::vector<PauliTermDev> terms = pauli_terms(coeffs, T, paulis, n, false);
        d.terms = static_cast<const PauliTermDev*>(ring.push(terms.data(), T * sizeof(PauliTermDev)));
        d.count = T;
        return d;
    }
    // one region: groups, then terms (both multiples of 8 bytes)
    const size_t gb = h.groups.size() * sizeof(PauliGroupDev), tb = h.signs.size() * sizeof(PauliSignDev);
    std::vector<char> blob(gb + tb);
    std::memcpy(blob.data(), h.groups.data(), gb);
    std::memcpy(blob.data() + gb, h.signs.data(), tb);
    const char* p = static_cast<const char*>(ring.push(blob.data(), blob.size()));
    d.groups = reinterpret_cast<const PauliGroupDev*>(p);
    d.signs = reinterpret_cast<const PauliSignDev*>(p + gb);
    d.count = (unsigned)h.groups.size();
    return d;
}

HOp inverse(const HOp& op) {
    HOp v = op;
    switch (op.kind) {
    case OP_MAT1:
    case OP_MATK: {
        uint64_t d = op.kind == OP_MAT1 ? 2 : (1ULL << op.q.size());
        for (uint64_t r = 0; r < d; r++)
            for (uint64_t k = 0; k < d; k++) v.mat[r * d + k] = std::conj(op.mat[k * d + r]);
        break;
    }
    case OP_PAULI:
        if (op.gadget) { v.theta = -op.theta; refresh_angle(v); }
        break;
    case OP_PHASE: v.theta = -op.theta; break;
    default: break;
    }
    return v;
}


}  // namespace fsa

namespace {


Circuit& cc(fsa_circuit* c) {
    need(c != nullptr, FSA_ERR_ARG, "null circuit");
    return c->c;
}

void check_list(const unsigned* q, unsigned num, const char* what) {
    need(num == 0 || q != nullptr, FSA_ERR_ARG, std::string("null ") + what);
    uint64_t seen = 0;
    for (unsigned i = 0; i < num; i++) {
        need(q[i] < 40, FSA_ERR_QUBIT, std::string(what) + " index out of range");
        need(!((seen >> q[i]) & 1), FSA_ERR_DUPLICATE, std::string("repeated qubit among ") + what);
        seen |= 1ULL << q[i];
    }
}

void add(Circuit& c, HOp op) {
    unsigned mx = 0;
    for (unsigned q = 0; q < 64; q++) if (((op.touch | op.ctrl) >> q) & 1) mx = q + 1;
    c.maxQubit = std::max(c.maxQubit, mx);
    c.ops.push_back(std::move(op));
    c.cachedPrec = -1;
    c.sweepPrec[0] = c.sweepPrec[1] = -1;
}

std::vector<cd> mat_of(const double* g, uint64_t dim) {
    need(g != nullptr, FSA_ERR_ARG, "null gate matrix");
    std::vector<cd> m(dim * dim);
    for (uint64_t i = 0; i < dim * dim; i++) m[i] = cd(g[2 * i], g[2 * i + 1]);
    return m;
}

HOp pauli_op(const unsigned* t, const unsigned* p, unsigned num, bool gadget, double theta) {
    HOp o;
    o.kind = OP_PAULI;
    o.pw = 1.0;
    for (unsigned i = 0; i < num; i++) {
        need(p[i] <= 3, FSA_ERR_ARG, "Pauli codes are 0..3 (I, X, Y, Z)");
        if (p[i] == 2) o.pw *= cd(0, 1);
        if (p[i] == 1 || p[i] == 2) o.mxy |= 1ULL << t[i];
        if (p[i] == 2 || p[i] == 3) o.myz |= 1ULL << t[i];
    }
    o.gadget = gadget;
    o.theta = theta;
    refresh_angle(o);
    finish_op(o);
    return o;
}

const Plan& plan_for(Circuit& c, unsigned nq, int prec) {
    if (c.cachedNq != nq || c.cachedPrec != prec) {
        c.cached = make_plan(c.ops, nq, prec);
        c.cachedNq = nq;
        c.cachedPrec = prec;
    }
    return c.cached;
}


// ---- register-tile passes of the adjoint (k_wave_sweep) -----------------------

// ops with a register-tile form: diagonal gadgets, Pauli strings with one X/Y
// qubit, one-target matrices (controls and Z factors anywhere)
bool sweep_form(const HOp& op) {
    return op.kind == OP_PHASE || op.kind == OP_MAT1 ||
           (op.kind == OP_PAULI && __builtin_popcountll(op.mxy) <= 1);
}
// the qubit such an op mixes, or -1
int sweep_mixes(const HOp& op) { return op.nd ? __builtin_ctzll(op.nd) : -1; }

// Stages of the forward or reverse (rev) sweep on register tiles.  Ops move past
// others they commute with (schedule()); a gadget's gradient term
// <lambda|P|phi> does not change when such an op is undone before or after it.
template <typename R>
const std::vector<Stage>& sweep_stages(Circuit& c, unsigned n, int prec, bool rev) {
    if (c.sweepNq[rev] != n || c.sweepPrec[rev] != prec) {
        const size_t L = c.ops.size();
        std::vector<HOp> order(L);
        for (size_t r = 0; r < L; r++) {
            const HOp& o = c.ops[rev ? L - 1 - r : r];
            order[r].kind = o.kind;
            order[r].nd = o.nd;
            order[r].touch = o.touch;
            order[r].tileable = sweep_form(o);
        }
        // the low qubits of one 128-byte line are in every tile
        const unsigned M = SWEEP_LANE_BITS + sweep_reg_bits<R>(rev), low = sizeof(R) == 8 ? 3u : 4u;
        c.sweepStages[rev] = schedule(order, n, n <= M ? SchedParams{n, n} : SchedParams{M, low});
        if (rev)
            for (Stage& st : c.sweepStages[rev])
                for (int& i : st.ops) i = (int)L - 1 - i;
        c.sweepNq[rev] = n;
        c.sweepPrec[rev] = prec;
    }
    return c.sweepStages[rev];
}

struct SweepPass {
    SweepGeom geom;
    size_t first = 0;        // its ops: sops[first .. first + count)
    unsigned count = 0, grads = 0;
};

// Turns a stage into passes: places its qubits on lane and register bits, adds
// exchanges where an op needs a qubit on a register bit, groups diagonal
// gadgets.  Qubits 0-2 (FP32: 0-3) stay on the same lane bits, so that every
// access covers whole 128-byte lines, which the streaming stores need (FP32
// without qubit 3: 1% slower).
template <typename R>
class SweepBuilder {
public:
    SweepBuilder(const Circuit& c, bool rev, std::vector<SweepOp>& sops)
        : c_(c), rev_(rev), G_(sweep_reg_bits<R>(rev)), sops_(sops) {}

    std::vector<SweepPass> stage(const Stage& st) {
        place(st);
        passes_.clear();
        open(st);
        for (size_t i = 0; i < st.ops.size(); i++) {
            const HOp& op = c_.ops[st.ops[i]];
            const bool grad = rev_ && op.param >= 0;
            if (grad && passes_.back().grads == SWEEP_MAX_GRADS) {
                flush_run();
                close();
                open(st);
            }
            if (grad) passes_.back().grads++;
            const int q = sweep_mixes(op);
            if (q < 0) {
                run_.push_back(&op);
                continue;
            }
            flush_run();
            if (lane_[4] == q || lane_[5] == q) {
                // the register bit whose qubit is mixed again last gives way
                const unsigned l = lane_[4] == q ? 4 : 5;
                unsigned B = 0;
                size_t far = 0;
                for (unsigned b = 0; b < G_; b++) {
                    size_t next = i + 1;
                    while (next < st.ops.size() && sweep_mixes(c_.ops[st.ops[next]]) != reg_[b]) next++;
                    if (next > far) { far = next; B = b; }
                }
                std::swap(lane_[l], reg_[B]);
                SweepOp t;
                std::memset(&t, 0, sizeof(t));
                t.code = SWEEP_SWAP + 5 * (l - 4) + B;
                emit(t, nullptr);
            }
            emit(translate(op), &op);
        }
        flush_run();
        close();
        return passes_;
    }

private:
    const Circuit& c_;
    const bool rev_;
    const unsigned G_;
    std::vector<SweepOp>& sops_;
    std::vector<SweepPass> passes_;
    std::vector<const HOp*> run_;      // diagonal ops since the last mixing one
    unsigned grads_ = 0;
    int lane_[SWEEP_LANE_BITS], reg_[8];

    void place(const Stage& st) {
        // register bits: the qubits mixed first; lane bit 3 (FP64), whose partners
        // come by moves, the one mixed least often of the rest
        constexpr unsigned low = sizeof(R) == 8 ? 3 : 4;
        std::vector<int> rest(st.tq.begin() + low, st.tq.end());
        unsigned uses[64] = {0};
        std::vector<int> byUse;
        for (int oi : st.ops) {
            const int q = sweep_mixes(c_.ops[oi]);
            if (q < 0) continue;
            if (!uses[q]++ && std::find(rest.begin(), rest.end(), q) != rest.end()) byUse.push_back(q);
        }
        for (auto q = rest.rbegin(); q != rest.rend(); ++q) if (!uses[*q]) byUse.push_back(*q);
        for (unsigned b = 0; b < G_; b++) reg_[b] = byUse[b];
        std::vector<int> ln(byUse.begin() + G_, byUse.end());
        std::stable_sort(ln.begin(), ln.end(), [&](int a, int b) { return uses[a] < uses[b]; });
        for (unsigned b = 0; b < low; b++) lane_[b] = (int)st.tq[b];
        for (unsigned b = low; b < SWEEP_LANE_BITS; b++) lane_[b] = ln[b - low];
    }
    void open(const Stage& st) {
        SweepPass p;
        std::memset(&p.geom, 0, sizeof(p.geom));
        for (unsigned q : st.tq) p.geom.tileMask |= 1ULL << q;
        for (unsigned b = 0; b < SWEEP_LANE_BITS; b++) p.geom.lane[b] = (uint8_t)lane_[b];
        for (unsigned b = 0; b < G_; b++) p.geom.reg[b] = (uint8_t)reg_[b];
        p.first = sops_.size();
        grads_ = 0;
        passes_.push_back(p);
    }
    void close() {
        SweepPass& p = passes_.back();
        for (unsigned b = 0; b < SWEEP_LANE_BITS; b++) p.geom.laneOut[b] = (uint8_t)lane_[b];
        for (unsigned b = 0; b < G_; b++) p.geom.regOut[b] = (uint8_t)reg_[b];
        p.count = (unsigned)(sops_.size() - p.first);
    }
    void emit(SweepOp t, const HOp* op) {
        if (op && rev_ && op->param >= 0) {
            t.flags |= grads_ & 1u ? SWEEP_GRAD_ODD : SWEEP_GRAD_EVEN;
            t.row = grads_ / 2;
            t.slot = (uint32_t)op->param;
            grads_++;
        }
        sops_.push_back(t);
    }
    // turn()'s c for the rotation with cosine t.c >= 0 and sine t.g: -tan(a / 2), or t.c itself
    double turn_c(const SweepOp& t) const { return sizeof(R) == 8 || rev_ ? -t.g / (1.0 + t.c) : t.c; }

    // diagonal ops commute: those with the same slot signs go together
    void flush_run() {
        std::vector<std::pair<SweepOp, const HOp*>> ts;
        for (const HOp* op : run_) ts.emplace_back(translate(*op), op);
        run_.clear();
        std::stable_sort(ts.begin(), ts.end(), [](const auto& a, const auto& b) { return a.first.sw < b.first.sw; });
        for (size_t i = 0; i < ts.size(); i++) {
            if (i == 0 || ts[i].first.sw != ts[i - 1].first.sw) ts[i].first.flags |= SWEEP_GROUP_FIRST;
            if (i + 1 == ts.size() || ts[i].first.sw != ts[i + 1].first.sw) ts[i].first.flags |= SWEEP_GROUP_LAST;
            const uint32_t one = SWEEP_GROUP_FIRST | SWEEP_GROUP_LAST;
            if ((ts[i].first.flags & one) == one) {
                ts[i].first.code += SWEEP_DIAG_ONE - SWEEP_DIAG;
                ts[i].first.c = turn_c(ts[i].first);
            }
            emit(ts[i].first, ts[i].second);
        }
    }
    // op (rev: the op that undoes it) in the current layout
    SweepOp translate(const HOp& op) const {
        SweepOp t;
        std::memset(&t, 0, sizeof(t));
        uint32_t rmask = 0;
        auto lane_bit = [&](int q) { return (int)(std::find(lane_, lane_ + SWEEP_LANE_BITS, q) - lane_); };
        auto reg_bit = [&](int q) { return (int)(std::find(reg_, reg_ + G_, q) - reg_); };
        auto split = [&](uint64_t m) {
            for (; m; m &= m - 1) {
                const int q = __builtin_ctzll(m), lb = lane_bit(q), rb = reg_bit(q);
                if (lb < (int)SWEEP_LANE_BITS) t.lz |= 1u << lb;
                else if (rb < (int)G_) rmask |= 1u << rb;
                else t.oz |= 1ULL << q;
            }
        };
        const int q = sweep_mixes(op), rb = q < 0 ? 0 : reg_bit(q);
        const bool onReg = q >= 0 && rb < (int)G_;
        if (op.kind == OP_MAT1) {
            split(op.ctrl);
            for (uint32_t i = 0; i < (1u << G_); i++) if ((i & rmask) == rmask) t.sw |= 1u << i;
            t.code = onReg ? SWEEP_MAT_REG + (uint32_t)rb : (uint32_t)SWEEP_MAT_LANE;
            t.bit = onReg ? 0u : (uint32_t)lane_bit(q);
            for (unsigned i = 0; i < 4; i++) {       // rev: conjugate transpose
                const cd v = rev_ ? std::conj(op.mat[(i & 1) * 2 + (i >> 1)]) : op.mat[i];
                t.f[2 * i] = v.real();
                t.f[2 * i + 1] = v.imag();
            }
            return t;
        }
        // A Pauli tensor P is exp(i pi/2 P), and exp(i (theta - pi) P) is
        // -exp(i theta P): phases common to phi and lambda, which neither <H>
        // nor a gradient term sees.  So the cosine is taken to be >= 0.
        const bool tensor = op.kind == OP_PAULI && !op.gadget;
        double cs = tensor ? 0.0 : std::cos(op.theta), sn = tensor ? 1.0 : std::sin(op.theta);
        if (rev_) sn = -sn;
        if (cs < 0) { cs = -cs; sn = -sn; }
        split(op.kind == OP_PHASE ? op.pmask : op.myz);
        for (uint32_t i = 0; i < (1u << G_); i++) if (par32(i & rmask)) t.sw |= 1u << i;
        const uint32_t ss = t.sw != 0;
        t.c = cs;
        t.g = sn;                                    // exp(i theta Z..Z)
        if (q < 0) {
            t.code = SWEEP_DIAG + ss;
            return t;
        }
        // exp(i theta P) = cos + i sin i^{#Y} (...): imaginary factor for X, real for Y (#Y = 1)
        const bool y = (op.mxy & op.myz) != 0;
        if (y) t.g = -sn;
        if (onReg) {
            t.code = SWEEP_REG + 4u * (uint32_t)rb;
            t.c = turn_c(t);
        } else {
            t.code = SWEEP_LANE + 4u * (uint32_t)lane_bit(q);
            if (y) t.lz |= SWEEP_CONST_SIGN;         // the factor is the partner lane's
        }
        t.code += (y ? 0u : 2u) + ss;
        return t;
    }
};

// every tiled stage's passes, their ops in one list on the device
template <typename R>
std::vector<std::vector<SweepPass>> sweep_passes(const Circuit& c, const std::vector<Stage>& stages, bool rev,
                                                 ParamRing& ring, std::vector<SweepOp>& sops, const SweepOp*& dops) {
    std::vector<std::vector<SweepPass>> passes(stages.size());
    SweepBuilder<R> b(c, rev, sops);
    for (size_t si = 0; si < stages.size(); si++)
        if (stages[si].tiled) passes[si] = b.stage(stages[si]);
    dops = sops.empty() ? nullptr : static_cast<const SweepOp*>(ring.push(sops.data(), sops.size() * sizeof(SweepOp)));
    return passes;
}

// a statevector work state on a stream it does not own
struct Scratch {
    State s;
    Scratch(unsigned n, int prec, hipStream_t stream) {
        s.N = n;
        s.nq = n;
        s.prec = prec;
        s.mode = FSA_EXEC_EAGER;
        s.stream = stream;
        s.ring.stream = stream;
        hip_check(hipMalloc(&s.amps, s.num() * s.amp_bytes()), "hipMalloc(adjoint scratch)");
    }
    ~Scratch() {
        (void)hipStreamSynchronize(s.stream);
        if (s.amps) (void)hipFree(s.amps);
        if (s.ws) (void)hipFree(s.ws);
    }
};

}  // namespace

namespace fsa {

// phi and lambda of the adjoint sweep on a stream of their own, with their
// parameter rings and workspace: allocated on the first call for a size and
// precision and reused by the next ones (a call allocates nothing then)
struct AdjointScratch {
    unsigned n;
    int prec;
    hipStream_t stream = nullptr;
    hipEvent_t ready = nullptr;
    std::unique_ptr<Scratch> phi, lam;
    AdjointScratch(unsigned n_, int prec_) : n(n_), prec(prec_) {
        try {
            hip_check(hipStreamCreateWithFlags(&stream, hipStreamNonBlocking), "hipStreamCreate");
            hip_check(hipEventCreateWithFlags(&ready, hipEventDisableTiming), "hipEventCreate");
            phi = std::make_unique<Scratch>(n, prec, stream);
            lam = std::make_unique<Scratch>(n, prec, stream);
        } catch (...) {
            release();
            throw;
        }
    }
    ~AdjointScratch() { release(); }
    void release() {
        phi.reset();      // each synchronises the stream before freeing
        lam.reset();
        if (ready) (void)hipEventDestroy(ready);
        if (stream) (void)hipStreamDestroy(stream);
        ready = nullptr;
        stream = nullptr;
    }
};

}  // namespace fsa

namespace {

template <typename R>
void adjoint_impl(Circuit& c, State& psi0, const double* coeffs, unsigned T, const unsigned* paulis, double* expec,
                  double* grads) {
    const unsigned n = psi0.N;
    flush(psi0);
    if (!c.adj || c.adj->n != n || c.adj->prec != psi0.prec) {
        c.adj.reset();
        c.adj = std::make_shared<AdjointScratch>(n, psi0.prec);
    }
    AdjointScratch& A = *c.adj;
    hipStream_t st = A.stream;
    // psi0 is read below: after the work already queued on its own stream
    hip_check(hipEventRecord(A.ready, psi0.stream), "hipEventRecord");
    hip_check(hipStreamWaitEvent(st, A.ready, 0), "hipStreamWaitEvent");
    Scratch& phi = *A.phi;
    Scratch& lam = *A.lam;
    // results: slot 0 = <phi|lambda>, slot 1 + p = <lambda|P_p|phi>, then the
    // FP64 norms <psi0|psi0> and <phi|phi> (FP32 renormalisation), then the
    // gradient rows of the sweep
    const unsigned P = c.numParams;
    const size_t red = reduce_workspace_doubles(phi.s.num());
    const uint64_t stride = adjoint_row_stride(n);
    double* ws = phi.s.workspace(red + 2 * (P + 1) + 2 + stride * P + 8);
    double* res = ws + red;
    double* norms = res + 2 * (P + 1);
    double* rows = norms + 2;
    const bool renorm = psi0.prec == FSA_FP32;
    if (renorm) launch_norm2<R>(st, (const cx<R>*)psi0.amps, psi0.num(), ws, norms);
    hip_check(hipMemcpyAsync(phi.s.amps, psi0.amps, psi0.num() * psi0.amp_bytes(), hipMemcpyDeviceToDevice, st),
              "hipMemcpyAsync");
    // circuits of ops with a register-tile form run in such passes forward, too
    if (n >= sweep_min_qubits<R>() && std::all_of(c.ops.begin(), c.ops.end(), sweep_form)) {
        const std::vector<Stage>& stages = sweep_stages<R>(c, n, psi0.prec, false);
        ParamRing::Hold hold(phi.s.ring);
        std::vector<SweepOp> sops;
        const SweepOp* dops = nullptr;
        const auto passes = sweep_passes<R>(c, stages, false, phi.s.ring, sops, dops);
        for (size_t si = 0; si < stages.size(); si++) {
            if (!stages[si].tiled) {
                std::vector<HOp> alone;
                for (int oi : stages[si].ops) alone.push_back(c.ops[oi]);
                execute_now(phi.s, alone);
                continue;
            }
            for (const SweepPass& p : passes[si]) {
                ProfScope prof("forward_sweep", st);
                launch_sweep<R>(st, false, (cx<R>*)phi.s.amps, (cx<R>*)nullptr, n, p.geom, dops + p.first, p.count, 0,
                                nullptr, 0);
                hip_check(hipGetLastError(), "forward sweep launch");
            }
        }
    } else {
        execute(phi.s, plan_for(c, n, psi0.prec));
    }
    // a unitary circuit keeps the norm; FP32 rounding does not quite.  <H> and
    // every gradient term are quadratic in phi (lambda = H phi), so the
    // forward drift is undone by scaling them by <psi0|psi0> / <phi|phi> at
    // the end instead of rescaling the states
    if (renorm) launch_norm2<R>(st, (const cx<R>*)phi.s.amps, phi.s.num(), ws, norms + 1);

    const PauliSumDev h = push_pauli_sum(phi.s.ring, coeffs, T, paulis, n, psi0.prec, false);
    auto* a_phi = (cx<R>*)phi.s.amps;
    auto* a_lam = (cx<R>*)lam.s.amps;
    launch_apply_pauli_sum<R>(st, a_phi, a_lam, n, h);

    // Reverse sweep, op by op: for a gadget, <lambda|P_k|phi> and U_k^dag on phi
    // and on lambda in one pass over both states (k_adjoint_step); any other op
    // is undone on each state by its own kernel.
    // Runs of consecutive parametrised diagonal gadgets (phase gadgets, Z-only
    // Pauli gadgets) take one pass per ADJ_DIAG_MAX of them (k_adjoint_diag).
    // Every gadget's partial sums go to the row slot of its parameter; one
    // launch adds each slot's rows after the sweep (launch_grad_sums).
    std::vector<uint32_t> nbs(P, 0);
    launch_inner<R>(st, a_phi, a_lam, phi.s.num(), ws, res);
    auto diag_gadget = [](const HOp& o) {
        return o.param >= 0 && (o.kind == OP_PHASE || (o.kind == OP_PAULI && o.mxy == 0));
    };
    // Runs of consecutive parametrised one-qubit X/Y gadgets on distinct
    // qubits take one pass per ADJ_QRUN_MAX of them (k_adjoint_qrun).
    auto qubit_gadget = [](const HOp& o) {
        return o.param >= 0 && o.kind == OP_PAULI && __builtin_popcountll(o.mxy) == 1 && (o.myz & ~o.mxy) == 0;
    };
    // the diagonal run starting at op j (going backwards): returns its length
    auto build_diag = [&](size_t j0, AdjointDiagDev& d) {
        std::memset(&d, 0, sizeof(d));
        size_t j = j0 + 1;
        while (j-- > 0 && d.count < ADJ_DIAG_MAX && diag_gadget(c.ops[j])) {
            const HOp& g = c.ops[j];
            const HOp gi = inverse(g);
            const unsigned i = d.count++;
            cd e0, e1;
            if (g.kind == OP_PAULI) {              // th v + (+-fe) v, f = i^{#Y} (1: no Y)
                d.myz[i] = g.myz;
                d.fr[i] = g.pw.real(); d.fi[i] = g.pw.imag();
                e0 = gi.th + gi.fe;
                e1 = gi.th - gi.fe;
            } else {
                d.myz[i] = g.pmask;
                d.fr[i] = 1.0; d.fi[i] = 0.0;
                e0 = cd(std::cos(gi.theta), std::sin(gi.theta));
                e1 = cd(std::cos(gi.theta), -std::sin(gi.theta));
            }
            d.e0r[i] = e0.real(); d.e0i[i] = e0.imag();
            d.e1r[i] = e1.real(); d.e1i[i] = e1.imag();
            d.slot[i] = (uint32_t)g.param;
        }
        return d.count;
    };
    // one op on its own: a gadget by k_adjoint_step, any other by its own kernel
    auto undo = [&](const HOp& op) {
        const HOp inv = inverse(op);
        if (op.param >= 0) {
            AdjointStepDev d;
            std::memset(&d, 0, sizeof(d));
            if (op.kind == OP_PAULI) {
                d.mxy = op.mxy; d.myz = op.myz;
                d.fr = op.pw.real(); d.fi = op.pw.imag();
                d.thr = inv.th.real(); d.thi = inv.th.imag();
                d.fer = inv.fe.real(); d.fei = inv.fe.imag();
            } else {
                d.mxy = 0; d.myz = op.pmask;
                d.fr = 1.0; d.fi = 0.0;
                d.phase = 1;
                d.e0r = std::cos(inv.theta); d.e0i = std::sin(inv.theta);
                d.e1r = std::cos(inv.theta); d.e1i = -std::sin(inv.theta);
            }
            d.slot = (uint32_t)op.param;
            ProfScope prof("adjoint_step", st);
            nbs[op.param] = launch_adjoint_step<R>(st, a_phi, a_lam, n, d, rows, stride);
            hip_check(hipGetLastError(), "adjoint step launch");
            return;
        }
        std::vector<HOp> invs{inv};
        execute_now(phi.s, invs);
        execute_now(lam.s, invs);
    };
    if (n >= sweep_min_qubits<R>()) {
        // register-tile passes; stages of one op and ops without such a form alone
        const std::vector<Stage>& stages = sweep_stages<R>(c, n, psi0.prec, true);
        ParamRing::Hold hold(phi.s.ring);        // undo() may push parameters of its own
        std::vector<SweepOp> sops;
        const SweepOp* dops = nullptr;
        const auto passes = sweep_passes<R>(c, stages, true, phi.s.ring, sops, dops);
        for (size_t si = 0; si < stages.size(); si++) {
            if (!stages[si].tiled) {
                for (int oi : stages[si].ops) undo(c.ops[oi]);
                continue;
            }
            for (const SweepPass& p : passes[si]) {
                ProfScope prof("adjoint_sweep", st);
                const unsigned nb = launch_sweep<R>(st, true, a_phi, a_lam, n, p.geom, dops + p.first, p.count, p.grads,
                                                    rows, stride);
                hip_check(hipGetLastError(), "adjoint sweep launch");
                for (size_t i = p.first; i < p.first + p.count; i++)
                    if (sops[i].flags & (SWEEP_GRAD_EVEN | SWEEP_GRAD_ODD)) nbs[sops[i].slot] = nb;
            }
        }
    } else {
    for (size_t k = c.ops.size(); k-- > 0;) {
        const HOp& op = c.ops[k];
        if (qubit_gadget(op) && k > 0 && qubit_gadget(c.ops[k - 1]) && c.ops[k - 1].mxy != op.mxy) {
            AdjointQubitRunDev d;
            std::memset(&d, 0, sizeof(d));
            uint64_t used = 0;
            size_t j = k + 1;
            while (j-- > 0 && d.count < ADJ_QRUN_MAX && qubit_gadget(c.ops[j]) && !(c.ops[j].mxy & used)) {
                const HOp& g = c.ops[j];
                const HOp gi = inverse(g);
                const unsigned i = d.count++;
                used |= g.mxy;
                d.q[i] = (uint32_t)__builtin_ctzll(g.mxy);
                d.y[i] = g.myz != 0;
                d.fr[i] = g.pw.real(); d.fi[i] = g.pw.imag();
                d.thr[i] = gi.th.real(); d.thi[i] = gi.th.imag();
                d.fer[i] = gi.fe.real(); d.fei[i] = gi.fe.imag();
                d.slot[i] = (uint32_t)g.param;
            }
            std::copy(d.q, d.q + d.count, d.sorted);
            std::sort(d.sorted, d.sorted + d.count);
            // a run on qubits below 6 takes the diagonal run after it (if any)
            // into the same pass
            AdjointDiagDev tail;
            unsigned nt = 0;
            if (used < 64 && n >= 6 && k >= d.count && diag_gadget(c.ops[k - d.count]))
                nt = build_diag(k - d.count, tail);
            ProfScope prof("adjoint_qrun", st);
            const unsigned nb = launch_adjoint_qrun<R>(st, a_phi, a_lam, n, d, rows, stride, nt ? &tail : nullptr);
            hip_check(hipGetLastError(), "adjoint qubit run launch");
            for (unsigned i = 0; i < d.count; i++) nbs[d.slot[i]] = nb;
            for (unsigned i = 0; i < nt; i++) nbs[tail.slot[i]] = nb;
            k -= d.count + nt - 1;  // the loop's k-- moves past the run and its tail
            continue;
        }
        if (diag_gadget(op) && k > 0 && diag_gadget(c.ops[k - 1])) {
            AdjointDiagDev d;
            build_diag(k, d);
            ProfScope prof("adjoint_diag", st);
            const unsigned nb = launch_adjoint_diag<R>(st, a_phi, a_lam, n, d, rows, stride);
            hip_check(hipGetLastError(), "adjoint diagonal run launch");
            for (unsigned i = 0; i < d.count; i++) nbs[d.slot[i]] = nb;
            k -= d.count - 1;       // the loop's k-- moves past the run
            continue;
        }
        undo(op);
    }
    }
    if (P) {
        auto* dnb = (const uint32_t*)phi.s.ring.push(nbs.data(), nbs.size() * sizeof(uint32_t));
        launch_grad_sums(st, rows, stride, dnb, P, res + 2);
        hip_check(hipGetLastError(), "gradient sums launch");
    }
    std::vector<double> host(2 * (P + 1) + 2);
    hip_check(hipMemcpyAsync(host.data(), res, host.size() * sizeof(double), hipMemcpyDeviceToHost, st), "hipMemcpyAsync");
    hip_check(hipStreamSynchronize(st), "hipStreamSynchronize");
    const double sc = renorm && host[2 * (P + 1) + 1] > 0 ? host[2 * (P + 1)] / host[2 * (P + 1) + 1] : 1.0;
    *expec = host[0] * sc;
    for (unsigned p = 0; p < P; p++) grads[p] = -2.0 * host[2 * (1 + p) + 1] * sc;
}

}  // namespace

extern "C" {

int fsa_circuit_create(fsa_circuit** out) {
    return guard([&] {
        need(out != nullptr, FSA_ERR_ARG, "null output handle");
        *out = new fsa_circuit();
    });
}

int fsa_circuit_destroy(fsa_circuit* c) {
    delete c;
    return FSA_OK;
}

int fsa_circuit_num_ops(const fsa_circuit* c, unsigned* out) {
    return guard([&] {
        need(c && out, FSA_ERR_ARG, "null argument");
        *out = (unsigned)c->c.ops.size();
    });
}

int fsa_circuit_num_params(const fsa_circuit* c, unsigned* out) {
    return guard([&] {
        need(c && out, FSA_ERR_ARG, "null argument");
        *out = c->c.numParams;
    });
}

int fsa_circuit_oneTargGate(fsa_circuit* h, unsigned target, const double* gate) {
    return guard([&] {
        Circuit& c = cc(h);
        check_list(&target, 1, "target");
        HOp o;
        o.kind = OP_MAT1;
        o.q = {target};
        o.mat = mat_of(gate, 2);
        finish_op(o);
        add(c, std::move(o));
    });
}

int fsa_circuit_manyCtrlOneTargGate(fsa_circuit* h, const unsigned* controls, unsigned numControls, unsigned target,
                                    const double* gate) {
    return guard([&] {
        Circuit& c = cc(h);
        need(numControls == 0 || controls, FSA_ERR_ARG, "null controls");
        std::vector<unsigned> all(controls, controls + numControls);
        all.push_back(target);
        check_list(all.data(), (unsigned)all.size(), "control/target");
        HOp o;
        o.kind = OP_MAT1;
        o.q = {target};
        for (unsigned i = 0; i < numControls; i++) o.ctrl |= 1ULL << controls[i];
        o.mat = mat_of(gate, 2);
        finish_op(o);
        add(c, std::move(o));
    });
}

int fsa_circuit_swapGate(fsa_circuit* h, unsigned qb1, unsigned qb2) {
    return guard([&] {
        Circuit& c = cc(h);
        need(qb1 < 40 && qb2 < 40, FSA_ERR_QUBIT, "qubit index out of range");
        if (qb1 == qb2) return;
        HOp o;
        o.kind = OP_SWAP;
        o.q = {std::min(qb1, qb2), std::max(qb1, qb2)};
        finish_op(o);
        add(c, std::move(o));
    });
}

int fsa_circuit_manyTargGate(fsa_circuit* h, const unsigned* targets, unsigned numTargets, const double* gate) {
    return guard([&] {
        Circuit& c = cc(h);
        need(numTargets >= 1, FSA_ERR_ARG, "manyTargGate needs at least one target");
        check_list(targets, numTargets, "target");
        need(numTargets <= 12, FSA_ERR_SIZE, "manyTargGate supports at most 12 targets");
        HOp o;
        o.kind = numTargets == 1 ? OP_MAT1 : OP_MATK;
        o.q.assign(targets, targets + numTargets);
        o.mat = mat_of(gate, 1ULL << numTargets);
        finish_op(o);
        add(c, std::move(o));
    });
}

int fsa_circuit_pauliTensor(fsa_circuit* h, const unsigned* targets, const unsigned* paulis, unsigned num) {
    return guard([&] {
        Circuit& c = cc(h);
        check_list(targets, num, "target");
        need(num == 0 || paulis, FSA_ERR_ARG, "null paulis");
        add(c, pauli_op(targets, paulis, num, false, 0.0));
    });
}

int fsa_circuit_pauliGadget(fsa_circuit* h, const unsigned* targets, const unsigned* paulis, unsigned num,
                            double theta) {
    return guard([&] {
        Circuit& c = cc(h);
        check_list(targets, num, "target");
        need(num == 0 || paulis, FSA_ERR_ARG, "null paulis");
        HOp o = pauli_op(targets, paulis, num, true, theta);
        o.param = (int)c.numParams++;
        add(c, std::move(o));
    });
}

int fsa_circuit_phaseGadget(fsa_circuit* h, const unsigned* targets, unsigned num, double theta) {
    return guard([&] {
        Circuit& c = cc(h);
        check_list(targets, num, "target");
        HOp o;
        o.kind = OP_PHASE;
        for (unsigned i = 0; i < num; i++) o.pmask |= 1ULL << targets[i];
        o.theta = theta;
        o.param = (int)c.numParams++;
        finish_op(o);
        add(c, std::move(o));
    });
}

int fsa_circuit_set_params(fsa_circuit* h, const double* thetas, unsigned numParams) {
    return guard([&] {
        Circuit& c = cc(h);
        need(numParams == c.numParams && (numParams == 0 || thetas), FSA_ERR_ARG, "parameter count mismatch");
        for (HOp& o : c.ops)
            if (o.param >= 0) {
                o.theta = thetas[o.param];
                refresh_angle(o);
            }
        for (HOp& o : c.cached.ops)
            if (o.param >= 0) {
                o.theta = thetas[o.param];
                refresh_angle(o);
            }
    });
}

int fsa_circuit_apply(fsa_circuit* h, fsa_state* psi) {
    return guard([&] {
        Circuit& c = cc(h);
        need(psi != nullptr, FSA_ERR_ARG, "null state");
        State& s = psi->s;
        need(!s.dm, FSA_ERR_KIND, "circuits act on statevectors");
        need(c.maxQubit <= s.N, FSA_ERR_QUBIT, "circuit uses a qubit the state does not have");
        flush(s);
        execute(s, plan_for(c, s.nq, s.prec));
    });
}

int fsa_circuit_num_passes(fsa_circuit* h, unsigned numQubits, int precision, unsigned* out) {
    return guard([&] {
        Circuit& c = cc(h);
        need(out != nullptr, FSA_ERR_ARG, "null output");
        need(precision == FSA_FP64 || precision == FSA_FP32, FSA_ERR_ARG, "bad precision");
        need(c.maxQubit <= numQubits, FSA_ERR_QUBIT, "circuit uses a qubit the state does not have");
        const auto& stages = plan_for(c, numQubits, precision).stages;
        unsigned n = 0;
        for (const Stage& st : stages) n += st.tiled ? 1 : (unsigned)st.ops.size();
        *out = n;
    });
}

int fsa_adjoint_gradient(fsa_circuit* h, fsa_state* psi0, const double* coeffs, unsigned numTerms,
                         const unsigned* paulis, double* expec, double* grads) {
    return guard([&] {
        Circuit& c = cc(h);
        need(psi0 != nullptr && expec != nullptr, FSA_ERR_ARG, "null argument");
        need(c.numParams == 0 || grads != nullptr, FSA_ERR_ARG, "null gradient output");
        need(numTerms >= 1 && coeffs && paulis, FSA_ERR_ARG, "the observable needs at least one term");
        State& s = psi0->s;
        need(!s.dm, FSA_ERR_KIND, "the adjoint gradient acts on statevectors");
        need(c.maxQubit <= s.N, FSA_ERR_QUBIT, "circuit uses a qubit the state does not have");
        for (uint64_t i = 0; i < (uint64_t)numTerms * s.N; i++)
            need(paulis[i] <= 3, FSA_ERR_ARG, "Pauli codes are 0..3 (I, X, Y, Z)");
        if (s.prec == FSA_FP64) adjoint_impl<double>(c, s, coeffs, numTerms, paulis, expec, grads);
        else adjoint_impl<float>(c, s, coeffs, numTerms, paulis, expec, grads);
    });
}

}  // extern "C"
