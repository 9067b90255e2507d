// Checks of the host planners that no public call can trigger, compiled against
// the CPU stand-in with the planner's source in the same unit.  Prints one line
// per check; exit status 0 unless one failed.
#include "../../distributed-full-state-algorithms_amd/csrc/batch.cpp"

#include <cstdio>
#include <functional>

static int failures = 0;

static void refuses(const char* what, const std::function<void()>& f) {
    bool threw = false;
    try { f(); } catch (const Error&) { threw = true; }
    std::printf("%s %s\n", what, threw ? "refused" : "ACCEPTED");
    failures += !threw;
}

static HOp gadget(uint64_t mxy, uint64_t myz, int param) {
    HOp o;
    o.kind = OP_PAULI;
    o.gadget = true;
    o.mxy = mxy;
    o.myz = myz;
    o.theta = 0.3;
    o.param = param;
    refresh_angle(o);
    finish_op(o);
    return o;
}

// a reverse plan of these ops on 6 qubits
static void plan(const std::vector<HOp>& ops, const std::vector<int>& sign) {
    BlobBuilder<double> bb;
    uint32_t first = 0, count = 0;
    bb.add_plan(ops, sign, 6, SchedParams{6, 6}, 1, true, first, count);
}

// an MFMA pass over tiles of 2^m amplitudes
template <typename R>
static void mfma_pass(unsigned m) {
    TileGeom g{};
    g.m = m;
    for (unsigned q = 0; q < m; q++) g.tileMask |= 1ULL << q;
    launch_tile<R>(nullptr, nullptr, m, g, nullptr, 1, nullptr, nullptr, 2u << 2, 0);
}

int main() {
    const HOp a = gadget(1, 0, 0), b = gadget(2, 0, 1);
    const HOp ga = grad_op(a, 0), gb = grad_op(b, 1), ia = inverse(a), ib = inverse(b);
    plan({gb, ib, ga, ia}, {0, -1, 0, -1});
    // the kernel sums a gradient term in the sweep of the inverse next to it
    refuses("gradient_last", [&] { plan({ia, ga}, {-1, 0}); });
    refuses("gradient_before_another_inverse", [&] { plan({ga, ib, ia}, {0, -1, -1}); });
    refuses("gradient_before_a_forward_gadget", [&] { plan({ga, a}, {0, 1}); });
    // a wave's column blocks would leave the tile
    refuses("mfma_pass_on_a_2^11_fp64_tile", [] { mfma_pass<double>(11); });
    refuses("mfma_pass_on_a_2^11_fp32_tile", [] { mfma_pass<float>(11); });
    return failures ? 1 : 0;
}
