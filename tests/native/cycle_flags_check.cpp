// Host-side check of the end flags of a GMRES cycle (vivlasov1d_amd/csrc/
// gmres_dev.h, the functions the kernels themselves call).  A launch that
// carries a Hessenberg update or a cycle's start runs it in its first
// workgroup while its other workgroups ask, wavefront by wavefront, whether
// the instance is done.  So for every launch of every history of solves
//   * the answer is the same before and after what the first workgroup writes;
//   * it is "done" exactly when the instance's cycle had ended as of the launch
//     before (at a start: when it does not take part).
// Histories: solves of 1 .. 3 cycles of 1 .. 8 steps, three instances that end
// at every step or start, by convergence or by the cycle's length, or do not
// take part, one solve after another on the same states.
// Prints "checked L launches, F failures"; exit status 1 on any failure.
#include <cstdio>
#include <cstring>
#include <random>
#include <vector>

#include "../../vivlasov1d_amd/csrc/gmres_dev.h"

using namespace vv;

static long launches = 0, failures = 0;

static void expect(bool ok, const char *what, int start, int it, int b)
{
    if (!ok && failures++ < 20) std::printf("FAIL %s start=%d it=%d instance %d\n", what, start, it, b);
}

struct Instance {
    bool part = true, over = false, done = true;   // takes part; solve ended; cycle ended
    int end_cycle = 0, end_step = 0;               // converges at this cycle's step (-1: at its start; past the last: never)
};

// the writes of hess_update at the end of step it, by the flags it sets
static void step_writes(GmresState *g, int it, bool converged, int max_k)
{
    if (g->st.done) {
        set_skip(g, it, true);
        return;
    }
    g->st.it = it + 1;
    if (converged) g->st.reason = VV_KSP_CONVERGED_RTOL;
    const bool end = converged || g->st.it >= max_k;
    if (end) g->st.done = 1;
    set_skip(g, it, end);
}

int main()
{
    std::mt19937 rng(7);
    auto pick = [&](int lo, int hi) { return lo + (int)(rng() % (unsigned)(hi - lo + 1)); };
    const int B = 3;
    std::vector<GmresState> gs(B);
    std::memset(static_cast<void *>(gs.data()), 0, B * sizeof(GmresState));
    for (int solve = 0; solve < 4000; ++solve) {
        const int max_k = pick(1, 8), max_cycles = pick(1, 3);
        std::vector<Instance> in(B);
        std::vector<int32_t> active(B);
        for (int b = 0; b < B; ++b) {
            in[b].part = pick(0, 4) != 0;
            in[b].end_cycle = pick(0, max_cycles);
            in[b].end_step = pick(-1, max_k - 1);
            active[b] = in[b].part;
        }
        for (int cycle = 0; cycle < max_cycles; ++cycle) {
            HessArgs a{};
            a.it = -1;
            a.start = cycle == 0 ? 2 : 1;
            a.init = SolveStart{active.data(), 1e-8, 1e-50, 1e5, 1000, max_k};
            for (int b = 0; b < B; ++b) {
                GmresState *g = &gs[b];
                Instance &s = in[b];
                const bool before = carried_skip(a, g, b), out = !s.part || s.over;
                expect(before == out, "answer at a start", a.start, -1, b);
                const bool conv = s.end_cycle == cycle && s.end_step == -1;
                // a first start converges on a zero right-hand side, a restart within ttol
                cycle_start(a, g, b, conv ? 0.0 : 1.0);
                expect(carried_skip(a, g, b) == before, "start's own writes", a.start, -1, b);
                if (!out && conv) s.over = true;
                s.done = out || conv;
                ++launches;
            }
            a.start = 0;
            // the host stops once every instance is done, at the earliest one step late
            bool all = false;
            for (int it = 0; it < max_k && !all; ++it) {
                all = true;
                for (int b = 0; b < B; ++b) all = all && in[b].done;
                a.it = it;
                for (int b = 0; b < B; ++b) {
                    GmresState *g = &gs[b];
                    Instance &s = in[b];
                    const bool before = carried_skip(a, g, b);
                    expect(before == s.done, "answer at a step", 0, it, b);
                    const bool conv = !s.done && s.end_cycle == cycle && s.end_step == it;
                    step_writes(g, it, conv, max_k);
                    expect(carried_skip(a, g, b) == before, "update's own writes", 0, it, b);
                    if (conv) s.over = true;
                    if (conv || it + 1 >= max_k) s.done = true;
                    ++launches;
                }
            }
            // update_kernel, the cycle's last launch
            for (int b = 0; b < B; ++b) gs[b].over = !gs[b].st.active || gs[b].st.reason != 0;
        }
    }
    std::printf("checked %ld launches, %ld failures\n", launches, failures);
    return failures != 0;
}
