// The shared-state executor's rules of dispatch on a program's plan, for the
// CPU test.
#include "svm_tree_plan.h"
#include "svm_tree_shape.h"

using namespace csvm;

static bool profile(const clifft_program_view* v, const int32_t* khist, TreeProfile& p) {
    const std::vector<int32_t> kh(khist, khist + v->num_instructions);
    const TreePlan plan = TreePlanner(v, kh).run();
    p.ok = plan.ok;
    p.code = (uint32_t)plan.code.size();
    p.words = plan.words;
    p.set_program(v);
    p.set_passes(plan.sizes);
    return plan.ok;
}

// copies: in a batch of so many like it, 0: a launch of its own.  out: threads, shots a team, entries a buffer, LDS bytes, buffers in memory;
// 0: on the per-shot executors, -1: no plan
extern "C" int shape(const clifft_program_view* v, const int32_t* khist, uint64_t shots, uint32_t faults, uint32_t cus, int mode,
                     uint32_t copies, uint64_t* out) {
    TreeProfile p;
    if (!profile(v, khist, p)) return -1;
    TreeShape s;
    if (copies) {
        s = tree_batch(std::vector<const TreeProfile*>(copies, &p), std::vector<uint64_t>(copies, shots), cus, mode)[0];
        if (!s.threads) return 0;
    } else if (!tree_shape(p, shots, faults, cus, mode, s)) {
        return 0;
    }
    out[0] = s.threads, out[1] = s.chunk, out[2] = s.elems, out[3] = s.lds, out[4] = s.global;
    return 1;
}
