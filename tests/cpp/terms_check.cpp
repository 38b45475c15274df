// A TermPlan's values and gradients as plain scalar code, for the CPU test.
#include <vector>

#include "svm_terms.h"

using namespace csvm;

// Returns the number of terms, or -1 when the planner refuses the program.
extern "C" int64_t terms_eval(const clifft_program_view* v, const int32_t* rank, const int32_t* slot_of, uint32_t np,
                              uint64_t limit, const double* angle, double* ev, double* grad) {
    TermPlanner planner(v->bytecode, v->num_instructions, rank, slot_of, np, v->num_exp_vals, v->ev_x, v->ev_z, v->ev_sign,
                        v->words);
    const TermPlan P = planner.run(limit);
    if (!P.ok) return -1;
    for (uint32_t j = 0; j < v->num_exp_vals; ++j) {
        ev[j] = 0;
        for (uint32_t i = 0; i < np; ++i) grad[j * np + i] = 0;
        for (uint32_t t = P.first[j]; t < P.first[j + 1]; ++t) {
            const AdjTerm& x = P.terms[t];
            if (x.probe != j) return -2;
            for (uint32_t d = 0; d <= np; ++d) {  // the value, then each derivative
                double y = x.coef;
                if (d < np && !(((x.cos_of | x.sin_of) >> d) & 1)) continue;
                for (uint32_t i = 0; i < np; ++i) {
                    const bool c = (x.cos_of >> i) & 1, s = (x.sin_of >> i) & 1;
                    if (c) y *= i == d ? -std::sin(angle[i]) : std::cos(angle[i]);
                    if (s) y *= i == d ? std::cos(angle[i]) : std::sin(angle[i]);
                }
                (d < np ? grad[j * np + d] : ev[j]) += y;
            }
        }
    }
    return (int64_t)P.terms.size();
}
