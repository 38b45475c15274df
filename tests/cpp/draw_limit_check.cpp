#include "svm_tree_plan.h"

extern "C" uint64_t limit(double p) { return csvm::draw_limit(p); }
