#include "svm_terms.h"

extern "C" uint64_t limit(uint64_t ops, uint32_t rank, uint32_t params) { return csvm::term_limit(ops, rank, params); }
