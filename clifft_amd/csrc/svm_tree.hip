// svm_tree.hip -- kernels of the shared-state executor (svm_tree.h) and
// their launchers.
#include <atomic>

#include "svm_internal.h"
#include "svm_tree.h"

namespace csvm {

// One program: workgroups stride over the launch's chunks of shots.
template <class FW, class AmpT>
__global__ void __launch_bounds__(1024, 4) tree_kernel(const DevProgram* P, const ShotArgs* A) {
    cptr<ShotArgs> Ag = cp(A);
    dv2* buf = Ag->gscratch ? Ag->gscratch + (size_t)blockIdx.x * 2u * Ag->amp_elems : nullptr;
    tree_range<FW, AmpT>(cp(P), Ag, blockIdx.x, gridDim.x, 0, Ag->shot_count, Ag->seed, buf);
}

// Batched: workgroups pop items (one chunk of one program each) until the
// queue is empty.
template <class FW, class AmpT>
__global__ void __launch_bounds__(1024, 4) batch_tree_kernel(const BatchArgs* B) {
    __shared__ uint32_t head;
    cptr<BatchArgs> Bg = cp(B);
    dv2* buf = Bg->gscratch ? Bg->gscratch + (size_t)blockIdx.x * Bg->team_elems : nullptr;
    for (;;) {
        if (threadIdx.x == 0) head = atomicAdd(Bg->counter, 1u);
        __syncthreads();
        const uint32_t it = uni(head);
        __syncthreads();
        cptr<BatchArgs> Bc = opaque(Bg);
        if (it >= Bc->n_items) break;
        cptr<BatchItem> I = cp(Bc->items) + it;
        const uint32_t pid = I->prog;
        tree_range<FW, AmpT>(cp(cp(Bc->progs)[pid]), cp(Bc->args) + pid, 0, 1, I->shot_lo, I->shot_hi, cp(Bc->seeds)[pid], buf);
    }
}

template <bool BATCH>
static const void* tree_fn(const LaunchShape& L) {
#define CSVM_TREE_FN(FW, AMP) \
    (BATCH ? reinterpret_cast<const void*>(batch_tree_kernel<FW, AMP>) : reinterpret_cast<const void*>(tree_kernel<FW, AMP>))
    if (L.lane_narrow) return L.global_amps ? CSVM_TREE_FN(uint32_t, glb_d2) : CSVM_TREE_FN(uint32_t, lds_d2);
    return L.global_amps ? CSVM_TREE_FN(uint64_t, glb_d2) : CSVM_TREE_FN(uint64_t, lds_d2);
#undef CSVM_TREE_FN
}

const void* tree_kernel_fn(const LaunchShape& L, bool batch) { return batch ? tree_fn<true>(L) : tree_fn<false>(L); }

uint32_t tree_team_lds(uint32_t threads, uint32_t chunk, uint32_t rec_words) { return tree_lds_bytes(threads, chunk, rec_words); }

}  // namespace csvm
