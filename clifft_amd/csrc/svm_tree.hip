// svm_tree.hip -- kernels of the shared-state executor (svm_tree.h) and
// their launchers.
#include <atomic>

#include "svm_internal.h"
#include "svm_tree.h"

namespace csvm {

struct TreeLaunch {
    const DevProgram* P;
    ShotArgs A;
};

// One program: workgroups stride over the launch's chunks of shots.  The
// arguments are read where the launch put them.
template <class AmpT>
__global__ void __launch_bounds__(1024, 4) tree_kernel(TreeLaunch) {
    cptr<TreeLaunch> K = (cptr<TreeLaunch>)__builtin_amdgcn_kernarg_segment_ptr();
    cptr<ShotArgs> A = &K->A;
    dv2* buf = A->gscratch ? A->gscratch + (size_t)blockIdx.x * 2u * A->amp_elems : nullptr;
    tree_range<AmpT>(cp(K->P), A, blockIdx.x, gridDim.x, 0, A->shot_count, A->seed, buf);
}

// Batched: workgroups pop items (one chunk of one program each) until the
// queue is empty.
template <class AmpT>
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
        tree_range<AmpT>(cp(cp(Bc->progs)[pid]), cp(Bc->args) + pid, 0, 1, I->shot_lo, I->shot_hi, cp(Bc->seeds)[pid], buf);
    }
}

template <bool BATCH>
static const void* tree_fn(const LaunchShape& L) {
    if (BATCH)
        return L.global_amps ? reinterpret_cast<const void*>(batch_tree_kernel<glb_d2>)
                             : reinterpret_cast<const void*>(batch_tree_kernel<lds_d2>);
    return L.global_amps ? reinterpret_cast<const void*>(tree_kernel<glb_d2>)
                         : reinterpret_cast<const void*>(tree_kernel<lds_d2>);
}

const void* tree_kernel_fn(const LaunchShape& L, bool batch) { return batch ? tree_fn<true>(L) : tree_fn<false>(L); }

// (shot_occupancy, which sizes the grid, has set the dynamic-LDS limit)
hipError_t launch_tree(const LaunchShape& L, const DevProgram* P, const ShotArgs& A, hipStream_t st) {
    TreeLaunch K{P, A};
    void* args[] = {&K};
    return hipLaunchKernel(tree_kernel_fn(L, false), dim3(L.grid), dim3(L.block), args, L.lds_bytes, st);
}

}  // namespace csvm
