// svm_terms.hip -- kernel of the expectation values and gradients given as
// sums of products of sines and cosines (svm_terms.h).
#include "svm_internal.h"

namespace csvm {

// Row stride of the per-lane tables: odd, so that 64 lanes reading down 64
// rows meet different banks.
constexpr uint32_t kTermRow = 65;
static uint32_t term_lds(uint32_t num_params) { return (4u * 64u + 2u * num_params * kTermRow) * 8u; }

CSVM_INLINE static void term_fence() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// One wavefront per angle vector, one term per lane: the products before and
// after each factor give every derivative without a division (a factor may be
// zero), and each lane adds its terms' derivatives up in its own column, so
// the sums' order does not depend on the launch.
// What bounds it: up to 64 terms the launch (512 vectors of 16 angles with 32
// probes, one term each, take 9 us; the adjoint sweeps, 77 MB of state a
// vector, 6.1 ms), beyond that the two walks over the parameters, 5.5 ns a
// term and parameter.  A lane per probe and per parameter, the other factors
// multiplied anew for each, took 20 times as long at 1000 terms (2400 us
// against 124 at 20 parameters).
__global__ void __launch_bounds__(64) term_kernel(TermArgs A) {
    extern __shared__ double lds[];
    const uint32_t lane = threadIdx.x, np = A.num_params, nt = A.num_terms;
    double *co = lds, *si = lds + 64, *value = lds + 128, *carry = lds + 192;
    double *before = lds + 256, *sum = before + np * kTermRow;  // [parameter][lane]
    // A weight that is not finite spreads over the whole state of the sweeps
    // (svm_adjoint.h): no angle held at its probe has a derivative.
    uint64_t lost = 0;
    if (A.grad_out) {
        for (uint32_t j = lane; j < A.num_ev; j += 64u)
            if (!isfinite(A.coeffs[j])) lost |= A.before[j];
        if (__any(lost != 0))
            for (int o = 32; o; o >>= 1) lost |= __shfl_xor(lost, o, 64);
    }
    for (uint64_t b = blockIdx.x; b < A.batch; b += gridDim.x) {
        bool finite = true;
        if (lane < np) {
            const double a = A.psign[lane] * A.thetas[b * np + lane];
            finite = isfinite(a);
            sincos(a, si + lane, co + lane);
        }
        const uint64_t bad = __ballot(!finite) & A.active;
        term_fence();
        double* ev = A.ev_out ? A.ev_out + b * A.num_ev : nullptr;
        auto finish = [&](uint32_t j, double v) {
            if (v > 1.0) v = 1.0;
            if (v < -1.0) v = -1.0;
            if (bad & A.before[j]) v = 0.0;  // a state that is not finite has no norm
            ev[j] = v;
        };
        if (ev)
            for (uint32_t j = lane; j < A.num_ev; j += 64u)
                if (A.first[j] == A.first[j + 1u]) finish(j, 0.0);
        if (A.grad_out)
            for (uint32_t i = 0; i < np; ++i) sum[i * kTermRow + lane] = 0.0;
        for (uint32_t t0 = 0; t0 < nt; t0 += 64u) {
            const uint32_t t = t0 + lane, end = t0 + 64u < nt ? t0 + 64u : nt;
            AdjTerm x{0.0, 0, 0, 0, 0};
            if (t < nt) x = A.terms[t];
            double v = x.coef;
            for (uint32_t i = 0; i < np; ++i) {
                const bool c = (x.cos_of >> i) & 1u, s = (x.sin_of >> i) & 1u;
                if (A.grad_out) before[i * kTermRow + lane] = v;
                v *= c ? co[i] : s ? si[i] : 1.0;
            }
            if (A.grad_out) {
                double after = t < nt ? A.coeffs[x.probe] : 0.0;
                for (uint32_t i = np; i-- > 0;) {
                    const bool c = (x.cos_of >> i) & 1u, s = (x.sin_of >> i) & 1u;
                    const double cs = co[i], sn = si[i], d = c ? -sn : cs;
                    if (c || s) sum[i * kTermRow + lane] += before[i * kTermRow + lane] * after * d;
                    after *= c ? cs : s ? sn : 1.0;
                }
            }
            if (ev) {  // each probe's terms lie side by side; one probe at most goes on in the next 64
                term_fence();
                value[lane] = v;
                term_fence();
                const uint32_t p0 = A.terms[t0].probe, p1 = A.terms[end - 1u].probe;
                for (uint32_t j = p0 + lane; j <= p1; j += 64u) {
                    const uint32_t f = A.first[j], g = A.first[j + 1u];
                    if (f == g) continue;
                    double y = f < t0 ? *carry : 0.0;
                    for (uint32_t e = f < t0 ? t0 : f; e < (g < end ? g : end); ++e) y += value[e - t0];
                    if (g > end)
                        *carry = y;
                    else
                        finish(j, y);
                }
            }
        }
        term_fence();
        if (A.grad_out && lane < np) {
            double g = 0.0;
            const uint32_t lanes = nt < 64u ? nt : 64u;
            for (uint32_t l = 0; l < lanes; ++l) g += sum[lane * kTermRow + l];
            const double nan = __longlong_as_double(0x7FF8000000000000ll);
            A.grad_out[b * np + lane] = !((A.active >> lane) & 1u) ? 0.0 : bad || ((lost >> lane) & 1u) ? nan : g * A.psign[lane];
        }
        term_fence();
    }
}

hipError_t launch_terms(const TermArgs& A, uint32_t num_cus, hipStream_t st) {
    const uint32_t lds = term_lds(A.num_params);
    if (lds > 64u * 1024u) {
        const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(term_kernel),
                                                 hipFuncAttributeMaxDynamicSharedMemorySize, (int)term_lds(64));
        if (e != hipSuccess) return e;
    }
    const uint64_t most = 16ull * num_cus;
    hipLaunchKernelGGL(term_kernel, dim3((uint32_t)(A.batch < most ? A.batch : most)), dim3(64), lds, st, A);
    return hipGetLastError();
}

}  // namespace csvm
