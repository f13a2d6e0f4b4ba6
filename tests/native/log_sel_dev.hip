// The branch-free logarithm of csrc/fastmath.hh next to the branching one, over
// device arrays. Test support only; the product library does not export it.
#include <hip/hip_runtime.h>

#include <cstdint>

#include "../../noa_amd/csrc/fastmath.hh"

namespace {

__global__ __launch_bounds__(256) void log_kernel(const double* __restrict__ x, int64_t n, double* __restrict__ sel,
                                                  double* __restrict__ ref) {
    namespace fm = noa_hip::fm;
    __shared__ __attribute__((aligned(fm::TABLE_LDS_ALIGN))) double block[fm::TABLE_DOUBLES];
    for (int i = threadIdx.x; i < fm::TABLE_DOUBLES; i += blockDim.x) block[i] = fm::table_entry(i);
    __syncthreads();
    const fm::Tab t = fm::tab_from_block(block);
    for (int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; i < n; i += int64_t(gridDim.x) * blockDim.x) {
        sel[i] = fm::log_sel(x[i], t);
        ref[i] = fm::log(x[i], t);
    }
}

}  // namespace

extern "C" int log_sel_eval(const double* x, int64_t n, double* sel, double* ref) {
    if (n < 1) return 1;
    const int64_t blocks = (n + 255) / 256;
    hipLaunchKernelGGL(log_kernel, dim3(unsigned(blocks < 1024 ? blocks : 1024)), dim3(256), 0, nullptr, x, n, sel, ref);
    if (hipGetLastError() != hipSuccess) return 2;
    return hipDeviceSynchronize() == hipSuccess ? 0 : 3;
}
