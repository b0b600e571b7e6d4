// FP64 kernels: the reference's arithmetic, bit-exact.  Built with
// -ffp-contract=off so no multiply-add is fused.
#define HF_MATH MathF64
#include "hf_kernels_inst.h"

namespace hf {
namespace {
__global__ __launch_bounds__(256) void k_clear(const ClearArgs a)
{
    for (int k = 0; k < HF_CLEARS; k++)
        for (int i = blockIdx.x * 256 + threadIdx.x; i < a.n[k]; i += gridDim.x * 256) a.p[k][i] = 0u;
}
}  // namespace

hipError_t launch_clear(const ClearArgs& a, hipStream_t s)
{
    int most = 0;
    for (int n : a.n) most = n > most ? n : most;
    const int grid = most > 256 * 64 ? 64 : (most + 255) / 256;
    if (grid > 0) hipLaunchKernelGGL(k_clear, dim3(grid), dim3(256), 0, s, a);
    return hipGetLastError();
}
}  // namespace hf
