//----------------------------------*-C++-*----------------------------------//
// celeritas_amd: MI355X-native per-step transport loop
//---------------------------------------------------------------------------//
//! \file corecel/ElementaryVerify.hip
//! Runs the step kernels' FP64 logarithm, sine and cosine on given arguments.
//---------------------------------------------------------------------------//
#include "celeritas_amd.h"

#include <hip/hip_runtime.h>

#include "Elementary.hh"

namespace celeritas_amd
{
namespace
{
constexpr int block_size = 256;

//! Logarithms, sines and cosines of n arguments, one array after the other
__global__ void __launch_bounds__(block_size)
    verify_elementary_kernel(double const* __restrict__ x,
                             std::uint32_t const n,
                             double* __restrict__ out)
{
    std::uint32_t const t = blockIdx.x * block_size + threadIdx.x;
    if (t >= n)
        return;
    out[t] = elem::log(x[t]);
    elem::sincos(x[t], &out[std::size_t(n) + t], &out[2 * std::size_t(n) + t]);
}
}  // namespace
}  // namespace celeritas_amd

using namespace celeritas_amd;

extern "C" int
celer_verify_elementary(const double* x, uint32_t n, double* out, void* stream)
{
    auto st = static_cast<hipStream_t>(stream);
    if (n == 0)
        return 0;
    std::size_t const bytes = sizeof(double) * std::size_t(n);
    double* d_x = nullptr;
    double* d_o = nullptr;
    hipError_t err = hipSuccess;
    auto check = [&](hipError_t e) {
        if (err == hipSuccess)
            err = e;
    };
    check(hipMalloc(&d_x, bytes));
    check(hipMalloc(&d_o, 3 * bytes));
    if (err == hipSuccess)
    {
        check(hipMemcpyAsync(d_x, x, bytes, hipMemcpyHostToDevice, st));
        verify_elementary_kernel<<<(n - 1) / block_size + 1, block_size, 0, st>>>(d_x, n, d_o);
        check(hipGetLastError());
        check(hipMemcpyAsync(out, d_o, 3 * bytes, hipMemcpyDeviceToHost, st));
        check(hipStreamSynchronize(st));
    }
    (void)hipFree(d_x);
    (void)hipFree(d_o);
    return static_cast<int>(err);
}
