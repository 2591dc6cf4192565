// Library-wide pieces of libkerops_hip.so: version, per-thread error text.
#include <stdarg.h>
#include <stdio.h>

#include <mutex>

#include "common.hpp"

namespace kerops {

static thread_local char g_err[512] = "";

void set_error(const char* fmt, ...)
{
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(g_err, sizeof(g_err), fmt, ap);
    va_end(ap);
}

int check_launch(const char* what)
{
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) {
        set_error("%s: %s", what, hipGetErrorString(e));
        return KEROPS_E_LAUNCH;
    }
    return KEROPS_OK;
}

DeviceGeometry device_geometry()
{
    static std::mutex mutex;
    static DeviceGeometry known[64];  // cus == 0: not looked up yet
    const DeviceGeometry fallback{256, 8};
    int dev = -1;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) {
        (void)hipGetLastError();  // a query without a device must not leave an error behind for the next launch check
        return fallback;
    }
    std::lock_guard<std::mutex> lock(mutex);
    if (known[dev].cus == 0) {
        int cus = 0, xcds = 0;
        if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || cus <= 0) {
            (void)hipGetLastError();
            return fallback;
        }
        if (hipDeviceGetAttribute(&xcds, hipDeviceAttributeNumberOfXccs, dev) != hipSuccess || xcds <= 0) {
            (void)hipGetLastError();
            xcds = cus >= 64 ? cus / 32 : 1;  // a runtime without the attribute: 32 compute units per die
        }
        known[dev] = DeviceGeometry{cus, xcds};
    }
    return known[dev];
}

}  // namespace kerops

extern "C" int kerops_hip_version(void) { return KEROPS_HIP_VERSION; }

extern "C" const char* kerops_last_error_string(void) { return kerops::g_err; }

namespace kerops {

// Sums the rows of a partial buffer column by column in a fixed order (fp64, sum_columns) and writes scale * sum to out0
// (columns below split) or out1.  A workgroup owns 16 columns.
template <class T>
__global__ __launch_bounds__(1024) void reduce_rows_kernel(const T* __restrict__ ws, int nrows, int ncols,
                                                           float* __restrict__ out0, float* __restrict__ out1,
                                                           int split, double scale)
{
    __shared__ double part[16][17];
    const int j = blockIdx.x * 16 + threadIdx.x % 16;
    const double v = sum_columns(ws, nrows, ncols, j, ncols, part) * scale;
    if (threadIdx.x < 16 && j < ncols) {
        if (j < split) {
            out0[j] = (float)v;
        } else {
            out1[j - split] = (float)v;
        }
    }
}

// The same sums where the columns come in whole groups of 32.
// Out0, Out1: fp32, or fp16 = the fp32 result rounded once (what a cast of it gives, without the cast's launch).
template <class Out0, class Out1>
__global__ __launch_bounds__(1024) void reduce_lines_kernel(const float* __restrict__ ws, int nrows, int ncols,
                                                            Out0* __restrict__ out0, Out1* __restrict__ out1,
                                                            int split, double scale)
{
    __shared__ double part[16][33];
    const double v = sum_lines(ws, nrows, ncols, part) * scale;
    const int j = blockIdx.x * 32 + threadIdx.x;
    if (threadIdx.x < 32) {
        if (j < split) out0[j] = (Out0)(float)v;
        else out1[j - split] = (Out1)(float)v;
    }
}

void launch_reduce_rows(const float* ws, int nrows, int ncols, float* out0, float* out1, int split, double scale,
                        hipStream_t stream, bool pairs)
{
    if (pairs) {
        hipLaunchKernelGGL((reduce_rows_kernel<fp32_pair_t>), dim3(ceil_div(ncols, 16)), dim3(1024), 0, stream,
                           reinterpret_cast<const fp32_pair_t*>(ws), nrows, ncols, out0, out1, split, scale);
        return;
    }
    // A line's 32 columns per workgroup pay where the columns fill the chip.  The statistics of up to 512 channels are
    // few columns of up to 4096 rows, which a narrower split spreads over twice the workgroups (256 columns: statistics
    // and pool of (1,128,103,82,48) 105.0 us, 107.0 by lines).
    if (ncols % 32 == 0 && ncols > 1024) {
        hipLaunchKernelGGL((reduce_lines_kernel<float, float>), dim3(ncols / 32), dim3(1024), 0, stream, ws, nrows, ncols,
                           out0, out1, split, scale);
        return;
    }
    hipLaunchKernelGGL((reduce_rows_kernel<float>), dim3(ceil_div(ncols, 16)), dim3(1024), 0, stream, ws, nrows, ncols,
                       out0, out1, split, scale);
}

void launch_reduce_rows_f16(const float* ws, int nrows, int ncols, half_t* out0, float* out1, int split,
                            hipStream_t stream)
{
    hipLaunchKernelGGL((reduce_lines_kernel<half_t, float>), dim3(ncols / 32), dim3(1024), 0, stream, ws, nrows, ncols,
                       out0, out1, split, 1.0);
}

}  // namespace kerops
