// Self-check of the EXACT division sequences (vg_quot.h) against the
// compiler's IEEE division, on the device.  No counterpart in the reference:
// the check behind the claim that the shortened sequences round like the IEEE
// division wherever the solvers use them.
#include <cstdint>

#include "vg_quot.h"
#include "vg_runtime.h"

namespace {

__global__ __launch_bounds__(256) void division_check_kernel(const double *a, const double *b, long long n,
                                                             double *shared_q, double *in_range_q, double *ieee_q)
{
    const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const double x = a[i], y = b[i];
    const vg::SharedDivisor d = vg::shared_divisor(y);
    shared_q[i] = vg::quot(x, d);
    in_range_q[i] = vg::div_in_range(x, y);
    ieee_q[i] = x / y;
}

__global__ __launch_bounds__(256) void scaled_division_check_kernel(const double *a, const double *b, const double *c,
                                                                    long long n, double *scaled_q, double *ieee_q)
{
    const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const double x = a[i], y = b[i], z = c[i];
    const vg::SharedDivisor d = vg::shared_divisor(y);
    scaled_q[i] = (d.fast && vg::scale_in_range(z)) ? vg::quot_scaled(x, d, z, 1.0 / z) : x / (z * y);
    ieee_q[i] = x / (z * y);
}

__global__ __launch_bounds__(256) void third_check_kernel(const double *a, long long n, double *third_q, double *ieee_q)
{
    const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    third_q[i] = vg::third(a[i]);
    ieee_q[i] = a[i] / 3.0;
}

}  // namespace

extern "C" int vg_third_selfcheck(vg_ctx *ctx, int64_t n, const double *a, double *third_q, double *ieee_q)
{
    vg::clear_error();
    VG_CHECK(ctx != nullptr && a && third_q && ieee_q, "null argument");
    VG_CHECK(n >= 1 && n <= (int64_t(1) << 26), "n must be in 1 .. 2^26");
    int rc = vg::bind(ctx);
    if (rc) return rc;
    const size_t bytes = sizeof(double) * (size_t)n;
    double *buf = nullptr;
    VG_HIP(hipMalloc(&buf, 3 * bytes));
    hipStream_t s = ctx->stream;
    hipError_t e = hipMemcpyAsync(buf, a, bytes, hipMemcpyHostToDevice, s);
    if (e == hipSuccess) {
        third_check_kernel<<<(unsigned)((n + 255) / 256), 256, 0, s>>>(buf, n, buf + n, buf + 2 * n);
        e = hipGetLastError();
    }
    if (e == hipSuccess) e = hipMemcpyAsync(third_q, buf + n, bytes, hipMemcpyDeviceToHost, s);
    if (e == hipSuccess) e = hipMemcpyAsync(ieee_q, buf + 2 * n, bytes, hipMemcpyDeviceToHost, s);
    if (e == hipSuccess) e = hipStreamSynchronize(s);
    hipFree(buf);
    if (e != hipSuccess) {
        vg::set_error(std::string("vg_third_selfcheck: ") + hipGetErrorString(e));
        return VG_ERR_HIP;
    }
    return VG_OK;
}

extern "C" int vg_scaled_division_selfcheck(vg_ctx *ctx, int64_t n, const double *a, const double *b, const double *c,
                                            double *scaled_q, double *ieee_q)
{
    vg::clear_error();
    VG_CHECK(ctx != nullptr && a && b && c && scaled_q && ieee_q, "null argument");
    VG_CHECK(n >= 1 && n <= (int64_t(1) << 26), "n must be in 1 .. 2^26");
    int rc = vg::bind(ctx);
    if (rc) return rc;
    const size_t bytes = sizeof(double) * (size_t)n;
    double *buf = nullptr;
    VG_HIP(hipMalloc(&buf, 5 * bytes));
    hipStream_t s = ctx->stream;
    const double *in[3] = {a, b, c};
    hipError_t e = hipSuccess;
    for (int k = 0; k < 3 && e == hipSuccess; k++)
        e = hipMemcpyAsync(buf + k * n, in[k], bytes, hipMemcpyHostToDevice, s);
    if (e == hipSuccess) {
        scaled_division_check_kernel<<<(unsigned)((n + 255) / 256), 256, 0, s>>>(buf, buf + n, buf + 2 * n, n,
                                                                                buf + 3 * n, buf + 4 * n);
        e = hipGetLastError();
    }
    if (e == hipSuccess) e = hipMemcpyAsync(scaled_q, buf + 3 * n, bytes, hipMemcpyDeviceToHost, s);
    if (e == hipSuccess) e = hipMemcpyAsync(ieee_q, buf + 4 * n, bytes, hipMemcpyDeviceToHost, s);
    if (e == hipSuccess) e = hipStreamSynchronize(s);
    hipFree(buf);
    if (e != hipSuccess) {
        vg::set_error(std::string("vg_scaled_division_selfcheck: ") + hipGetErrorString(e));
        return VG_ERR_HIP;
    }
    return VG_OK;
}

extern "C" int vg_division_selfcheck(vg_ctx *ctx, int64_t n, const double *a, const double *b, double *shared_q,
                                     double *in_range_q, double *ieee_q)
{
    vg::clear_error();
    VG_CHECK(ctx != nullptr && a && b && shared_q && in_range_q && ieee_q, "null argument");
    VG_CHECK(n >= 1 && n <= (int64_t(1) << 26), "n must be in 1 .. 2^26");
    int rc = vg::bind(ctx);
    if (rc) return rc;
    const size_t bytes = sizeof(double) * (size_t)n;
    double *buf = nullptr;
    VG_HIP(hipMalloc(&buf, 5 * bytes));
    double *da = buf, *db = buf + n, *d0 = buf + 2 * n, *d1 = buf + 3 * n, *d2 = buf + 4 * n;
    hipStream_t s = ctx->stream;
    hipError_t e = hipMemcpyAsync(da, a, bytes, hipMemcpyHostToDevice, s);
    if (e == hipSuccess) e = hipMemcpyAsync(db, b, bytes, hipMemcpyHostToDevice, s);
    if (e == hipSuccess) {
        division_check_kernel<<<(unsigned)((n + 255) / 256), 256, 0, s>>>(da, db, n, d0, d1, d2);
        e = hipGetLastError();
    }
    if (e == hipSuccess) e = hipMemcpyAsync(shared_q, d0, bytes, hipMemcpyDeviceToHost, s);
    if (e == hipSuccess) e = hipMemcpyAsync(in_range_q, d1, bytes, hipMemcpyDeviceToHost, s);
    if (e == hipSuccess) e = hipMemcpyAsync(ieee_q, d2, bytes, hipMemcpyDeviceToHost, s);
    if (e == hipSuccess) e = hipStreamSynchronize(s);
    hipFree(buf);
    if (e != hipSuccess) {
        vg::set_error(std::string("vg_division_selfcheck: ") + hipGetErrorString(e));
        return VG_ERR_HIP;
    }
    return VG_OK;
}
