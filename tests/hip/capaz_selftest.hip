// Device self-tests of the kernels' arithmetic building blocks (test
// infrastructure, built by capaz_amd/build.py into tests/hip/): each compares
// a rewritten operation with the plain IEEE operation it replaces, on the
// GPU, and counts mismatching bit patterns.
#include <hip/hip_runtime.h>

#include <cstdint>

#include "capaz_cell.h"
#include "capaz_derive.h"

namespace {

__device__ uint64_t mix(uint64_t x) {  // splitmix64 finaliser
    x += 0x9E3779B97F4A7C15ull;
    x = (x ^ (x >> 30)) * 0xBF58476D1CE4E5B9ull;
    x = (x ^ (x >> 27)) * 0x94D049BB133111EBull;
    return x ^ (x >> 31);
}

// Random doubles: uniform significand and sign, exponent in [emin, emax];
// every 16th draw has an all-ones significand, every 16th a power of two.
__device__ double draw(uint64_t seed, uint64_t i, int emin, int emax) {
    uint64_t r = mix(seed ^ mix(i));
    uint64_t mant = r & ((1ull << 52) - 1);
    uint64_t sel = (r >> 52) & 15;
    if (sel == 0) mant = (1ull << 52) - 1;
    if (sel == 1) mant = 0;
    int e = emin + (int)(mix(r) % (uint64_t)(emax - emin + 1));
    uint64_t bits = ((uint64_t)(e + 1023) << 52) | mant | ((r >> 63) << 63);
    return __longlong_as_double((long long)bits);
}

__global__ void k_rcp(uint64_t n, uint64_t seed, int emin, int emax, unsigned long long* bad) {
    uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
    unsigned long long local = 0;
    for (; i < n; i += stride) {
        double b = draw(seed, i, emin, emax);
        double want = 1. / b, got = capaz::rcp_rn(b);
        if (__double_as_longlong(want) != __double_as_longlong(got)) ++local;
    }
    if (local) atomicAdd(bad, local);
}

__global__ void k_rcp_in_range(uint64_t n, uint64_t seed, int emin, int emax, unsigned long long* bad) {
    uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
    unsigned long long local = 0;
    for (; i < n; i += stride) {
        double b = draw(seed, i, emin, emax);
        double want = 1. / b, got = capaz::rcp_in_range(b);
        if (__double_as_longlong(want) != __double_as_longlong(got)) ++local;
    }
    if (local) atomicAdd(bad, local);
}

__global__ void k_div(uint64_t n, uint64_t seed, int emin, int emax, unsigned long long* bad) {
    uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
    unsigned long long local = 0;
    for (; i < n; i += stride) {
        double a = draw(seed, 2 * i, emin, emax), b = draw(seed, 2 * i + 1, emin, emax);
        double want = a / b;
        double got = capaz::exact_div(a, b, capaz::rcp_rn(b));
        if (__double_as_longlong(want) != __double_as_longlong(got)) ++local;
    }
    if (local) atomicAdd(bad, local);
}

// log_cl exists on the device only (the host build of the closures calls pow)
__global__ void k_log(const double* x, double* y, uint64_t n) {
#if defined(__HIP_DEVICE_COMPILE__)
    const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) y[i] = capaz::log_cl(x[i]);
#else
    (void)x, (void)y, (void)n;
#endif
}

__global__ void k_pow(const double* x, double e, double* y, uint64_t n) {
    const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) y[i] = capaz::pow_cl(x[i], e);
}

__global__ void k_map(int which, const double* x, double* y, uint64_t n) {
    const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) y[i] = which == 0 ? capaz::pow_half(x[i]) : capaz::pow_two(x[i]);
}

// A cell's closure and, for two phases, its Newton with the powers that go
// without selects (p.pow_fast) and without: differing values (NaNs aside).
__global__ void k_closures(capaz::DevParams p, const double* x, const double* y, uint64_t n, unsigned long long* bad) {
#if defined(__HIP_DEVICE_COMPILE__)
    const uint64_t l = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (l >= n) return;
    auto differ = [](double a, double b) {
        return __double_as_longlong(a) != __double_as_longlong(b) && !(a != a && b != b);
    };
    capaz::DevParams g = p;
    g.pow_fast = 0;
    double a[3] = {}, b[3] = {};
    if (p.model == 3) {
        capaz::relperm3(p, x[l], y[l], a[0], a[1], a[2]);
        capaz::relperm3(g, x[l], y[l], b[0], b[1], b[2]);
    } else {
        capaz::relperm2(p, x[l], a[0], a[1], a[2]);
        capaz::relperm2(g, x[l], b[0], b[1], b[2]);
    }
    bool d = differ(a[0], b[0]) || differ(a[1], b[1]) || differ(a[2], b[2]);
    if (p.model == 2) {
        double P[2] = {1.1e5, 1.1e5}, S[2] = {x[l], x[l]};
        const double rw = 0.4 * p.ro0_w * (1 - y[l]), rn = 0.4 * p.ro0_n * y[l];
        if (capaz::newton2_fast<0>(p, P[0], S[0], rw, rn)) {
            capaz::newton2_ieee<0>(p, P[1], S[1], rw, rn);
            d = d || differ(P[0], P[1]) || differ(S[0], S[1]);
        }
    }
    if (d) atomicAdd(bad, 1ull);
#else
    (void)p, (void)x, (void)y, (void)n, (void)bad;
#endif
}

}  // namespace

extern "C" {

// Number of the n states (two phases: S_n = x and, for Newton's right side,
// y; three: S_w = x, S_n = y) whose reference closure, with the exponent
// lambda, differs with and without its powers' selects; -1 on a HIP error, -2
// if the exponent has no path without them.
long long capaz_selftest_closures(int model, double lambda, const double* x, const double* y, unsigned long long n) {
    capaz_params u = {};
    u.model = model;
    u.Nx = u.Ny = u.Nz = 3;
    u.hx = u.hy = u.hz = u.dt = 1.;
    u.newton_iterations = 3;
    u.P_atm = 1e5;
    u.mu_w = u.mu_n = u.mu_g = 1e-3;
    u.ro0_w = 1000., u.ro0_n = 1460., u.ro0_g = 1.4;
    u.beta_w = u.beta_n = 4.4e-10;
    u.lambda = lambda;
    u.S_wr = 0.09, u.S_nr = 0.05, u.S_gr = 0.01;
    u.P_d = 755.;
    const capaz::DevParams p = capaz::derive(u);
    if (!p.pow_fast) return -2;
    double *dx = nullptr, *dy = nullptr;
    unsigned long long *d = nullptr, h = 0;
    long long rc = -1;
    const size_t b = n * sizeof(double);
    if (hipMalloc(&dx, b) == hipSuccess && hipMalloc(&dy, b) == hipSuccess && hipMalloc(&d, sizeof(h)) == hipSuccess &&
        hipMemcpy(dx, x, b, hipMemcpyHostToDevice) == hipSuccess &&
        hipMemcpy(dy, y, b, hipMemcpyHostToDevice) == hipSuccess &&
        hipMemcpy(d, &h, sizeof(h), hipMemcpyHostToDevice) == hipSuccess) {
        hipLaunchKernelGGL(k_closures, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, 0, p, dx, dy, (uint64_t)n, d);
        if (hipGetLastError() == hipSuccess && hipMemcpy(&h, d, sizeof(h), hipMemcpyDeviceToHost) == hipSuccess)
            rc = (long long)h;
    }
    if (dx) (void)hipFree(dx);
    if (dy) (void)hipFree(dy);
    if (d) (void)hipFree(d);
    return rc;
}

// y = pow_half(x) (which = 0) or pow_two(x) (which = 1) on the device for n
// host doubles; 0, or -1 on a HIP error.
int capaz_selftest_map(int which, const double* x, double* y, unsigned long long n) {
    double *dx = nullptr, *dy = nullptr;
    int rc = -1;
    if (hipMalloc(&dx, n * sizeof(double)) == hipSuccess && hipMalloc(&dy, n * sizeof(double)) == hipSuccess &&
        hipMemcpy(dx, x, n * sizeof(double), hipMemcpyHostToDevice) == hipSuccess) {
        hipLaunchKernelGGL(k_map, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, 0, which, dx, dy, (uint64_t)n);
        if (hipGetLastError() == hipSuccess && hipMemcpy(y, dy, n * sizeof(double), hipMemcpyDeviceToHost) == hipSuccess)
            rc = 0;
    }
    if (dx) (void)hipFree(dx);
    if (dy) (void)hipFree(dy);
    return rc;
}

// y = log_cl(x) on the device (the closures' powers' log) for n host doubles;
// 0, or -1 on a HIP error.
int capaz_selftest_log(const double* x, double* y, unsigned long long n) {
    double *dx = nullptr, *dy = nullptr;
    int rc = -1;
    if (hipMalloc(&dx, n * sizeof(double)) == hipSuccess && hipMalloc(&dy, n * sizeof(double)) == hipSuccess &&
        hipMemcpy(dx, x, n * sizeof(double), hipMemcpyHostToDevice) == hipSuccess) {
        hipLaunchKernelGGL(k_log, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, 0, dx, dy, (uint64_t)n);
        if (hipGetLastError() == hipSuccess && hipMemcpy(y, dy, n * sizeof(double), hipMemcpyDeviceToHost) == hipSuccess)
            rc = 0;
    }
    if (dx) (void)hipFree(dx);
    if (dy) (void)hipFree(dy);
    return rc;
}

// y = pow_cl(x, e) on the device (the closures' powers) for n host doubles;
// 0, or -1 on a HIP error.
int capaz_selftest_pow(const double* x, double e, double* y, unsigned long long n) {
    double *dx = nullptr, *dy = nullptr;
    int rc = -1;
    if (hipMalloc(&dx, n * sizeof(double)) == hipSuccess && hipMalloc(&dy, n * sizeof(double)) == hipSuccess &&
        hipMemcpy(dx, x, n * sizeof(double), hipMemcpyHostToDevice) == hipSuccess) {
        hipLaunchKernelGGL(k_pow, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, 0, dx, e, dy, (uint64_t)n);
        if (hipGetLastError() == hipSuccess && hipMemcpy(y, dy, n * sizeof(double), hipMemcpyDeviceToHost) == hipSuccess)
            rc = 0;
    }
    if (dx) (void)hipFree(dx);
    if (dy) (void)hipFree(dy);
    return rc;
}

// Number of draws where rcp_rn(b) != 1.0/b (which = 0),
// exact_div(a, b, rcp_rn(b)) != a/b (which = 1) or rcp_in_range(b) != 1.0/b
// (which = 2); -1 on a HIP error.
long long capaz_selftest(int which, unsigned long long n, unsigned long long seed, int emin, int emax) {
    unsigned long long* d = nullptr;
    if (hipMalloc(&d, sizeof(*d)) != hipSuccess) return -1;
    if (hipMemset(d, 0, sizeof(*d)) != hipSuccess) return -1;
    if (which == 0)
        hipLaunchKernelGGL(k_rcp, dim3(4096), dim3(256), 0, 0, (uint64_t)n, (uint64_t)seed, emin, emax, d);
    else if (which == 2)
        hipLaunchKernelGGL(k_rcp_in_range, dim3(4096), dim3(256), 0, 0, (uint64_t)n, (uint64_t)seed, emin, emax, d);
    else
        hipLaunchKernelGGL(k_div, dim3(4096), dim3(256), 0, 0, (uint64_t)n, (uint64_t)seed, emin, emax, d);
    unsigned long long h = 0;
    if (hipMemcpy(&h, d, sizeof(h), hipMemcpyDeviceToHost) != hipSuccess) return -1;
    (void)hipFree(d);
    return (long long)h;
}

}  // extern "C"
