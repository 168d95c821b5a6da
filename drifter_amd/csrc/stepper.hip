// CFL wave-speed reduction (SimulationDriver::compute_max_wave_speed,
// src/solver/simulation_driver.cpp:153-168).
#include "drf_internal.hpp"

namespace drf {
namespace {

__device__ __forceinline__ double wave_max(double a, double b) { return a > b ? a : b; }

// Per element: sqrt(9.81 * max H) + max(max|u|, max|v|) on the derived state
// of U (update_derived, src/physics/primitive_equations.cpp:21-28).  One
// thread per grid line (e, L) of n nodes: in the line layout consecutive
// lines of a plane are consecutive addresses, so a wavefront's loads are
// contiguous.  The n^2 line maxima of an element meet in LDS, where one
// thread per element forms its wave speed; partial[block] = max over the
// block's elements.  max and sqrt are exact, so any grouping gives the
// reference's value.  HBM-bound (32 B per node): the order is a template
// argument so that a thread's 4 n loads are in flight together, and the next
// batch's are issued before this one's maxima meet (32,768 elements, N = 4,
// from HBM: 40.3 us with a loop over the nodes, now 31.6 us).
template <int n> struct WaveLine {
    double hu[n], hv[n], et[n], h[n];
    __device__ __forceinline__ void load(const View<const double> &U, const View<const double> &hb,
                                         int64_t e, int L)
    {
        // the line's offsets, once per line (the element part of the blocked
        // layout takes a division)
        const int64_t uo = node_offset(U, e, L, 0), ho = node_offset(hb, e, L, 0);
#pragma unroll
        for (int i = 0; i < n; ++i) {
            const int64_t o = uo + (int64_t)i * U.is;
            hu[i] = U.p[o];
            hv[i] = U.p[1 * U.fs + o];
            et[i] = U.p[2 * U.fs + o];
            h[i] = hb.p[ho + (int64_t)i * hb.is];
        }
    }
};

template <int n>
__global__ void __launch_bounds__(256)
    wave_speed_kernel(int64_t E, View<const double> U, View<const double> h, double *partial)
{
    __shared__ double lm[2][3][256]; // by batch parity: one barrier per batch
    __shared__ double red[4];
    constexpr int nl = n * n, epb = 256 / nl;
    const int t = threadIdx.x;
    const int le = t / nl, L = t - le * nl;
    double cmax = 0.0;
    const int64_t nbatch = (E + epb - 1) / epb;
    auto on = [&](int64_t b) { return b < nbatch && le < epb && b * epb + le < E; };
    WaveLine<n> w;
    int64_t b = blockIdx.x;
    if (on(b))
        w.load(U, h, b * epb + le, L);
    for (int par = 0; b < nbatch; b += gridDim.x, par ^= 1) {
        if (on(b)) {
            double hm = -INFINITY, um = 0.0, vm = 0.0;
#pragma unroll
            for (int i = 0; i < n; ++i) {
                const double H = w.et[i] + w.h[i];
                const double hi = (H > 1e-10) ? 1.0 / H : 0.0;
                hm = wave_max(hm, H);
                um = wave_max(um, fabs(w.hu[i] * hi));
                vm = wave_max(vm, fabs(w.hv[i] * hi));
            }
            lm[par][0][t] = hm;
            lm[par][1][t] = um;
            lm[par][2][t] = vm;
        }
        if (on(b + gridDim.x))
            w.load(U, h, (b + gridDim.x) * epb + le, L);
        __syncthreads();
        if (t < epb && b * epb + t < E) {
            double hm = -INFINITY, um = 0.0, vm = 0.0;
            for (int q = t * nl; q < (t + 1) * nl; ++q) {
                hm = wave_max(hm, lm[par][0][q]);
                um = wave_max(um, lm[par][1][q]);
                vm = wave_max(vm, lm[par][2][q]);
            }
            cmax = wave_max(cmax, sqrt(9.81 * hm) + wave_max(um, vm));
        }
    }
    for (int o = 32; o > 0; o >>= 1)
        cmax = wave_max(cmax, __shfl_xor(cmax, o));
    if ((t & 63) == 0)
        red[t >> 6] = cmax;
    __syncthreads();
    if (t == 0)
        partial[blockIdx.x] = wave_max(wave_max(red[0], red[1]), wave_max(red[2], red[3]));
}

template <int WAVES>
__global__ void __launch_bounds__(64 * WAVES)
    wave_speed_derived_kernel(int64_t E, int nd, const double *H, const double *u,
                              const double *v, int64_t es, double *partial)
{
    __shared__ double red[WAVES];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    double cmax = 0.0;
    for (int64_t e = (int64_t)blockIdx.x * WAVES + w; e < E; e += (int64_t)gridDim.x * WAVES) {
        double hm = -INFINITY, um = 0.0, vm = 0.0;
        for (int d = lane; d < nd; d += 64) {
            hm = wave_max(hm, H[e * es + d]);
            um = wave_max(um, fabs(u[e * es + d]));
            vm = wave_max(vm, fabs(v[e * es + d]));
        }
        for (int o = 32; o > 0; o >>= 1) {
            hm = wave_max(hm, __shfl_xor(hm, o));
            um = wave_max(um, __shfl_xor(um, o));
            vm = wave_max(vm, __shfl_xor(vm, o));
        }
        cmax = wave_max(cmax, sqrt(9.81 * hm) + wave_max(um, vm));
    }
    if (lane == 0)
        red[w] = cmax;
    __syncthreads();
    if (threadIdx.x == 0) {
        double m = red[0];
        for (int i = 1; i < WAVES; ++i)
            m = wave_max(m, red[i]);
        partial[blockIdx.x] = m;
    }
}

// out[0] = the maximum of the partials, and with dt set,
// AdaptiveTimeController::compute_dt (src/solver/time_stepper.cpp:261-268) of
// it and the driver's time_ += dt_ (simulation_driver.cpp:130) in the same
// launch (N = 2, 741 elements: adaptive Euler step 18.1 -> 14.4 us).
struct AdaptiveDt {
    double dx_min, cfl, dt_min, dt_max;
    double *dt, *t;
};

__global__ void __launch_bounds__(256)
    max_reduce_kernel(const double *__restrict__ p, int64_t np, double *out, AdaptiveDt a)
{
    __shared__ double red[4];
    double m = 0.0;
#pragma unroll 8
    for (int64_t i = threadIdx.x; i < np; i += 256)
        m = wave_max(m, p[i]);
    for (int o = 32; o > 0; o >>= 1)
        m = wave_max(m, __shfl_xor(m, o));
    if ((threadIdx.x & 63) == 0)
        red[threadIdx.x >> 6] = m;
    __syncthreads();
    if (threadIdx.x == 0) {
        const double c = wave_max(wave_max(red[0], red[1]), wave_max(red[2], red[3]));
        out[0] = c;
        if (a.dt) {
            double d = a.dt_max; // stationary: the largest step
            if (!(c < 1e-14)) {
                d = a.cfl * a.dx_min / c;
                d = (d < a.dt_min) ? a.dt_min : ((a.dt_max < d) ? a.dt_max : d);
            }
            *a.dt = d;
            if (a.t)
                *a.t = *a.t + d;
        }
    }
}

} // namespace

hipError_t launch_wave_speed(int order, int64_t E, View<const double> U, View<const double> h,
                             double *partial, int64_t npart, hipStream_t s)
{
    const dim3 g((unsigned)npart), b(256);
    switch (order) {
    case 1: hipLaunchKernelGGL(wave_speed_kernel<2>, g, b, 0, s, E, U, h, partial); break;
    case 2: hipLaunchKernelGGL(wave_speed_kernel<3>, g, b, 0, s, E, U, h, partial); break;
    case 3: hipLaunchKernelGGL(wave_speed_kernel<4>, g, b, 0, s, E, U, h, partial); break;
    case 4: hipLaunchKernelGGL(wave_speed_kernel<5>, g, b, 0, s, E, U, h, partial); break;
    case 5: hipLaunchKernelGGL(wave_speed_kernel<6>, g, b, 0, s, E, U, h, partial); break;
    case 6: hipLaunchKernelGGL(wave_speed_kernel<7>, g, b, 0, s, E, U, h, partial); break;
    case 7: hipLaunchKernelGGL(wave_speed_kernel<8>, g, b, 0, s, E, U, h, partial); break;
    case 8: hipLaunchKernelGGL(wave_speed_kernel<9>, g, b, 0, s, E, U, h, partial); break;
    default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

hipError_t launch_wave_speed_derived(int order, int64_t E, const double *H, const double *u,
                                     const double *v, int64_t es, double *partial,
                                     int64_t npart, hipStream_t s)
{
    const int n = order + 1, nd = n * n * n;
    hipLaunchKernelGGL(wave_speed_derived_kernel<4>, dim3((unsigned)npart), dim3(256), 0, s, E,
                       nd, H, u, v, es, partial);
    return hipGetLastError();
}

hipError_t launch_max_reduce(const double *partial, int64_t npart, double *out, hipStream_t s)
{
    hipLaunchKernelGGL(max_reduce_kernel, dim3(1), dim3(256), 0, s, partial, npart, out,
                       AdaptiveDt{});
    return hipGetLastError();
}

hipError_t launch_adaptive_dt(const double *partial, int64_t npart, double *out, double dx_min,
                              double cfl, double dt_min, double dt_max, double *dt, double *t,
                              hipStream_t s)
{
    hipLaunchKernelGGL(max_reduce_kernel, dim3(1), dim3(256), 0, s, partial, npart, out,
                       AdaptiveDt{dx_min, cfl, dt_min, dt_max, dt, t});
    return hipGetLastError();
}

} // namespace drf
