// check_forms.hip -- the short forms that the sweeps use for ordinary cells
// (NormalRange of exact_math.hpp, augrie_normal.hpp) one edge or one operation
// at a time, for the tests: swe_hip_solve_edges runs the general form, and inside
// a sweep a wave chooses between the two.  Host arrays in and out; a library of
// its own (libswe_hip_check.so), which nothing but the tests loads.
#include <hip/hip_runtime.h>

#include <cstdint>

#include "edge_solver.hpp"

namespace {

using swe::dev::EdgeOut;
using A = swe::dev::NormalRange;

template <int S>
__global__ void edges_kernel(int64_t n, const float* in, float* out) {
    const int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= n) return;
    const EdgeOut e = swe::dev::solve_raw<S, A>(in[k], in[n + k], in[2 * n + k], in[3 * n + k], in[4 * n + k],
                                                in[5 * n + k]);
    out[k] = e.hL;
    out[n + k] = e.hR;
    out[2 * n + k] = e.huL;
    out[3 * n + k] = e.huR;
    out[4 * n + k] = e.speed;
}

__global__ void arith_kernel(int op, int64_t n, const float* in, float* out) {
    const int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= n) return;
    const float a = in[k], b = in[n + k];
    out[k] = op == 0 ? A::rcp(b) : op == 1 ? A::div(a, b) : op == 2 ? A::sqrt(a) : A::sqrt0(a);
}

// `ins` arrays of n numbers in and `outs` out, one after the other
template <class Launch>
int on_device(int64_t n, int ins, int outs, const float* in, float* out, Launch launch) {
    if (n < 1 || n > (int64_t(1) << 28) || !in || !out) return -1;
    float *din = nullptr, *dout = nullptr;
    hipError_t e = hipMalloc(&din, sizeof(float) * n * ins);
    if (e == hipSuccess) e = hipMalloc(&dout, sizeof(float) * n * outs);
    if (e == hipSuccess) e = hipMemcpy(din, in, sizeof(float) * n * ins, hipMemcpyHostToDevice);
    if (e == hipSuccess) {
        launch(dim3((unsigned)((n + 255) / 256)), dim3(256), din, dout);
        e = hipGetLastError();
    }
    if (e == hipSuccess) e = hipMemcpy(out, dout, sizeof(float) * n * outs, hipMemcpyDeviceToHost);
    (void)hipFree(din);
    (void)hipFree(dout);
    return e == hipSuccess ? 0 : -3;
}

template <int S>
int edges(int64_t n, const float* in, float* out) {
    return on_device(n, 6, 5, in, out, [&](dim3 grid, dim3 block, const float* din, float* dout) {
        hipLaunchKernelGGL(edges_kernel<S>, grid, block, 0, nullptr, n, din, dout);
    });
}

}  // namespace

extern "C" {

// Edges of cells in in_normal_range: in = hL, hR, huL, huR, bL, bR, out = hNetL,
// hNetR, huNetL, huNetR, speed, n of each.
int swe_check_edges(int solver, int64_t n, const float* in, float* out) {
    switch (solver) {
        case swe::SOLVER_HLLE: return edges<swe::SOLVER_HLLE>(n, in, out);
        case swe::SOLVER_FWAVE: return edges<swe::SOLVER_FWAVE>(n, in, out);
        case swe::SOLVER_AUGRIE: return edges<swe::SOLVER_AUGRIE>(n, in, out);
        case swe::SOLVER_HYBRID: return edges<swe::SOLVER_HYBRID>(n, in, out);
        default: return -1;
    }
}

// op 0: 1 / b, 1: a / b, 2: sqrt(a), 3: sqrt(a) with zero allowed; in = a, b.
int swe_check_arith(int op, int64_t n, const float* in, float* out) {
    if (op < 0 || op > 3) return -1;
    return on_device(n, 2, 1, in, out, [&](dim3 grid, dim3 block, const float* din, float* dout) {
        hipLaunchKernelGGL(arith_kernel, grid, block, 0, nullptr, op, n, din, dout);
    });
}

}  // extern "C"
