// The FP64 LU and substitutions of the workgroup kernels by themselves, for
// tests/test_gpu_wg_lu_check.py: lu_check factors and solves one matrix a workgroup.
// Built once for each number of row slots (ODEMI_N = 64, 128, 135: as large as a
// CU's LDS holds); launched with 256 or 512 threads.
#include <hip/hip_runtime.h>
#define ODEMI_NP 1
#define ODEMI_WITH_WG 1
#define ODEMI_RODAS_MIN_WAVES 1
#define ODEMI_MIN_WAVES 1
// the workgroup engine's problem functions, which nothing here calls
template <typename T>
__device__ void odemi_f(T*, const T*, const T*, T) {}
template <typename T>
__device__ void odemi_jac(T*, const T*, const T*, T) {}
template <typename T>
__device__ void odemi_tgrad(T*, const T*, const T*, T) {}
template <typename T>
__device__ void odemi_f_wg(T*, const T*, const T*, T, int, int, int) {}
template <typename T>
__device__ void odemi_jac_wg(T*, int, const T*, const T*, T, int, int, int) {}
template <typename T>
__device__ void odemi_tgrad_wg(T*, const T*, const T*, T, int, int, int) {}
template <typename T>
__device__ void odemi_jvp_wg(T*, const T*, const T*, const T*, T, int, int, int) {}
#include "odemi_device.h"

// A [grid][n][n], b [grid][n] -> LU [grid][n][n] (rows at their positions), the row
// gather perm [grid][n], x and xneg [grid][n] = +-A^{-1} b.  LDS: W [n][ld], the
// right-hand side [n], 16 ints (16-byte aligned), perm [n].  Elements of W past
// column n start as NaN: no result may depend on them.
extern "C" __global__ void __launch_bounds__(512)
lu_check(const double* A, const double* b, int n, int ld, double* LU, int* perm_out, double* x, double* xneg) {
    extern __shared__ __attribute__((aligned(16))) double lu_lds[];
    double* W = lu_lds;
    double* v = W + n * ld;
    int* tab = (int*)(((size_t)(v + n) + 15) & ~(size_t)15);
    int* perm = tab + 16;
    const int tid = threadIdx.x, NT = blockDim.x;
    const size_t m = blockIdx.x;
    for (int e = tid; e < n * ld; e += NT) {
        const int i = e / ld, j = e % ld;
        W[e] = j < n ? A[(m * n + i) * n + j] : __builtin_nan("");
    }
    if (tid < 16) tab[tid] = 0;
    for (int i = tid; i < n; i += NT) v[i] = b[m * n + i];
    __syncthreads();
    odemi::wg_lu_blocked<ODEMI_WG_ROWS>(W, ld, n, tab, perm);
    odemi::wg_lu_solve<double, false>(W, ld, n, perm, v);
    for (int i = tid; i < n; i += NT) {
        x[m * n + i] = v[i];
        v[i] = b[m * n + i];
        perm_out[m * n + i] = perm[i];
    }
    __syncthreads();
    odemi::wg_lu_solve<double, true>(W, ld, n, perm, v);
    for (int i = tid; i < n; i += NT) xneg[m * n + i] = v[i];
    for (int e = tid; e < n * n; e += NT) LU[m * n * n + e] = W[(e / n) * ld + e % n];
}
