// One matrix-core instruction on operands of the caller's choice, for the test of what the first layer's error bound assumes
// of it: D[i] = C[i] + A[i] B[i]^T, one wave per product.  A, B: [n][32][K], C, D: [n][32][32], row-major; the caller
// allocates exactly that.
#include <hip/hip_runtime.h>

typedef _Float16 h8 __attribute__((ext_vector_type(8)));
typedef float v16f __attribute__((ext_vector_type(16)));

// accumulator register i of lane (column j, half h): row 8 (i / 4) + 4 h + i % 4
__device__ int place(int i, int lane) { return (8 * (i / 4) + 4 * (lane >> 5) + i % 4) * 32 + (lane & 31); }

__global__ __launch_bounds__(64) void f16_kernel(const _Float16* a, const _Float16* b, const float* c, float* d) {
    const int lane = threadIdx.x, at = (blockIdx.x * 32 + (lane & 31)) * 16 + 8 * (lane >> 5);
    h8 av, bv;
    v16f acc;
    for (int i = 0; i < 8; ++i) av[i] = a[at + i], bv[i] = b[at + i];
    for (int i = 0; i < 16; ++i) acc[i] = c[blockIdx.x * 1024 + place(i, lane)];
    acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(av, bv, acc, 0, 0, 0);
    for (int i = 0; i < 16; ++i) d[blockIdx.x * 1024 + place(i, lane)] = acc[i];
}

__global__ __launch_bounds__(64) void f32_kernel(const float* a, const float* b, const float* c, float* d) {
    const int lane = threadIdx.x, at = (blockIdx.x * 32 + (lane & 31)) * 2 + (lane >> 5);
    v16f acc;
    for (int i = 0; i < 16; ++i) acc[i] = c[blockIdx.x * 1024 + place(i, lane)];
    acc = __builtin_amdgcn_mfma_f32_32x32x2f32(a[at], b[at], acc, 0, 0, 0);
    for (int i = 0; i < 16; ++i) d[blockIdx.x * 1024 + place(i, lane)] = acc[i];
}

extern "C" int matrix_core_f16(const void* a, const void* b, const float* c, float* d, int n) {
    hipLaunchKernelGGL(f16_kernel, dim3(n), dim3(64), 0, nullptr, (const _Float16*)a, (const _Float16*)b, c, d);
    return (int)hipDeviceSynchronize();
}
extern "C" int matrix_core_f32(const float* a, const float* b, const float* c, float* d, int n) {
    hipLaunchKernelGGL(f32_kernel, dim3(n), dim3(64), 0, nullptr, a, b, c, d);
    return (int)hipDeviceSynchronize();
}
