// A Q16.16 matrix as digit planes for the matrix cores (Q16Planes).
#include <mutex>

#include "q8_gemm_common.h"

namespace {

__global__ __launch_bounds__(256) void q16_digits_kernel(const int32_t* w, size_t n, int* need) {
    int most = 1;
    for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (size_t)gridDim.x * 256)
        most = max(most, limbs_needed(digits5(w[i])));
    for (int off = 32; off >= 1; off >>= 1) most = max(most, __shfl_xor(most, off));
    if (threadIdx.x % 64 == 0) atomicMax(need, most);
}

// One thread per (row, 32-wide block); the first block's thread also leaves
// the row's shift.
__global__ __launch_bounds__(256) void q16_planes_kernel(const int32_t* w, uint32_t rows, uint32_t nb, size_t plane_bytes,
                                                         int8_t* planes, int32_t* shift) {
    const size_t idx = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (idx >= (size_t)rows * nb) return;
    const uint32_t row = (uint32_t)(idx / nb), b = (uint32_t)(idx % nb);
    if (b == 0) shift[row] = 8;
    const int4* src = (const int4*)(w + (size_t)row * nb * 32 + b * 32);
    int8_t* dst = planes + ((size_t)(row / Q8_TILE_ROWS) * nb + b) * Q8_TILE_BLOCK_BYTES + row % Q8_TILE_ROWS * 16;
    for (int h = 0; h < 2; h++) {
        uint32_t out[2][4];
#pragma unroll
        for (int c = 0; c < 4; c++) {
            const int4 v = src[4 * h + c];
            const uint64_t d0 = digits5(v.x), d1 = digits5(v.y), d2 = digits5(v.z), d3 = digits5(v.w);
#pragma unroll
            for (int l = 0; l < 2; l++) out[l][c] = plane_byte4(d0, d1, d2, d3, l);
        }
#pragma unroll
        for (int l = 0; l < 2; l++)
            *(uint4*)(dst + l * plane_bytes + h * 256) = make_uint4(out[l][0], out[l][1], out[l][2], out[l][3]);
    }
}

}  // namespace

int iris_q16_prepare(const int32_t* w, uint32_t rows, uint32_t cols, Q16Planes* p, hipStream_t stream) {
    static std::mutex lock;  // a matrix is prepared once, whichever thread gets there first
    std::lock_guard<std::mutex> guard(lock);
    if (!w || p->tried) return 0;
    p->tried = true;
    if (!rows || !cols || cols % 64 || cols > 16384) return 0;
    const uint32_t nb = cols / 32, tiles = (rows + Q8_TILE_ROWS - 1) / Q8_TILE_ROWS;
    const size_t plane_bytes = (size_t)tiles * nb * Q8_TILE_BLOCK_BYTES, blocks = (size_t)rows * nb;
    int* d_need = nullptr;
    int need = 0;
    hipError_t st = hipMalloc((void**)&d_need, sizeof(int));
    if (st == hipSuccess) st = hipMemsetAsync(d_need, 0, sizeof(int), stream);
    if (st == hipSuccess) {
        hipLaunchKernelGGL(q16_digits_kernel, dim3((unsigned)((blocks * 32 + 4095) / 4096)), dim3(256), 0, stream, w,
                           blocks * 32, d_need);
        st = hipGetLastError();
    }
    if (st == hipSuccess) st = hipMemcpyAsync(&need, d_need, sizeof(int), hipMemcpyDeviceToHost, stream);
    if (st == hipSuccess) st = hipStreamSynchronize(stream);
    (void)hipFree(d_need);
    if (st != hipSuccess || need > 2) return (int)st;
    int8_t* planes = nullptr;
    int32_t* shift = nullptr;
    // Rows past the matrix in its last tile keep zero digits.
    st = hipMalloc((void**)&planes, 2 * plane_bytes);
    if (st == hipSuccess) st = hipMalloc((void**)&shift, (size_t)tiles * Q8_TILE_ROWS * sizeof(int32_t));
    if (st != hipSuccess) {  // no room for the planes: the per-row kernel serves
        (void)hipGetLastError();
        (void)hipFree(planes);
        return 0;
    }
    st = hipMemsetAsync(planes, 0, 2 * plane_bytes, stream);
    if (st == hipSuccess) st = hipMemsetAsync(shift, 0, (size_t)tiles * Q8_TILE_ROWS * sizeof(int32_t), stream);
    if (st == hipSuccess) {
        hipLaunchKernelGGL(q16_planes_kernel, dim3((unsigned)((blocks + 255) / 256)), dim3(256), 0, stream, w, rows, nb,
                           plane_bytes, planes, shift);
        st = hipGetLastError();
    }
    if (st == hipSuccess) st = hipStreamSynchronize(stream);
    if (st != hipSuccess) {
        (void)hipFree(planes);
        (void)hipFree(shift);
        return (int)st;
    }
    p->planes = planes;
    p->shift = shift;
    p->device_bytes = 2 * plane_bytes + (uint64_t)tiles * Q8_TILE_ROWS * sizeof(int32_t);
    return 0;
}

void iris_q16_free(Q16Planes* p) {
    (void)hipFree(p->planes);
    (void)hipFree(p->shift);
    *p = Q16Planes{};
}
