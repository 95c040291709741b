// Carried keys in and out of a layer's K cache, whose layout is transposed
// ([kv_rows][k_pos_stride]): position rows on the host's side of the copy.
//
// The copies' bound is the host link; what they cost before was the strided
// copy of kv_rows short runs and a transpose on the host (a 45-row layer
// stage with its keys read back 8.4 -> 0.69 ms, a 512-row one 11.8 -> 1.83
// ms, the layer itself included). Here a 32 x 32 tile per
// workgroup goes through LDS, so both sides of the transpose are read and
// written as whole lines, and one contiguous copy follows (or precedes) it.
#include "layer_kernels.h"

namespace {

constexpr uint32_t KT = 32;

// rows[p][c] = cache[c][pos0 + p] (OUT), or the other way round.
template <bool OUT>
__global__ __launch_bounds__(256) void kv_rows_kernel(int32_t* cache, uint32_t stride, uint32_t pos0, uint32_t count,
                                                      uint32_t kvw, int32_t* rows) {
    __shared__ int32_t tile[KT][KT + 1];
    const uint32_t p0 = blockIdx.x * KT, c0 = blockIdx.y * KT, x = threadIdx.x % KT;
    for (uint32_t y = threadIdx.x / KT; y < KT; y += 256 / KT) {
        if (OUT && c0 + y < kvw && p0 + x < count) tile[y][x] = cache[(size_t)(c0 + y) * stride + pos0 + p0 + x];
        if (!OUT && p0 + y < count && c0 + x < kvw) tile[y][x] = rows[(size_t)(p0 + y) * kvw + c0 + x];
    }
    __syncthreads();
    for (uint32_t y = threadIdx.x / KT; y < KT; y += 256 / KT) {
        if (OUT && p0 + y < count && c0 + x < kvw) rows[(size_t)(p0 + y) * kvw + c0 + x] = tile[x][y];
        if (!OUT && c0 + y < kvw && p0 + x < count) cache[(size_t)(c0 + y) * stride + pos0 + p0 + x] = tile[x][y];
    }
}

}  // namespace

int iris_kv_rows_launch(bool out, int32_t* cache, uint32_t stride, uint32_t pos0, uint32_t count, uint32_t kvw,
                        int32_t* rows, hipStream_t stream) {
    if (count == 0 || kvw == 0) return 0;
    const dim3 grid((count + KT - 1) / KT, (kvw + KT - 1) / KT);
    if (out) hipLaunchKernelGGL(kv_rows_kernel<true>, grid, dim3(256), 0, stream, cache, stride, pos0, count, kvw, rows);
    else hipLaunchKernelGGL(kv_rows_kernel<false>, grid, dim3(256), 0, stream, cache, stride, pos0, count, kvw, rows);
    return (int)hipGetLastError();
}
