// uwshcu_chunks.hip -- gather many physics chunks into one column range and scatter
// the results back, so that a timestep's chunks run as one launch of the column
// pipeline instead of one launch per chunk (the reference calls the scheme once per
// chunk, physpkg.F90:782-803 -> convect_shallow.F90:605-619).
//
// Each field is a [rows][pcols] array per chunk (Fortran (pcols, rows) layout) and a
// [rows][n] array in the packed range, n = sum of the chunks' ncol.  Thread (g, f) of the
// launch owns column g of field f: it finds the chunk (binary search in the column offsets)
// and copies its rows, eight in flight at a time, so consecutive threads touch
// consecutive addresses of both sides.  Only the first ncol columns of a chunk are
// read or written; its padding up to pcols stays untouched.
//
// Bound by memory latency: a timestep's chunks are some 10^4 columns, and one thread per
// column for all fields left most of the chip idle (715 us for the two
// copies of 48 chunks of up to 1000 columns; 180 us with a thread per column and field).
#include <hip/hip_runtime.h>

#include "uwshcu_kernels.h"

namespace uwshcu {

namespace {

__device__ inline int chunk_of(const ChunkTable& t, long long g) {
    int lo = 0, hi = t.nchunk;   // t.off[lo] <= g < t.off[hi]
    while (hi - lo > 1) {
        const int mid = (lo + hi) >> 1;
        if (t.off[mid] <= g) lo = mid;
        else hi = mid;
    }
    return lo;
}

__device__ inline void copy_rows(double* dst, long long dld, const double* src, long long sld, int rows) {
    int r = 0;
    for (; r + 8 <= rows; r += 8) {
        double v[8];
#pragma unroll
        for (int q = 0; q < 8; ++q) v[q] = src[(long long)(r + q) * sld];
#pragma unroll
        for (int q = 0; q < 8; ++q) dst[(long long)(r + q) * dld] = v[q];
    }
    for (; r < rows; ++r) dst[(long long)r * dld] = src[(long long)r * sld];
}

__global__ __launch_bounds__(256) void chunks_gather_kernel(ChunkTable t) {
    const long long stride = (long long)gridDim.x * blockDim.x;
    const int f = blockIdx.y, rows = t.rows[f];
    double* const dst = t.packed[f];
    for (long long g = (long long)blockIdx.x * blockDim.x + threadIdx.x; g < t.n; g += stride) {
        const int c = chunk_of(t, g);
        const double* src = t.ptr[(size_t)f * t.nchunk + c];
        if (src) copy_rows(dst + g, t.n, src + (g - t.off[c]), t.pcols[c], rows);
        else
            for (int r = 0; r < rows; ++r) dst[(long long)r * t.n + g] = 0.0;
    }
}

__global__ __launch_bounds__(256) void chunks_scatter_kernel(ChunkTable t) {
    const long long stride = (long long)gridDim.x * blockDim.x;
    const int f = blockIdx.y, rows = t.rows[f];
    const double* const src = t.packed[f];
    for (long long g = (long long)blockIdx.x * blockDim.x + threadIdx.x; g < t.n; g += stride) {
        const int c = chunk_of(t, g);
        double* dst = t.ptr[(size_t)f * t.nchunk + c];
        if (dst) copy_rows(dst + (g - t.off[c]), t.pcols[c], src + g, t.n, rows);
    }
}

unsigned grid_for(long long n) {
    const long long b = (n + 255) / 256;
    return (unsigned)(b < 8192 ? (b > 0 ? b : 1) : 8192);
}

}  // namespace

hipError_t launch_chunks_gather(const ChunkTable& t, hipStream_t stream) {
    hipLaunchKernelGGL(chunks_gather_kernel, dim3(grid_for(t.n), (unsigned)t.nfield), dim3(256), 0, stream, t);
    return hipGetLastError();
}

hipError_t launch_chunks_scatter(const ChunkTable& t, hipStream_t stream) {
    hipLaunchKernelGGL(chunks_scatter_kernel, dim3(grid_for(t.n), (unsigned)t.nfield), dim3(256), 0, stream, t);
    return hipGetLastError();
}

}  // namespace uwshcu
