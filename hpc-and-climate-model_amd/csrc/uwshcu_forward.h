// uwshcu_forward.h -- the forward kernel template, instantiated per precision.
#ifndef UWSHCU_FORWARD_H
#define UWSHCU_FORWARD_H

#include "uwshcu_kernels.h"

namespace uwshcu {

// The work items of a launch (slots, or entries of args.list) among n.
__device__ inline int valid_items(const FwdArgs& args, int n) {
    if (args.list) {
        const int left = *args.list_count;
        return left < n ? left : n;
    }
    if (args.colmap) {
        const int left = *args.colcount - args.col0;
        return left < n ? left : n;
    }
    return n;
}
// Work item j's workspace slot and column: slot j serves column col0 + j, or, with a
// column map, column colmap[col0 + j]; item j of a list is the slot it names.
__device__ inline void item_column(const FwdArgs& args, int j, int& slot, int& col) {
    slot = args.list ? args.list[j] : j;
    const int c = (args.list ? args.slot0 : args.col0) + slot;
    col = args.colmap ? args.colmap[c] : c;
}

// One thread per column; the saturation table is staged into LDS once per workgroup.
template <class R, bool ZW, bool SPLIT, bool FAST, int PART = PART_ALL>
__device__ __forceinline__ void forward_body(const FwdArgs& args, int n, const uwshcu_consts* __restrict__ consts,
                                             const double* __restrict__ estbl) {
    __shared__ double s_estbl[UWSHCU_ESTBL_LEN];
    const int nvalid = valid_items(args, n);
    if ((int)(blockIdx.x * blockDim.x) >= nvalid) return;     // whole workgroup idle
    for (int t = threadIdx.x; t < UWSHCU_ESTBL_LEN; t += blockDim.x) s_estbl[t] = estbl[t];
    __syncthreads();
    const int j = blockIdx.x * blockDim.x + threadIdx.x;
    if (j >= nvalid) return;
    int slot, col;
    item_column(args, j, slot, col);
    const ThermoT<double, FAST> T{consts, s_estbl};
    const Column<R, double, ZW, FAST> c(args, T, col, slot);
    c.template run_body<SPLIT, PART>();
}

// The whole column pass in one kernel, with all 512 registers of a lane: for calls
// without list storage (the allocation-free entry point).
template <class R, bool ZW = false, bool FAST = false>
__global__ __launch_bounds__(128) __attribute__((amdgpu_waves_per_eu(1)))
void forward_kernel(FwdArgs args, int n, const uwshcu_consts* __restrict__ consts, const double* __restrict__ estbl) {
    forward_body<R, ZW, false, FAST>(args, n, consts, estbl);
}

// One part (PART_*) of a split launch, with OCC wavefronts per SIMD as its register budget.
template <class R, bool ZW, bool FAST, int PART, int OCC>
__global__ __launch_bounds__(128) __attribute__((amdgpu_waves_per_eu(OCC)))
void forward_kernel_part(FwdArgs args, int n, const uwshcu_consts* __restrict__ consts,
                         const double* __restrict__ estbl) {
    forward_body<R, ZW, true, FAST, PART>(args, n, consts, estbl);
}

// S12-S21 of the listed columns: a workgroup takes 64 of them, wavefront w the levels
// w, w + kRestWaves, ... (uwshcu_rest.h).
constexpr int kRestWaves = 8;
struct TileTeam {
    int rank;
    static constexpr int size = kRestWaves;
    int* s_fail;      // [64] smallest failure of each column
    int* s_borrow;    // [64]
    __device__ void sync() { __syncthreads(); }
    __device__ void fail(int key) { atomicMin(&s_fail[threadIdx.x & 63], key); }
    __device__ int failed() const { return s_fail[threadIdx.x & 63]; }
    __device__ void borrows() { s_borrow[threadIdx.x & 63] = 1; }
    __device__ bool borrowed() const { return s_borrow[threadIdx.x & 63] != 0; }
};
template <class R, bool ZW, bool FAST>
__global__ __launch_bounds__(64 * kRestWaves)
void rest_kernel(FwdArgs args, int n, int final_pass, const uwshcu_consts* __restrict__ consts,
                 const double* __restrict__ estbl) {
    __shared__ double s_estbl[UWSHCU_ESTBL_LEN];
    __shared__ int s_fail[64], s_borrow[64];
    const int nvalid = valid_items(args, n);
    if ((int)blockIdx.x * 64 >= nvalid) return;     // whole workgroup idle
    for (int t = threadIdx.x; t < UWSHCU_ESTBL_LEN; t += blockDim.x) s_estbl[t] = estbl[t];
    if (threadIdx.x < 64) {
        s_fail[threadIdx.x] = 0x7fffffff;
        s_borrow[threadIdx.x] = 0;
    }
    __syncthreads();
    const int j = blockIdx.x * 64 + (threadIdx.x & 63);
    int slot, col;
    item_column(args, j < nvalid ? j : nvalid - 1, slot, col);
    const ThermoT<double, FAST> T{consts, s_estbl};
    const Column<R, double, ZW, FAST> c(args, T, col, slot);
    TileTeam team{(int)threadIdx.x >> 6, s_fail, s_borrow};
    c.rest_team(team, j < nvalid, final_pass != 0);
}

// Level-parallel set-up: thread t of the launch handles workspace slot t % n and
// level t / n (+1 for stages 2-4), so that a wavefront covers consecutive columns.
// Stages 1 and 2: the set-A environment and the wet bulb, before the column pass.
// Stages 3 and 4: a listed column's set-B environment (S22) after the first pass of a
// split launch, in the column's own slot, where it continues.  Stage 1 also clears the
// launch's marks.
template <class R, int STAGE, bool ZW = false, bool FAST = false>
__global__ __launch_bounds__(256) void setup_kernel(FwdArgs args, int n, const uwshcu_consts* __restrict__ consts,
                                                    const double* __restrict__ estbl) {
    __shared__ double s_estbl[UWSHCU_ESTBL_LEN];
    const int nvalid = valid_items(args, n);
    if (STAGE == 1 && args.defer_mark) {   // all n marks, also of slots past a column map's end
        const long long t0 = (long long)blockIdx.x * blockDim.x + threadIdx.x;
        if (t0 < n) args.defer_mark[t0] = 0;
    }
    {   // whole workgroup past the listed columns (in one level row): nothing to do
        const long long t0 = (long long)blockIdx.x * blockDim.x;
        const long long j0 = t0 % n;
        if (j0 >= nvalid && j0 + blockDim.x <= n) return;
    }
    for (int t = threadIdx.x; t < UWSHCU_ESTBL_LEN; t += blockDim.x) s_estbl[t] = estbl[t];
    __syncthreads();
    const long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    const int j = (int)(t % n);
    const int k = (int)(t / n) + (STAGE == 1 ? 0 : 1);
    if (k > args.mkx || j >= nvalid) return;
    int slot, col;
    item_column(args, j, slot, col);
    const ThermoT<double, FAST> T{consts, s_estbl};
    const Column<R, double, ZW, FAST> c(args, T, col, slot);
    if (STAGE >= 3 && c.rstate(RS_CONT) == 0.0) return;   // it ended in its first pass
    if (STAGE == 1) c.setup_level1(k);
    else if (STAGE == 2) c.setup_level2(k);
    else if (STAGE == 3) c.setup_level_b1(k);
    else c.setup_level_b2(k);
}

// Ordered compaction of marks[0, n) into list (slots, ascending) and *count, in three
// steps: per-256 block sums, their exclusive scan (one workgroup), then each block's
// entries at its offset, which also clears the marks.  Keeping the column order keeps the
// listed columns' workspace accesses as coalesced as the marks allow.
static __device__ inline int block_prefix_256(int flag, int* s_wave, int& total) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const unsigned long long m = __ballot(flag);
    const int in_wave = __popcll(m & ((1ull << lane) - 1ull));
    if (lane == 0) s_wave[wave] = __popcll(m);
    __syncthreads();
    int before = 0;
    total = 0;
    for (int w = 0; w < 4; ++w) {
        if (w < wave) before += s_wave[w];
        total += s_wave[w];
    }
    return before + in_wave;
}
static __global__ __launch_bounds__(256) void mark_block_sum_kernel(const int* marks, int n, int* bsum) {
    __shared__ int s_wave[4];
    const int g = blockIdx.x * 256 + threadIdx.x;
    int total;
    block_prefix_256(g < n ? marks[g] : 0, s_wave, total);
    if (threadIdx.x == 0) bsum[blockIdx.x] = total;
}
static __global__ __launch_bounds__(1024) void block_sum_scan_kernel(int* bsum, int nb, int* count) {
    __shared__ int s[1024];
    int carry = 0;
    for (int c0 = 0; c0 < nb; c0 += 1024) {
        const int b = c0 + (int)threadIdx.x;
        const int v = b < nb ? bsum[b] : 0;
        s[threadIdx.x] = v;
        __syncthreads();
        for (int d = 1; d < 1024; d <<= 1) {   // inclusive Hillis-Steele scan
            const int add = (int)threadIdx.x >= d ? s[threadIdx.x - d] : 0;
            __syncthreads();
            s[threadIdx.x] += add;
            __syncthreads();
        }
        if (b < nb) bsum[b] = carry + s[threadIdx.x] - v;   // exclusive
        carry += s[1023];
        __syncthreads();
    }
    if (threadIdx.x == 0) *count = carry;
}
static __global__ __launch_bounds__(256) void mark_scatter_kernel(int* marks, int n, const int* boff, int* list) {
    __shared__ int s_wave[4];
    const int g = blockIdx.x * 256 + threadIdx.x;
    const int flag = g < n ? marks[g] : 0;
    int total;
    const int pos = block_prefix_256(flag, s_wave, total);
    if (flag) {
        list[boff[blockIdx.x] + pos] = g;
        marks[g] = 0;
    }
}

// The forward pass of columns [col0, col0 + n) (or of the mapped columns): the two
// level-parallel set-up stages, then the column pass, split so that wavefronts are not
// held by a few of their lanes and each kernel holds only the live state of its own
// stages (the column code as one kernel needs about 500 registers per lane):
//  1. every column runs the environment, CIN and trigger stages (PART_CLOSURE); a
//     column that reaches the cloud-base closure saves its scalars and marks itself,
//     and the marks are compacted into list 1 in column order;
//  2. the listed (triggered) columns, packed densely, run the rest of the first pass:
//     the buoyancy sorting (PART_SORT), the stages from the forcedCu filter through the
//     in-cloud diagnostics and the set-B environment, both level-parallel (rest_kernel,
//     setup stages 3 and 4), and the implicit-CIN iteration up to its CIN (PART_CIN2),
//     where a column that convects a second time (a few per cent) saves its scalars and
//     marks itself for list 2;
//  3. the columns of list 2 run their second convection pass: PART_SORT and rest_kernel.
// Each column keeps its workspace slot throughout.
//
// args0.defer_list / defer_state (nullable: the column pass then runs as one kernel) give
// the lists' storage: defer_count[0..1]; defer_list[0..defer_list_ints(n)): list 1, list 2,
// the marks and the compaction's block sums; and NRESUME x wld doubles.
template <class R, bool ZW = false, bool FAST = false>
hipError_t launch_column_pipeline(const FwdArgs& args0, int n, const uwshcu_consts* dconsts, const double* destbl,
                                  hipStream_t stream) {
    FwdArgs args = args0;
    args.env_ready = 1;
    args.resume = 0;
    args.defer_list = nullptr;
    args.defer_count = nullptr;
    args.list = nullptr;
    args.list_count = nullptr;
    args.slot0 = args0.col0;
    args.defer_at_closure = 0;
    const bool split = args0.defer_list && args0.defer_count && args0.defer_state;
    int* const list1 = args0.defer_list;
    int* const list2 = split ? list1 + (size_t)n : nullptr;
    int* const marks = split ? list1 + 2 * (size_t)n : nullptr;
    int* const bsum = split ? list1 + 3 * (size_t)n : nullptr;
    int* const count1 = args0.defer_count;
    int* const count2 = split ? count1 + 1 : nullptr;
    args.defer_mark = marks;

    const unsigned lvl0 = (unsigned)(((long long)n * (args.mkx + 1) + 255) / 256);
    const unsigned lvl1 = (unsigned)(((long long)n * args.mkx + 255) / 256);
    const dim3 cols((n + 127) / 128), tiles((n + 63) / 64);
    hipLaunchKernelGGL((setup_kernel<R, 1, ZW, FAST>), dim3(lvl0), dim3(256), 0, stream, args, n, dconsts, destbl);
    hipLaunchKernelGGL((setup_kernel<R, 2, ZW, FAST>), dim3(lvl1), dim3(256), 0, stream, args, n, dconsts, destbl);
    if (!split) {
        hipLaunchKernelGGL((forward_kernel<R, ZW, FAST>), cols, dim3(128), 0, stream, args, n, dconsts, destbl);
        return hipGetLastError();
    }
    const unsigned nblk = (unsigned)((n + 255) / 256);
    auto compact = [&](int* list, int* count) {   // marks -> list in column order
        hipLaunchKernelGGL(mark_block_sum_kernel, dim3(nblk), dim3(256), 0, stream, (const int*)marks, n, bsum);
        hipLaunchKernelGGL(block_sum_scan_kernel, dim3(1), dim3(1024), 0, stream, bsum, (int)nblk, count);
        hipLaunchKernelGGL(mark_scatter_kernel, dim3(nblk), dim3(256), 0, stream, marks, n, (const int*)bsum, list);
    };
    // The buoyancy sorting at two wavefronts per SIMD (256 registers, some spill) where a
    // launch has that many, else at one with all 512.
    const bool large = n >= 2 * 1024 * 64;
    auto sort = [&](const FwdArgs& f, bool two) {
        if (two)
            hipLaunchKernelGGL((forward_kernel_part<R, ZW, FAST, PART_SORT, 2>), cols, dim3(128), 0, stream, f, n,
                               dconsts, destbl);
        else
            hipLaunchKernelGGL((forward_kernel_part<R, ZW, FAST, PART_SORT, 1>), cols, dim3(128), 0, stream, f, n,
                               dconsts, destbl);
    };
    auto rest = [&](const FwdArgs& f, int final_pass) {
        hipLaunchKernelGGL((rest_kernel<R, ZW, FAST>), tiles, dim3(64 * kRestWaves), 0, stream, f, n, final_pass,
                           dconsts, destbl);
    };
    hipLaunchKernelGGL((forward_kernel_part<R, ZW, FAST, PART_CLOSURE, 2>), cols, dim3(128), 0, stream, args, n,
                       dconsts, destbl);
    compact(list1, count1);
    FwdArgs b = args;
    b.defer_mark = nullptr;
    b.list = list1;
    b.list_count = count1;
    b.resume = 1;
    sort(b, large);
    rest(b, 0);
    hipLaunchKernelGGL((setup_kernel<R, 3, ZW, FAST>), dim3(lvl1), dim3(256), 0, stream, b, n, dconsts, destbl);
    hipLaunchKernelGGL((setup_kernel<R, 4, ZW, FAST>), dim3(lvl1), dim3(256), 0, stream, b, n, dconsts, destbl);
    b.resume = 4;
    b.defer_mark = marks;
    hipLaunchKernelGGL((forward_kernel_part<R, ZW, FAST, PART_CIN2, 2>), cols, dim3(128), 0, stream, b, n, dconsts,
                       destbl);
    compact(list2, count2);
    b.list = list2;
    b.list_count = count2;
    b.resume = 2;
    b.defer_mark = nullptr;
    sort(b, false);
    rest(b, 1);
    return hipGetLastError();
}

}  // namespace uwshcu
#endif
