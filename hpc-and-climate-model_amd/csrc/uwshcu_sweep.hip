// uwshcu_sweep.hip -- the adjoint's backward sweep: each column's tape (recorded by
// uwshcu_adjoint.hip) is swept backwards from the outputs' cotangents to the gradients
// of t0, qv0, u0, v0, tke, pblh and (rpen, rle, rkm).  A translation unit of its own,
// apart from the recording kernel's large one.
// Compiled with -ffp-contract=off: products and sums round as the host build's do.
#include "uwshcu_adjoint.h"
#include "uwshcu_kernels.h"

namespace uwshcu {

// Backward sweep of L columns by one wavefront: lane t < L takes the steps of its own
// column (the steps of ad_reverse, in its order), and all 64 lanes share the loads.
//
// What bounds it: memory latency.  A launch has one wavefront per SIMD at most, and with
// its adjoints read when they enter the window, a wavefront waited for them, and for the
// additions issued before them, once per batch of 16 nodes: 11 of 30 ms at 65536 columns x
// 35 levels x 3 constituents (its tape loads 6, its additions 3 ms).  So:
//  - the lanes share the loads: consecutive lanes load consecutive 16 bytes of one column's
//    nodes (a batch is 384 contiguous bytes, its entering adjoints one 128-byte line), 24 + 8
//    loads of about 9 cache lines each instead of 48 of 64, and the data reach their
//    column's lane through LDS, four nodes (96 bytes, at a stride of 112 that spreads the
//    16-byte reads over the banks) at a time;
//  - a batch's entering line is read at its start and the batch's additions to it are made
//    in the window; the next batch's nodes are loaded before a batch's steps and their
//    page-table entry a batch earlier still;
//  - a step reads one window entry and adds to two without waiting (LDS FP64 adds).
// 28.5 to 22.5 ms there; at 4097 x 72 x 10, where L = 8 gives 513 wavefronts instead of 65,
// 57.6 to 36.4 ms.
//
// LDS: a window of 64 recent adjoints and its spare entry (520 B per column) and the four
// nodes, 40 448 B at L = 64: four workgroups a CU, one wavefront per SIMD.
// Columns whose recording did not complete are skipped.
constexpr int kSweepWindow = 64;
constexpr int kSubNodes = 4;                        // nodes of a batch that are in LDS at a time
constexpr int kSubBatches = kSweepBatch / kSubNodes;
constexpr int kSubChunks = kSubNodes * (int)sizeof(TapeNode) / 16;      // 16-byte pieces of them
static_assert(sizeof(TapeNode) == 24 && kSubChunks == 6, "four nodes are six 16-byte pieces");
static_assert(kSweepBatch * sizeof(double) == 128, "a batch's adjoints are one cache line");

typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
typedef double f64x2 __attribute__((ext_vector_type(2)));

__device__ inline const UWSHCU_GMEM char* shfl_ptr(const UWSHCU_GMEM char* p, int lane) {
    const unsigned long long v = (unsigned long long)p;
    const unsigned lo = __shfl((unsigned)v, lane), hi = __shfl((unsigned)(v >> 32), lane);
    return (const UWSHCU_GMEM char*)(((unsigned long long)hi << 32) | lo);
}
// LDS written by some lanes of the wavefront, read by others: LDS operations of one
// wavefront complete in order, so only the compiler must keep theirs.
__device__ inline void wave_lds_fence() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// An FP64 add in LDS, no value returned: the wavefront does not wait for it, and it takes
// its turn among the wavefront's LDS operations.
__device__ inline void lds_add(double& x, double c) {
    __hip_atomic_fetch_add(&x, c, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}

template <int L>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(1)))
void adjoint_sweep_kernel(int n, int col0, int mkx, int ncnst, long long wld, long long ldc, const TapeCtx* tapes,
                          const int* node_out, double* adj, AdCotangents cot, AdGradients g) {
    constexpr int S = kSweepWindow, K = kSweepBatch;
    constexpr int NT = (L * kSubChunks + 63) / 64;      // tape loads of a lane per sub-batch
    constexpr int NE = (L * 8 + 63) / 64;               // loads of entering adjoints (16 bytes) per batch
    __shared__ double s_win[S + 1][L];
    __shared__ u32x4 s_nodes[L][kSubChunks + 1];
    const int lane = threadIdx.x;
    const int j = blockIdx.x * L + lane;
    bool own = lane < L && j < n;
    TapeCtx th{};
    if (own) {
        th = tapes[j];
        own = th.overflow == 0;
    }
    const int nin = ad_inputs(mkx);
    const int nn = own ? th.hot.n : 0;
    UWSHCU_GMEM double* const adjv = (UWSHCU_GMEM double*)adj + th.adj;
    auto win = [&](int s) -> double& { return s_win[s][lane & (L - 1)]; };
    auto wslot = [](int x) { return x & (S - 1); };
    int q0 = (nn - 1) | (K - 1);
    if (own) {
        ad_seed(adjv, node_out, (size_t)wld, j, mkx, ncnst, (size_t)ldc, col0 + j, cot);
        for (int q = nn - 1; q >= 0 && q > q0 - S; --q) win(wslot(q)) = adj_load(adjv + q);
        win(S) = 0.0;
    }
    bool run = own && nn > nin;
    const UWSHCU_GMEM int* const pages = (const UWSHCU_GMEM int*)th.pages;
    const UWSHCU_GMEM char* const pool =
        own ? (const UWSHCU_GMEM char*)((const UWSHCU_GMEM TapePool*)th.pool)->base : nullptr;
    auto page_of = [&](int q) { return pages[(q > 0 ? q : 0) >> kTapePageLog2]; };
    // the nodes of the batch at q (reversed within the page: node q first)
    auto batch_at = [&](int q, int pg) {
        return pool + ((size_t)pg * kTapePage + (kTapePage - 1 - (q & (kTapePage - 1)))) * sizeof(TapeNode);
    };
    // lane's pieces: piece i*64 + lane of the columns' pieces, column-major
    auto tcol = [&](int i) { return (i * 64 + lane) / kSubChunks; };
    auto tpart = [&](int i) { return (i * 64 + lane) % kSubChunks; };
    u32x4 nx[kSubBatches][NT];
    auto load_batch = [&](const UWSHCU_GMEM char* mine) {
#pragma unroll
        for (int i = 0; i < NT; ++i) {
            const UWSHCU_GMEM char* src = shfl_ptr(mine, tcol(i) & (L - 1));
            if (tcol(i) < L && src) {
#pragma unroll
                for (int s = 0; s < kSubBatches; ++s)
                    nx[s][i] = *(const UWSHCU_GMEM u32x4*)(src + s * kSubChunks * 16 + tpart(i) * 16);
            }
        }
    };
    load_batch(run ? batch_at(q0, page_of(nn - 1)) : nullptr);
    int pg_next = run ? page_of(q0 - K) : 0;     // page of the next batch, read a batch ahead
    double ahead = 0.0;
    while (__any(run)) {
        u32x4 cur[kSubBatches][NT];
#pragma unroll
        for (int s = 0; s < kSubBatches; ++s)
#pragma unroll
            for (int i = 0; i < NT; ++i) cur[s][i] = nx[s][i];
        const bool more = run && q0 - K >= nin;
        load_batch(more ? batch_at(q0 - K, pg_next) : nullptr);
        if (more) pg_next = page_of(q0 - 2 * K);
        const int lo = q0 - S, lo1 = lo > -1 ? lo : -1;
        // Nodes lo - 15 .. lo enter the window at the batch's end: one line of the column's
        // adjoints (each column's start on a line, so it holds no other's and is read this
        // once, after every earlier batch's additions).  It is read now, so that its latency
        // hides behind the steps; this batch's additions to it are made in the window.
        const UWSHCU_GMEM char* line = run && lo >= 0 ? (const UWSHCU_GMEM char*)(adjv + (lo - (K - 1))) : nullptr;
        f64x2 enter[NE];
        int enter_at[NE];      // its first node, or below what may enter
#pragma unroll
        for (int i = 0; i < NE; ++i) {
            const int c = (i * 64 + lane) / 8, part = (i * 64 + lane) % 8;
            const UWSHCU_GMEM char* src = shfl_ptr(line, c & (L - 1));
            enter_at[i] = __shfl(lo, c & (L - 1)) - (K - 1) + 2 * part;
            if (c < L && src) enter[i] = *(const UWSHCU_GMEM f64x2*)(src + part * 16);
            else enter_at[i] = -S - K;
        }
        // ... and the line that enters two batches from now comes into the L2 (its value is
        // not used: it may still receive additions).
        asm volatile("" ::"v"(ahead));
        ahead = run && lo - 2 * K >= 0 ? adj_load(adjv + (lo - 2 * K)) : 0.0;
        const bool full = __all(!run || (q0 - (K - 1) >= nin && q0 < nn));
        int fx[2 * K];         // the batch's contributions to nodes outside the window: node (or -1), value
        double fc[2 * K];
#pragma unroll
        for (int s = 0; s < kSubBatches; ++s) {
            wave_lds_fence();
#pragma unroll
            for (int i = 0; i < NT; ++i)
                if (tcol(i) < L) s_nodes[tcol(i)][tpart(i)] = cur[s][i];
            wave_lds_fence();
            if (run) {
                u32x4 v[kSubChunks];
#pragma unroll
                for (int i = 0; i < kSubChunks; ++i) v[i] = s_nodes[lane & (L - 1)][i];
                auto word = [&](int w) { return v[w >> 2][w & 3]; };
                auto steps = [&](auto all) {
                    constexpr bool kAll = decltype(all)::value;
#pragma unroll
                    for (int x = 0; x < kSubNodes; ++x) {
                        const int u = s * kSubNodes + x, q = q0 - u;
                        const bool act = kAll || (q >= nin && q < nn);
                        const double da = __hiloint2double((int)word(6 * x + 1), (int)word(6 * x));
                        const double db = __hiloint2double((int)word(6 * x + 3), (int)word(6 * x + 2));
                        const int a = (int)word(6 * x + 4), b = (int)word(6 * x + 5);
                        const double w = win(act ? wslot(q) : S);
                        const bool live = act && w != 0.0;
                        const double ca = w * da, cb = w * db;
                        const bool inA = a > lo1, inB = b > lo1;
                        lds_add(win(live && inA ? wslot(a) : S), ca);
                        lds_add(win(live && inB ? wslot(b) : S), cb);
                        fx[2 * u] = live && !inA ? a : -1;
                        fx[2 * u + 1] = live && !inB ? b : -1;
                        fc[2 * u] = ca;
                        fc[2 * u + 1] = cb;
                    }
                };
                if (full) steps(std::true_type{});
                else steps(std::false_type{});
            }
        }
        // the entries of the batch's nodes pass to the entering ones (node x takes that of
        // x + S, which stays while that is an input), then the batch's additions outside
        // the window, in step order
        const int in1 = lo - K > nin - S - 1 ? lo - K : nin - S - 1;   // a node above in1 has entered
        wave_lds_fence();
#pragma unroll
        for (int i = 0; i < NE; ++i) {
            const int c = ((i * 64 + lane) / 8) & (L - 1), x = enter_at[i];
            if (x + S >= nin) s_win[x & (S - 1)][c] = enter[i].x;
            if (x + 1 + S >= nin) s_win[(x + 1) & (S - 1)][c] = enter[i].y;
        }
        wave_lds_fence();
        if (run) {
#pragma unroll
            for (int v = 0; v < 2 * K; ++v)
                if (fx[v] >= 0) {
                    if (fx[v] > in1) lds_add(win(wslot(fx[v])), fc[v]);
                    else adj_add(adjv + fx[v], fc[v]);
                }
        }
        q0 -= K;
        run = more;
    }
    if (own) {
        // the inputs' adjoints: the window holds nodes nin - S .. nin - 1, adjv the rest
        auto A = [&](int q) { return q >= nin - S ? win(wslot(q)) : adj_load(adjv + q); };
        ad_write_gradients(A, mkx, (size_t)ldc, col0 + j, g);
    }
}

// Zero n doubles (the sweep's adjoints; a kernel, not a memset, so that a captured
// graph records no memset node).
__global__ __launch_bounds__(256) void zero_kernel(double* p, long long n) {
    for (long long i = blockIdx.x * 256ll + threadIdx.x; i < n; i += (long long)gridDim.x * 256) p[i] = 0.0;
}

hipError_t launch_adjoint_sweep(const FwdArgs& args, int n, double* adj, long long nadj, const int* node_out,
                                const AdCotangents& cot, const AdGradients& g, hipStream_t stream) {
    if (nadj > 0) {
        long long blocks = (nadj + 255) / 256;
        if (blocks > 8192) blocks = 8192;
        hipLaunchKernelGGL(zero_kernel, dim3((unsigned)blocks), dim3(256), 0, stream, adj, nadj);
    }
    auto sweep = [&](auto kernel, int lanes) {
        hipLaunchKernelGGL(kernel, dim3((n + lanes - 1) / lanes), dim3(64), 0, stream, n, args.col0, args.mkx,
                           args.ncnst, args.wld, (long long)args.ldc, (const TapeCtx*)args.ad.tapes, node_out, adj, cot,
                           g);
    };
    switch (adjoint_lanes(n)) {
    case 8: sweep(adjoint_sweep_kernel<8>, 8); break;
    case 16: sweep(adjoint_sweep_kernel<16>, 16); break;
    case 32: sweep(adjoint_sweep_kernel<32>, 32); break;
    default: sweep(adjoint_sweep_kernel<64>, 64);
    }
    return hipGetLastError();
}

}  // namespace uwshcu
