// Graph coloring of the reference's GRAPH_COLOR_GPU (apps/graph-color/src/gpu/
// graph_color_wrapper.cu:598-635, 665-699; kernels graph_color_kernel.cu:14-35, 779-834).
//
// The reference colors in rounds c = 1, 2, ...: an uncolored vertex v takes color c unless one
// of its out-neighbours u with u < v is uncolored or has taken c in the same round
// (graph_color_kernel.cu:26-27).  A smaller neighbour that is uncolored when the round starts
// blocks v whether or not it is colored during the round, and one colored in an earlier round
// never does, so the outcome does not depend on thread timing:
//     color[v] = 1 + max { color[u] : v -> u, u < v }   (1 when there is no such u),
// the length of the longest path of decreasing ids that starts at v.
//
// MI355X mapping (method 0): the recurrence is a triangular solve in the order of the ids, so it
// is solved without rounds.  The vertices are cut, in id order, into tickets of at most COL_EDGES
// edges: runs of consecutive short rows, or one chunk of a long row.  A wavefront takes the next
// ticket, reads its edges once into registers and looks up the colors of the smaller neighbours;
// edges whose neighbour has no color yet are polled, and a vertex whose edges are all settled gets
// its color with one store.  Every dependency has a smaller id (or is an earlier chunk of the same
// row), so it belongs to the same wavefront or to a ticket taken earlier, and the wavefront that
// holds the lowest unfinished ticket never waits for anything unstarted: the solve ends whatever
// the number of resident wavefronts.  No transposed lists, no counters and no atomic per edge
// (atomics run at 27 G/s on the whole chip).  R-MAT s20 (1,048,576 / 16,777,216, about 1,080
// colors): 1.8 ms on the device, 1.7 us per hop of the longest chain, against 35.1 ms with one
// launch per color over a frontier fed by per-edge counters; a 1000 x 1000 grid with 1 % long-range
// edges (47,311 colors): 32 ms against 191.
// Method 1 runs the reference's rounds as they are (every uncolored vertex re-checks its
// smaller neighbours each round, one host readback per round): the baseline.
#include <hip/hip_runtime.h>
#include <cstring>
#include <rocprim/device/device_scan.hpp>
#include "np_internal.h"

namespace np {

__device__ __forceinline__ int col_lane() { return threadIdx.x & 63; }

static int col_grid(long long work, int cap) {
    long long g = (work + 255) / 256;
    return (int)(g < 1 ? 1 : (g > cap ? cap : g));
}

// One workgroup per CU and 256 edges per ticket: every wavefront that waits polls, and polls of a
// color that many others wait for queue behind one another and behind its store.  R-MAT s20, ms:
// 1.82 with 4 edges per lane and 1 workgroup per CU (2: 1.91), with 8 edges 2.21 (2: 2.30, 4: 2.53,
// 8: 13.0); a pause between polls only adds to the hop (8 per CU 4.8, 2 per CU 2.32-2.53).
constexpr int COL_UNR = 4;                 // edges per lane
constexpr int COL_WGS = 1;                 // workgroups per CU
constexpr int COL_EDGES = 64 * COL_UNR;    // edges per ticket at most
constexpr int COL_BLOCK = 64;              // a run lies inside a block of this many vertices
constexpr unsigned long long COL_SPIN_LIMIT = 1ull << 24;

// Tickets of one block of COL_BLOCK vertices, in id order: emit(first vertex, count) for a run of
// rows with at most COL_EDGES edges together, emit(vertex, -1 - chunk) for chunk after chunk of a
// longer row.
template <class F>
__device__ __forceinline__ void col_cut(const int *row, long long v0, long long v1, F emit) {
    long long first = v0;
    int acc = 0, r0 = row[v0];
    for (long long v = v0; v < v1; ++v) {
        const int r1 = row[v + 1], d = r1 - r0;
        r0 = r1;
        if (d > COL_EDGES || acc > COL_EDGES - d) {
            if (v > first) emit((int)first, (int)(v - first));
            first = v;
            acc = 0;
            if (d > COL_EDGES) {
                for (int j = 0; j <= (d - 1) / COL_EDGES; ++j) emit((int)v, -1 - j);
                first = v + 1;
                continue;
            }
        }
        acc += d;
    }
    if (v1 > first) emit((int)first, (int)(v1 - first));
}

// Tickets per block into cnt[block] (FILL false), or written from at[block] on (FILL true).
template <bool FILL>
__global__ void k_color_tickets(const int *row, int n, int *cnt, const int *at, int2 *tick) {
    const long long nb = ((long long)n + COL_BLOCK - 1) / COL_BLOCK;
    for (long long b = (long long)blockIdx.x * blockDim.x + threadIdx.x; b <= nb; b += (long long)gridDim.x * blockDim.x) {
        if (!FILL && b == nb) cnt[b] = 0;
        if (b == nb) continue;
        const long long v0 = b * COL_BLOCK, v1 = v0 + COL_BLOCK < n ? v0 + COL_BLOCK : n;
        int k = FILL ? at[b] : 0;
        col_cut(row, v0, v1, [&](int v, int what) {
            if (FILL) tick[k] = make_int2(v, what);
            ++k;
        });
        if (!FILL) cnt[b] = k;
    }
}

// One wavefront's ticket in LDS.
struct ColWave {
    int row[COL_BLOCK + 1];  // edge offsets of its vertices
    int best[COL_BLOCK];     // largest settled neighbour color
    int wait[COL_BLOCK];     // edges without one
    int color[COL_BLOCK];    // color once stored, else 0
};

__device__ __forceinline__ int col_load(const int *p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void col_store(int *p, int v) {
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// The solve: wavefronts take tickets until none is left (ntick = the number of tickets, on the
// device).  What bounds it is the longest chain of dependencies (about as many hops as colors),
// each hop one store and the poll that sees it; the edges themselves are read once.  The last
// chunk of a long row waits for part[] of the other chunks (their largest color + 1).
// ctl[0] = next ticket, ctl[1] = largest color, ctl[2] = set when a poll ran out of patience (the
// launch then drains).
__global__ __launch_bounds__(256) void k_color_solve(const int *row, const int *col, const int2 *tick, const int *ntick,
                                                     int *part, int *color, int *ctl) {
    __shared__ ColWave s_w[4];
    ColWave &w = s_w[threadIdx.x >> 6];
    const int lane = col_lane();
    const int nt = *ntick;
    int top = 0;
    for (;;) {
        int t = 0;
        if (lane == 0) t = atomicAdd(&ctl[0], 1);
        t = __builtin_amdgcn_readfirstlane(t);
        if (t >= nt) break;
        const int2 tk = tick[t];
        const int v0 = tk.x, nv = tk.y < 0 ? 1 : tk.y, chunk = tk.y < 0 ? -1 - tk.y : 0;
        if (lane < nv) {
            w.row[lane] = row[v0 + lane];
            w.best[lane] = 0;
            w.wait[lane] = 0;
            w.color[lane] = 0;
        }
        if (lane == 0) w.row[nv] = row[v0 + nv];
        wave_lds_order();
        const int e0 = w.row[0] + chunk * COL_EDGES;
        const int left = w.row[nv] - e0;                      // edges from this ticket's first on
        const int ne = left < COL_EDGES ? left : COL_EDGES;
        const bool leads = left <= COL_EDGES;                 // stores colors (else: its part only)
        int next = leads ? t - chunk : t;                     // parts [next, t) still to be seen
        int u[COL_UNR], sl[COL_UNR], c[COL_UNR];
#pragma unroll
        for (int k = 0; k < COL_UNR; ++k) u[k] = 64 * k + lane < ne ? col[e0 + 64 * k + lane] : -1;
#pragma unroll
        for (int k = 0; k < COL_UNR; ++k) {  // owner: the last vertex whose offset is at or before the edge
            int o = 0;
#pragma unroll
            for (int step = COL_BLOCK / 2; step > 0; step >>= 1)
                if (o + step < nv && w.row[o + step] - e0 <= 64 * k + lane) o += step;
            sl[k] = o;
            if (u[k] >= v0 + o) u[k] = -1;  // only smaller neighbours count
        }
#pragma unroll
        for (int k = 0; k < COL_UNR; ++k) c[k] = u[k] >= 0 && u[k] < v0 ? col_load(color + u[k]) : 0;
#pragma unroll
        for (int k = 0; k < COL_UNR; ++k) {
            if (u[k] < 0) continue;
            if (c[k]) { atomicMax(&w.best[sl[k]], c[k]); u[k] = -1; }
            else atomicAdd(&w.wait[sl[k]], 1);
        }
        bool mine = lane < nv;   // this lane's vertex (or part) is not stored yet
        bool fresh = false;      // a vertex of the ticket got its color in the last round
        unsigned long long spins = 0;
        for (;;) {
            wave_lds_order();
            const bool ready = mine && next == t && w.wait[lane] == 0;
            if (ready) {
                const int cv = w.best[lane] + 1;
                if (leads) {
                    w.color[lane] = cv;
                    col_store(color + v0 + lane, cv);
                    top = cv > top ? cv : top;
                } else {
                    col_store(part + t, cv);
                }
                mine = false;
            }
            if (__ballot(mine) == 0) break;
            fresh = __ballot(ready) != 0;
            wave_lds_order();
            // a color of the ticket's own vertices settles its successors from LDS; only without
            // one are the other wavefronts' colors read again
#pragma unroll
            for (int k = 0; k < COL_UNR; ++k) {
                c[k] = 0;
                if (u[k] >= v0) c[k] = w.color[u[k] - v0];
                else if (u[k] >= 0 && !fresh) c[k] = col_load(color + u[k]);
            }
            if (!fresh && next < t) {
                const int p = next + lane < t ? col_load(part + next + lane) : 1;
                if (__ballot(p == 0) == 0) {
                    if (p > 1) atomicMax(&w.best[0], p - 1);
                    next = next + 64 < t ? next + 64 : t;
                }
            }
#pragma unroll
            for (int k = 0; k < COL_UNR; ++k) {
                if (c[k] == 0) continue;
                atomicMax(&w.best[sl[k]], c[k]);
                atomicSub(&w.wait[sl[k]], 1);
                u[k] = -1;
            }
            if (!fresh && (++spins & 1023) == 0) {
                const int stop = __builtin_amdgcn_readfirstlane(col_load(&ctl[2]));
                if (stop || spins > COL_SPIN_LIMIT) {
                    if (lane == 0) col_store(&ctl[2], 1);
                    return;
                }
            }
        }
        wave_lds_order();
    }
    for (int o = 32; o > 0; o >>= 1) { const int x = __shfl_xor(top, o); top = x > top ? x : top; }
    if (lane == 0 && top) atomicMax(&ctl[1], top);
}

// The reference's round as it is (method 1): every uncolored vertex checks its smaller
// out-neighbours (graph_color_kernel.cu:14-35).
__global__ void k_color_round(const int *row, const int *col, int n, int *color, int c, int *nonstop) {
    for (long long v = (long long)blockIdx.x * blockDim.x + threadIdx.x; v < n; v += (long long)gridDim.x * blockDim.x) {
        if (color[v] != 0) continue;
        bool ok = true;
        for (int e = row[v]; e < row[v + 1]; ++e) {
            const int u = col[e];
            if (u < v) {
                const int cu = __hip_atomic_load(color + u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                if (cu == 0 || cu == c) { ok = false; break; }
            }
        }
        if (ok) {
            __hip_atomic_store(color + v, c, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            *nonstop = 1;
        }
    }
}

long long color_blocks(int n) { return ((long long)n + COL_BLOCK - 1) / COL_BLOCK; }
// a run or first chunk per vertex at most, and a further chunk per COL_EDGES edges
long long color_ticket_cap(int n, long long m) { return (long long)n + m / COL_EDGES + 1; }
hipError_t color_scan(void *temp, size_t *temp_bytes, const int *in, int *out, int n, hipStream_t s) {
    return rocprim::exclusive_scan(temp, *temp_bytes, in, out, 0, (size_t)color_blocks(n) + 1, rocprim::plus<int>(), s);
}
hipError_t launch_color_solve(const int *row, const int *col, int n, long long m, const ColorBufs &b, int num_cus,
                              hipStream_t s) {
    const long long nb = color_blocks(n);
    const dim3 tgrid(col_grid(nb + 1, 4096));
    hipLaunchKernelGGL(k_color_tickets<false>, tgrid, dim3(256), 0, s, row, n, b.cnt, (const int *)nullptr, (int2 *)nullptr);
    size_t tb = b.temp_bytes;
    hipError_t e = color_scan(b.temp, &tb, b.cnt, b.at, n, s);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(k_color_tickets<true>, tgrid, dim3(256), 0, s, row, n, (int *)nullptr, b.at, b.tick);
    hipLaunchKernelGGL(k_color_solve, dim3(col_grid((nb + m / COL_EDGES) * 64, num_cus * COL_WGS)), dim3(256), 0, s, row, col, b.tick, b.at + nb,
                       b.part, b.color, b.ctl);
    return hipGetLastError();
}
hipError_t launch_color_round(const int *row, const int *col, int n, int *color, int c, int *nonstop, hipStream_t s) {
    hipLaunchKernelGGL(k_color_round, dim3(col_grid(n, 8192)), dim3(256), 0, s, row, col, n, color, c, nonstop);
    return hipGetLastError();
}
}  // namespace np
