// PageRank of the reference's PAGERANK_GPU (apps/pagerank/src/gpu/pagerank_wrapper.cu:147-244,
// 565-661; kernels pagerank_kernel.cu:60-107; constants pagerank_wrapper.cu:5-6 and pagerank.h:15).
//
// The reference pulls over the inverted graph (invertGraph, common/global.cpp:237-276): per
// iteration new[v] = damping * sum over in-edges p -> v of rank[p] / outdeg[p]
//                    + (1 - damping) * TOTAL / n + damping * (rank held by dangling vertices) / n,
// from rank = TOTAL / n, until no vertex changes by more than EPSILON (damping 0.5, TOTAL 1000,
// EPSILON 1e-13).  Parallel edges count once per edge in both the sum and outdeg.
//
// MI355X mapping: the in-edge CSR is built once on the device (a rocPRIM radix sort of the
// (target, source) pairs, offsets from the sorted targets) from the solver's layout, which on a
// skewed graph numbers the vertices by decreasing in-degree, so that the contributions most often
// read lie together.  An iteration is one launch (k_pr_pull): it gathers the contributions
// rank/outdeg, writes each new rank in place and its contribution for the next iteration, and sums
// the next iteration's dangling ranks and the largest change (workgroup reductions, one float64
// atomicAdd and one integer atomicMax on the non-negative float64 bits per workgroup); whether the
// run has ended is read from the previous iteration's largest change.  The pull splits vertices by
// in-degree (bins built once): fewer than 32 in-edges, 8 lanes per vertex (consecutive in-edges,
// coalesced); up to PR_HUGE, one wavefront per vertex; longer (R-MAT hubs reach 10^5 in-edges, a
// single wavefront on one would be the whole pass's tail), PR_CHUNK-entry chunks on one wavefront
// each, whose partial sums the wavefront that finishes last adds in chunk order, so a row's sum does
// not depend on scheduling.  The dangling sum does, in its last bits: it is added up by atomics in
// order of arrival.  All in float64, so the reference's EPSILON is reachable (float ranks near 1000/n cannot move by
// less than an ulp ~1e-9); ranks are returned as float32, the reference's FLOAT_T.  The file also
// holds SpMV (apps/SpMV), the same row-split product without PageRank's terms.
#include <hip/hip_runtime.h>
#include <cstring>
#include <rocprim/device/device_radix_sort.hpp>
#include <rocprim/device/device_scan.hpp>
#include "np_internal.h"

namespace np {

__device__ __forceinline__ int pr_lane() { return threadIdx.x & 63; }

static int pr_grid(long long work, int cap) {
    long long g = (work + 255) / 256;
    return (int)(g < 1 ? 1 : (g > cap ? cap : g));
}

// Sum over entries [e0, e1) of term(e) (a medium row or a chunk: positions count from e0, so they
// cannot overflow), lanes striding by 64 with four loads in flight per lane, reduced over the
// wavefront (every lane returns the total).
template <class F>
__device__ __forceinline__ double pr_wave_sum(int e0, int e1, F term) {
    const int len = e1 - e0;
    double s0 = 0.0, s1 = 0.0, s2 = 0.0, s3 = 0.0;
    int k = pr_lane();
    for (; k + 192 < len; k += 256) {
        s0 += term(e0 + k);
        s1 += term(e0 + k + 64);
        s2 += term(e0 + k + 128);
        s3 += term(e0 + k + 192);
    }
    for (; k < len; k += 64) s0 += term(e0 + k);
    double s = (s0 + s1) + (s2 + s3);
    for (int x = 32; x > 0; x >>= 1) s += __shfl_xor(s, x);
    return s;
}

// The in-edge CSR is the transpose: a stable radix sort of the (target, source) pairs puts every
// vertex's in-edges together, sources ascending (the order the reference's invertGraph lists
// them, common/global.cpp:237-276), with no per-edge atomics (hub targets would serialise them).
// src[e] = the source of edge e: each vertex with out-edges writes its id at its first edge
// (heads, zero elsewhere), and an inclusive max-scan over the edges carries it to the rest of
// its edges (ids grow with the position).  One wavefront per vertex left most lanes idle on
// R-MAT's short rows (0.2 ms at scale 20).
__global__ void k_pr_heads(const int *row, int n, int *heads) {
    for (long long v = (long long)blockIdx.x * blockDim.x + threadIdx.x; v < n; v += (long long)gridDim.x * blockDim.x)
        if (row[v + 1] > row[v]) heads[row[v]] = (int)v;
}

// irow[u] = the first sorted position with target >= u, for u = 0..n (irow holds m before: the
// vertices after the last target, on a renumbered graph all without in-edges).
__global__ void k_pr_offsets(const unsigned *key, long long m, int *irow) {
    for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < m; i += (long long)gridDim.x * blockDim.x) {
        const long long prev = i > 0 ? (long long)key[i - 1] : -1;
        for (long long u = prev + 1; u <= (long long)key[i]; ++u) irow[u] = (int)i;
    }
}

// Row bins (rows: a vertex's in-edges for PageRank, a matrix row for SpMV), built once.  Rows
// of PR_HEAVY..PR_HUGE-1 entries go to med[]; longer rows to huge[], with their chunks (row,
// chunk index) in crow/ck from hc0[h] on: ceil(len / PR_CHUNK) <= 1.5 len / PR_CHUNK chunks per
// huge row, so at most 1.5 m / PR_CHUNK in all (pr_chunk_cap); the cap check never fires.
// Each workgroup takes a contiguous range of rows: it counts its medium rows, reserves their
// slots with one global atomic (one per wave or per row would serialise on the counter), then
// writes them at offsets taken from an LDS counter.  Huge rows are rare: plain atomics.
__global__ __launch_bounds__(256) void k_pr_bins(const int *off, int n, RowBins rb, long long chunk_cap) {
    __shared__ int cnt, base;
    const long long per = ((long long)n + gridDim.x - 1) / gridDim.x;
    const long long v0 = (long long)blockIdx.x * per;
    const long long v1 = v0 + per < n ? v0 + per : n;
    const int lane = pr_lane();
    if (threadIdx.x == 0) cnt = 0;
    __syncthreads();
    int mine = 0;
    for (long long v = v0 + threadIdx.x; v < v1; v += blockDim.x) {
        const long long len = (long long)(off[v + 1] - off[v]);
        mine += len >= PR_HEAVY && len < PR_HUGE;
        if (len >= PR_HUGE) {
            const int k = (int)((len + PR_CHUNK - 1) / PR_CHUNK);
            const int h = atomicAdd(rb.nhuge, 1);
            const int c0 = atomicAdd(rb.nchunk, k);
            rb.huge[h] = (int)v;
            rb.hc0[h] = c0;
            if (rb.hleft) rb.hleft[h] = k;
            if (c0 + (long long)k <= chunk_cap)
                for (int j = 0; j < k; ++j) { rb.crow[c0 + j] = (int)v; rb.ck[c0 + j] = j; if (rb.chuge) rb.chuge[c0 + j] = h; }
        }
    }
    for (int k = 32; k > 0; k >>= 1) mine += __shfl_xor(mine, k);
    if (lane == 0 && mine) atomicAdd(&cnt, mine);
    __syncthreads();
    if (threadIdx.x == 0) {
        base = cnt ? atomicAdd(rb.nmed, cnt) : 0;
        cnt = 0;
    }
    __syncthreads();
    for (long long t = v0; t < v1; t += blockDim.x) {  // trip count uniform over the workgroup
        const long long v = t + threadIdx.x;
        const long long len = v < v1 ? (long long)(off[v + 1] - off[v]) : 0;
        const bool take = len >= PR_HEAVY && len < PR_HUGE;
        const unsigned long long want = __ballot(take);
        if (want == 0) continue;
        const int leader = __ffsll((long long)want) - 1;
        int b = 0;
        if (lane == leader) b = atomicAdd(&cnt, __popcll(want));
        b = __shfl(b, leader);
        if (take) rb.med[base + b + __popcll(want & ((1ull << lane) - 1))] = (int)v;
    }
}

// workgroup sum of one double per thread -> one atomicAdd (all threads call it)
__device__ __forceinline__ void pr_block_add(double x, double *dst) {
    __shared__ double s[4];
    for (int o = 32; o > 0; o >>= 1) x += __shfl_xor(x, o);
    if (pr_lane() == 0) s[threadIdx.x >> 6] = x;
    __syncthreads();
    if (threadIdx.x == 0) {
        const double t = s[0] + s[1] + s[2] + s[3];
        if (t != 0.0) atomicAdd(dst, t);
    }
    __syncthreads();
}

// workgroup max of one non-negative double per thread -> one atomicMax on its bit pattern
__device__ __forceinline__ void pr_block_max(double x, unsigned long long *dst) {
    __shared__ double s[4];
    for (int o = 32; o > 0; o >>= 1) { const double y = __shfl_xor(x, o); x = y > x ? y : x; }
    if (pr_lane() == 0) s[threadIdx.x >> 6] = x;
    __syncthreads();
    if (threadIdx.x == 0) {
        double t = s[0];
        for (int k = 1; k < 4; ++k) t = s[k] > t ? s[k] : t;
        if (t > 0.0) atomicMax(dst, (unsigned long long)__double_as_longlong(t));
    }
    __syncthreads();
}

// Contribution of a vertex with d out-edges to each of its out-neighbours; a dangling vertex (no
// out-edges) contributes nothing there and its rank to *dang.
__device__ __forceinline__ double pr_share(double r, int d, double *dang) {
    if (d > 0) return r / (double)d;
    *dang += r;
    return 0.0;
}

// rank = r0, the first contributions and the first dangling sum; the counters of iteration 0
__global__ __launch_bounds__(256) void k_pr_init(const int *row, int n, double r0, double *rank, double *contrib,
                                                  PrSums *ps) {
    double dang = 0.0;
    for (long long v = (long long)blockIdx.x * blockDim.x + threadIdx.x; v < n; v += (long long)gridDim.x * blockDim.x) {
        rank[v] = r0;
        contrib[v] = pr_share(r0, row[v + 1] - row[v], &dang);
    }
    pr_block_add(dang, &ps->slot[blockIdx.x & (PR_SLOTS - 1)].dsum[0]);
}

// One iteration (the i-th).  Wavefront items: chunks of huge rows, medium rows, then groups of
// 64 / PR_GROUP consecutive vertices of which the light ones are taken.  The sums rotate over three
// entries: dsum[i % 3] and dmax[(i - 1) % 3] are read, dsum[(i + 1) % 3] and dmax[i % 3] are added to,
// dsum[(i + 2) % 3] and dmax[(i + 1) % 3] are cleared for the next iteration.  After an iteration
// that changed no vertex by more than eps the later ones only clear their slot and return.
// What bounds it is the gather of contributions (random 8-byte reads of an 8 MB array run at 81 G/s
// here; renumbered, R-MAT s20 reaches 160 G/s): 104 us per iteration against 192 us of five launches
// over the original numbering; one call 5.4 -> 3.2 ms.  16 workgroups per CU instead of 8: +23 us.
__global__ __launch_bounds__(256) void k_pr_pull(int i, PrSums *ps, RowBins rb, const int *irow, const int *pcol,
                                                  const int *row, const double *contrib, double *ncontrib, double *rank,
                                                  int n, double damping, double rw, double eps) {
    // the slots' sums, every wavefront for itself (lane l on slot l, the butterfly's order)
    static_assert(PR_SLOTS == 64, "a lane per slot");
    PrSlot &mine = ps->slot[threadIdx.x & 63];
    double dsum = mine.dsum[i % 3], change = __longlong_as_double((long long)mine.dmax[(i + 2) % 3]);
    for (int o = 32; o > 0; o >>= 1) {
        dsum += __shfl_xor(dsum, o);
        const double y = __shfl_xor(change, o);
        change = y > change ? y : change;
    }
    const bool ended = i > 0 && !(change > eps);
    if (blockIdx.x == 0 && threadIdx.x < 64) {
        mine.dmax[(i + 1) % 3] = 0;
        if (!ended) {
            mine.dsum[(i + 2) % 3] = 0.0;
            ps->iters = i + 1;
        }
    }
    if (ended) return;  // uniform over the grid, before any barrier
    const double base_add = rw + damping * dsum / (double)n;
    const int lane = pr_lane();
    const long long nc = *rb.nchunk, nm = *rb.nmed;
    constexpr int PER = 64 / PR_GROUP;
    const long long items = nc + nm + ((long long)n + PER - 1) / PER;
    const long long nw = (long long)gridDim.x * (blockDim.x >> 6);
    auto term = [&](int e) { return contrib[pcol[e]]; };
    double mx = 0.0, dang = 0.0;
    auto finish = [&](int v, double s) {
        const double r = damping * s + base_add, dd = fabs(r - rank[v]);
        rank[v] = r;
        ncontrib[v] = pr_share(r, row[v + 1] - row[v], &dang);
        mx = dd > mx ? dd : mx;
    };
    for (long long o = (long long)blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6); o < items; o += nw) {
        if (o >= nc + nm) {
            const long long v = (o - nc - nm) * PER + lane / PR_GROUP;
            const int e0 = v < n ? irow[v] : 0, len = v < n ? irow[v + 1] - e0 : 0;
            const bool light = v < n && len < PR_HEAVY;
            const int sub = lane & (PR_GROUP - 1);
            double t[PR_HEAVY / PR_GROUP];
#pragma unroll
            for (int k = 0; k < PR_HEAVY / PR_GROUP; ++k) {  // every load of the row in flight
                const int at = sub + k * PR_GROUP;
                t[k] = light && at < len ? term(e0 + at) : 0.0;
            }
            double s = 0.0;
#pragma unroll
            for (int k = 0; k < PR_HEAVY / PR_GROUP; ++k) s += t[k];
            for (int k = PR_GROUP / 2; k > 0; k >>= 1) s += __shfl_xor(s, k);
            if (light && sub == 0) finish((int)v, s);
        } else if (o >= nc) {
            const int v = rb.med[o - nc];
            const double s = pr_wave_sum(irow[v], irow[v + 1], term);
            if (lane == 0) finish(v, s);
        } else {
            const int v = rb.crow[o], h = rb.chuge[o];
            const int e0 = irow[v] + rb.ck[o] * PR_CHUNK, end = irow[v + 1];
            const double s = pr_wave_sum(e0, end - e0 < PR_CHUNK ? end : e0 + PR_CHUNK, term);
            int last = 0;
            if (lane == 0) {
                // the partial sum is in memory before the count tells so
                __hip_atomic_store(rb.part + o, s, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                stores_done();
                last = atomicSub(&rb.hleft[h], 1) == 1;
            }
            if (__builtin_amdgcn_readfirstlane(last)) {
                __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");  // no read of part[] before the count
                const int k = (int)(((long long)end - irow[v] + PR_CHUNK - 1) / PR_CHUNK);
                double t = 0.0;  // lane by lane and then the butterfly: the same order every time
                for (int j = lane; j < k; j += 64)
                    t += __hip_atomic_load(rb.part + rb.hc0[h] + j, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                for (int x = 32; x > 0; x >>= 1) t += __shfl_xor(t, x);
                if (lane == 0) {
                    rb.hleft[h] = k;  // for the next iteration
                    finish(v, t);
                }
            }
        }
    }
    PrSlot &to = ps->slot[blockIdx.x & (PR_SLOTS - 1)];
    pr_block_add(dang, &to.dsum[(i + 1) % 3]);
    pr_block_max(mx, &to.dmax[i % 3]);
}

// ---- SpMV (apps/SpMV/src/gpu/SpMV_kernel.cu:77-92, csr_spmv_kernel): y[v] = sum over the
// row's entries of data[e] * x[col[e]], with the pull's row bins.
__global__ __launch_bounds__(256) void k_spmv_light(const int *row, const int *col, const double *data,
                                                     const double *x, double *y, int n) {
    const int sub = threadIdx.x & (PR_GROUP - 1);
    const long long groups = (long long)gridDim.x * (blockDim.x / PR_GROUP);
    const long long nv = ((long long)n + 63) / 64 * 64;  // whole waves: same trips in every lane
    for (long long v = ((long long)blockIdx.x * blockDim.x + threadIdx.x) / PR_GROUP; v < nv; v += groups) {
        const bool light = v < n && row[v + 1] - row[v] < PR_HEAVY;
        double s = 0.0;
        if (light)
            for (int e = row[v] + sub; e < row[v + 1]; e += PR_GROUP) s += data[e] * x[col[e]];
        for (int o = PR_GROUP / 2; o > 0; o >>= 1) s += __shfl_xor(s, o);
        if (light && sub == 0) y[v] = s;
    }
}
__global__ __launch_bounds__(256) void k_spmv_wave(RowBins rb, const int *row, const int *col, const double *data,
                                                    const double *x, double *y) {
    const int nc = *rb.nchunk, nm = *rb.nmed;
    const long long nw = (long long)gridDim.x * (blockDim.x >> 6);
    auto term = [&](int e) { return data[e] * x[col[e]]; };
    for (long long o = (long long)blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6); o < (long long)nc + nm; o += nw) {
        if (o < nc) {
            const int v = rb.crow[o];
            const int e0 = row[v] + rb.ck[o] * PR_CHUNK;
            const int e1 = e0 + PR_CHUNK < row[v + 1] ? e0 + PR_CHUNK : row[v + 1];
            const double s = pr_wave_sum(e0, e1, term);
            if (pr_lane() == 0) rb.part[o] = s;
        } else {
            const int v = rb.med[o - nc];
            const double s = pr_wave_sum(row[v], row[v + 1], term);
            if (pr_lane() == 0) y[v] = s;
        }
    }
}
__global__ void k_spmv_huge(RowBins rb, const int *row, double *y) {
    const int nh = *rb.nhuge;
    for (long long h = (long long)blockIdx.x * blockDim.x + threadIdx.x; h < nh; h += (long long)gridDim.x * blockDim.x) {
        const int v = rb.huge[h];
        const int k = (row[v + 1] - row[v] + PR_CHUNK - 1) / PR_CHUNK;
        double s = 0.0;
        for (int j = 0; j < k; ++j) s += rb.part[rb.hc0[h] + j];
        y[v] = s;
    }
}

// ranks in original vertex ids (old2new null: the layout is the original one)
__global__ void k_pr_to_float(const double *rank, const int *old2new, int n, float *out) {
    for (long long v = (long long)blockIdx.x * blockDim.x + threadIdx.x; v < n; v += (long long)gridDim.x * blockDim.x)
        out[v] = (float)rank[old2new ? old2new[v] : v];
}

hipError_t pr_sources(void *temp, size_t *temp_bytes, const int *row, int n, long long m, int *heads, int *src,
                      hipStream_t s) {
    if (!temp)
        return rocprim::inclusive_scan(nullptr, *temp_bytes, heads, src, (size_t)m, rocprim::maximum<int>(), s);
    hipError_t e = hipMemsetAsync(heads, 0, sizeof(int) * (size_t)m, s);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(k_pr_heads, dim3(pr_grid(n, 4096)), dim3(256), 0, s, row, n, heads);
    if ((e = hipGetLastError()) != hipSuccess) return e;
    return rocprim::inclusive_scan(temp, *temp_bytes, heads, src, (size_t)m, rocprim::maximum<int>(), s);
}
hipError_t launch_pr_offsets(const unsigned *key, long long m, int n, int *irow, hipStream_t s) {
    hipError_t e = launch_fill_i32(irow, (long long)n + 1, (int)m, s);
    if (e != hipSuccess || m == 0) return e;
    hipLaunchKernelGGL(k_pr_offsets, dim3(pr_grid(m, 8192)), dim3(256), 0, s, key, m, irow);
    return hipGetLastError();
}
long long pr_chunk_cap(long long m) { return 3 * m / (2 * PR_CHUNK) + 1; }
hipError_t launch_row_bins(const int *off, int n, long long m, const RowBins &rb, hipStream_t s) {
    hipLaunchKernelGGL(k_pr_bins, dim3(pr_grid(n, 2048)), dim3(256), 0, s, off, n, rb, pr_chunk_cap(m));
    return hipGetLastError();
}
hipError_t launch_pr_init(const int *row, int n, double r0, double *rank, double *contrib, PrSums *ps, hipStream_t s) {
    hipLaunchKernelGGL(k_pr_init, dim3(pr_grid(n, 1024)), dim3(256), 0, s, row, n, r0, rank, contrib, ps);
    return hipGetLastError();
}
hipError_t launch_pr_iteration(int i, PrSums *ps, const int *row, const int *irow, const int *pcol, const RowBins &rb,
                               double *rank, const double *contrib, double *ncontrib, int n, long long m, double damping,
                               double rw, double eps, int num_cus, hipStream_t s) {
    const long long work = (long long)n * PR_GROUP + m / 4;  // lanes: light groups, and the rows of the wavefronts
    hipLaunchKernelGGL(k_pr_pull, dim3(pr_grid(work, num_cus * 8)), dim3(256), 0, s, i, ps, rb, irow, pcol, row, contrib,
                       ncontrib, rank, n, damping, rw, eps);
    return hipGetLastError();
}
hipError_t launch_spmv(const int *row, const int *col, const double *data, const double *x, double *y, int n,
                       const RowBins &rb, int num_cus, hipStream_t s) {
    hipLaunchKernelGGL(k_spmv_light, dim3(pr_grid((long long)n * PR_GROUP, num_cus * 16)), dim3(256), 0, s, row, col,
                       data, x, y, n);
    hipLaunchKernelGGL(k_spmv_wave, dim3(num_cus * 8), dim3(256), 0, s, rb, row, col, data, x, y);
    hipLaunchKernelGGL(k_spmv_huge, dim3(4), dim3(256), 0, s, rb, row, y);
    return hipGetLastError();
}
hipError_t launch_pr_to_float(const double *rank, const int *old2new, int n, float *out, hipStream_t s) {
    hipLaunchKernelGGL(k_pr_to_float, dim3(pr_grid(n, 4096)), dim3(256), 0, s, rank, old2new, n, out);
    return hipGetLastError();
}
// Stable sort of m (key, value) pairs on key bits [0, end_bit).
hipError_t pr_sort(void *temp, size_t *temp_bytes, const unsigned *key_in, unsigned *key_out, const int *val_in,
                   int *val_out, long long m, int end_bit, hipStream_t s) {
    return rocprim::radix_sort_pairs(temp, *temp_bytes, key_in, key_out, val_in, val_out, (size_t)m, 0u,
                                     (unsigned)end_bit, s);
}

}  // namespace np
