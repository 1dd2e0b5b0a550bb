// Betweenness centrality (Brandes) on the frontier machinery, up to 32 sources per batch.
//
// Reference: apps/bc/src/gpu/bc_wrapper.cu:678-761 (bc_np_consolidate_gpu: a level-synchronous
// forward BFS that counts shortest paths, then a backward sweep over the levels) with the
// kernels of bc_fp_kernel.cu:429-489 (forward: a vertex reached at level d+1 adds the path count
// of every level-d predecessor, sigma[w] += sigma[u]) and bc_bp_kernel.cu:4-36 (backward:
// delta[v] += sigma[v] / sigma[w] * (1 + delta[w]) over the edges v -> w into the next level;
// bc[v] += delta[v] for v != source).  Here the factor (1 + delta[w]) / sigma[w] is formed once
// per slot when w's level is final and read as one value by the level above.  The reference
// keeps an n x n predecessor byte matrix; here an edge u -> w is a predecessor edge exactly
// when level[w] = level[u] + 1, which is what that matrix records, so no n^2 state exists.
//
// Layout: the sources of a batch share rows of 2^ks slots, slot (v << ks) + j for source j, as
// the source-packed SSSP does: level (int), sigma and delta (double: path counts stay exact
// integers up to 2^53).  A forward expansion of level d turns the entries (v, mask of the
// sources for which v is at level d) into level d + 1 flags (nmask); the compaction writes the
// next level's entries after the previous ones, so the backward sweep replays every level's
// entries in reverse order.
//
// Work split: entry o has deg(v) x P' items, P' = popc(mask) rounded up to a power of two, item
// r = (edge r / P', source slot r % P').  Items are cut into BC_ITEMS-item chunks (one wavefront
// each, BC_UNR items per lane, their loads in flight together: a chain of five dependent accesses
// per chunk is what bounds the sweeps, so a chunk of 64 items ran at a quarter of the rate); each
// entry's chunks are reserved as one contiguous range of the level's chunk counter (one atomic per
// wavefront of entries, no prefix sum) and an owner array maps every chunk to its entry.  64 is a
// multiple of P', so a lane's source slot is lane % P' for all of its items and the lanes of one
// source are lane, lane ^ P', ...: the backward sweep sums them with xor-shuffles before one
// atomicAdd per source.  A forward level is two launches (compaction with owners, expansion), a
// backward level two (the finished level's factors with the next one's owners, sweep).  256 sources
// of R-MAT s16 (65,536 / 1 M): 5.9 ms per call; with 64-item chunks, a compare-and-swap per unseen
// slot and four launches per level 10.3 ms.
#include <hip/hip_runtime.h>
#include <algorithm>
#include "np_internal.h"

namespace np {

__device__ __forceinline__ int bc_lane() { return threadIdx.x & 63; }

constexpr int BC_UNR = 4;
constexpr int BC_ITEMS = 64 * BC_UNR;

// chunks of the entry (v, m): ceil(deg(v) x P' / BC_ITEMS)
__device__ __forceinline__ long long bc_nchunks(const BcDev &b, int v, unsigned m) {
    const int p = __popc(m);
    const int lp = p <= 1 ? 0 : 32 - __clz(p - 1);
    return (((long long)(b.row[v + 1] - b.row[v]) << lp) + BC_ITEMS - 1) / BC_ITEMS;
}

// Every lane of the wave calls it: k chunks for this lane's entry (0 for none) are reserved on
// *ctot; returns the first chunk of the lane's range.
__device__ __forceinline__ long long bc_reserve(long long k, unsigned long long *ctot) {
    const int lane = bc_lane();
    long long incl = k;
    for (int o = 1; o < 64; o <<= 1) {
        const long long t = __shfl_up(incl, o);
        if (lane >= o) incl += t;
    }
    const long long tot = __shfl(incl, 63);
    long long base = 0;
    if (lane == 0 && tot) base = (long long)atomicAdd(ctot, (unsigned long long)tot);
    base = __shfl(base, 0);
    return base + incl - k;
}

// k-th set bit of m (k < popc(m))
__device__ __forceinline__ int bc_nth_bit(unsigned m, int k) {
    for (int i = 0; i < k; ++i) m &= m - 1;
    return __ffs(m) - 1;
}

__global__ void k_bc_reset(BcDev b) {
    const long long slots = (long long)b.n << b.ks;
    for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < slots;
         i += (long long)gridDim.x * blockDim.x) {
        b.lvl[i] = BC_UNSEEN;
        b.sig[i] = 0.0;
        b.del[i] = 0.0;
        if (i < b.n) b.nmask[i] = 0u;
    }
}

__global__ void k_bc_sources(BcDev b, const int *srcs, int nsrc) {
    const int j = threadIdx.x;
    if (blockIdx.x != 0 || j >= nsrc) return;
    const int s = srcs[j];
    const long long k = ((long long)s << b.ks) + j;
    b.lvl[k] = 0;
    b.sig[k] = 1.0;
    atomicOr(&b.nmask[s], 1u << j);
}

// owner[c] = o for this lane's k chunks from `first` on (every lane of the wave calls it; the wave
// writes one lane's range after another).  A level has at most m / 8 + ne chunks (deg x 32 / 256 + 1
// per entry); a range past cap sets *err and nothing is written past it.
__device__ __forceinline__ void bc_own(long long first, long long k, int o, int *owner, long long cap, int *err) {
    const int lane = bc_lane();
    unsigned long long m = __ballot(k > 0);
    while (m) {
        const int l = __ffsll((long long)m) - 1;
        m &= m - 1;
        const long long c0 = __shfl(first, l), c1 = c0 + __shfl(k, l);
        const int ol = __shfl(o, l);
        if (c1 > cap && lane == 0) *err = 1;
        const long long ce = c1 < cap ? c1 : cap;
        for (long long c = c0 + lane; c < ce; c += 64) owner[c] = ol;
    }
}

// Flagged vertices -> entries (v, mask) at ent_v/ent_m + lv[d].x + (position counted in lv[d].y),
// the first chunk of each at cst[position] (chunks reserved on *ctot) and the chunks' owners.
// Entries of all levels fit in n x sources: every (vertex, source) pair is in one level's entry and
// every entry holds at least one.
__global__ void k_bc_compact(BcDev b, int *ent_v, unsigned *ent_m, int2 *lv, int d, long long *cst,
                             unsigned long long *ctot, int *owner, long long cap, int *err) {
    const int E = lv[d].x;
    int *count = &lv[d].y;
    for (long long base = (long long)blockIdx.x * blockDim.x; base < b.n; base += (long long)gridDim.x * blockDim.x) {
        const long long v = base + threadIdx.x;
        const unsigned m = v < b.n ? b.nmask[v] : 0u;
        const unsigned long long want = __ballot(m != 0);
        if (want == 0) continue;
        const int lane = bc_lane();
        const int leader = __ffsll((long long)want) - 1;
        int pos0 = 0;
        if (lane == leader) pos0 = atomicAdd(count, __popcll(want));
        pos0 = __shfl(pos0, leader);
        const long long k = m ? bc_nchunks(b, (int)v, m) : 0;
        const long long first = bc_reserve(k, ctot);
        const int pos = pos0 + __popcll(want & ((1ull << lane) - 1));
        if (m) {
            b.nmask[v] = 0u;
            ent_v[E + pos] = (int)v;
            ent_m[E + pos] = m;
            cst[pos] = first;
        }
        bc_own(first, k, pos, owner, cap, err);
    }
}

// One chunk per wavefront.  FWD: level d -> d + 1 with path counts; else the dependencies of level d
// from level d + 1.  The level's entries start at ent_v + lv[d].x (lv null: at ent_v); entry o's
// chunks start at cst[o]; *ctot is the chunk total.
template <bool FWD>
__global__ __launch_bounds__(256) void k_bc_expand(BcDev b, const int *ent_v, const unsigned *ent_m, int2 *lv,
                                                   const long long *cst, const int *owner,
                                                   const unsigned long long *ctot, long long cap, int d) {
    if (lv) {
        const int2 e = lv[d];
        ent_v += e.x;
        ent_m += e.x;
        // the next level's entries start after this one's (its record is not read in this launch)
        if (FWD && blockIdx.x == 0 && threadIdx.x == 0) lv[d + 1].x = e.x + e.y;
    }
    const int lane = bc_lane();
    const long long tot = (long long)*ctot;
    const long long nchunks = tot < cap ? tot : cap;
    const long long nw = (long long)gridDim.x * (blockDim.x >> 6);
    for (long long c = (long long)blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6); c < nchunks; c += nw) {
        const int o = owner[c];
        const int v = ent_v[o];
        const unsigned m = ent_m[o];
        const int p = __popc(m);
        const int lp = p <= 1 ? 0 : 32 - __clz(p - 1);
        const int e0 = b.row[v];
        const long long items = (long long)(b.row[v + 1] - e0) << lp;
        const long long r0 = (c - cst[o]) * BC_ITEMS + lane;
        const int j = lane & ((1 << lp) - 1);
        const int src = j < p ? bc_nth_bit(m, j) : 0;
        const double sv = j < p ? b.sig[((long long)v << b.ks) + src] : 0.0;
        int w[BC_UNR], cur[BC_UNR];
#pragma unroll
        for (int k = 0; k < BC_UNR; ++k)
            w[k] = j < p && r0 + 64 * k < items ? b.col[e0 + (int)((r0 + 64 * k) >> lp)] : -1;
#pragma unroll
        for (int k = 0; k < BC_UNR; ++k) cur[k] = w[k] >= 0 ? b.lvl[((long long)w[k] << b.ks) + src] : -1;
        if (FWD) {
            // Levels up to d were set by earlier launches and are final: <= d, w was reached before
            // (nothing to do).  d + 1 or unseen, v is a predecessor of w on level d + 1: the path
            // count; an unseen w (also one that this launch has set since: a read sees either) gets
            // its level, the same value from every writer, and is flagged, once per edge for all of
            // the edge's sources.
#pragma unroll
            for (int k = 0; k < BC_UNR; ++k) {
                const bool fresh = w[k] >= 0 && cur[k] > d + 1;
                const long long sw = ((long long)w[k] << b.ks) + src;
                if (w[k] >= 0 && cur[k] > d) atomicAdd(&b.sig[sw], sv);
                if (fresh) b.lvl[sw] = d + 1;
                if (__ballot(fresh) == 0) continue;
                unsigned bits = fresh ? 1u << src : 0u;
                for (int x = 1; x < (1 << lp); x <<= 1) bits |= (unsigned)__shfl_xor((int)bits, x);
                if (j == 0 && bits) atomicOr(&b.nmask[w[k]], bits);
            }
        } else {
            // level d + 1 is final: its slots hold (1 + delta) / sigma (k_bc_finish)
            double x = 0.0;
#pragma unroll
            for (int k = 0; k < BC_UNR; ++k)
                if (cur[k] == d + 1) x += sv * b.sig[((long long)w[k] << b.ks) + src];
            for (int off = 32; off >= (1 << lp); off >>= 1) x += __shfl_xor(x, off);
            if (lane < p && x != 0.0) atomicAdd(&b.del[((long long)v << b.ks) + src], x);
        }
    }
}

// Between two backward levels.  The finished level's ne entries (ent_v, ent_m): bc[v] += delta of v
// for every source of its entry (bc null: the level holds the sources), and the slot's sigma is
// replaced by (1 + delta) / sigma, the factor the level above needs from it (one gather there instead
// of two).  Each (vertex, source) slot is in exactly one level's entries, so it is transformed once,
// after its own level's sweep; the deepest level (delta 0) is passed through here too.  Half a
// wavefront per entry, lane j on the j-th source of its mask: the transforms run in parallel and the
// entry's deltas are summed with shuffles.
// The next level's nn entries (nxt_v, nxt_m), replayed: their chunk ranges (first chunk of each at
// cst[o], reserved on *ctot) and owners.
__global__ void k_bc_finish(BcDev b, const int *ent_v, const unsigned *ent_m, int ne, double *bc, const int *nxt_v,
                            const unsigned *nxt_m, int nn, long long *cst, unsigned long long *ctot, int *owner,
                            long long cap, int *err) {
    const int j = threadIdx.x & 31;
    const long long per = (long long)gridDim.x * (blockDim.x / 32);
    const long long half = ((long long)ne + 1) / 2 * 2;  // whole waves: both halves make the same trips
    for (long long o = ((long long)blockIdx.x * blockDim.x + threadIdx.x) / 32; o < half; o += per) {
        double dl = 0.0;
        int v = 0;
        if (o < ne) {
            v = ent_v[o];
            const unsigned m = ent_m[o];
            if (j < __popc(m)) {
                const long long k = ((long long)v << b.ks) + bc_nth_bit(m, j);
                dl = b.del[k];
                b.sig[k] = (1.0 + dl) / b.sig[k];
            }
        }
        for (int off = 16; off > 0; off >>= 1) dl += __shfl_xor(dl, off);
        if (o < ne && j == 0) bc[v] += dl;  // one entry per vertex per level
    }
    for (long long base = (long long)blockIdx.x * blockDim.x; base < nn; base += (long long)gridDim.x * blockDim.x) {
        const long long o = base + threadIdx.x;  // the trip count is uniform over the workgroup
        const long long k = o < nn ? bc_nchunks(b, nxt_v[o], nxt_m[o]) : 0;
        const long long first = bc_reserve(k, ctot);
        if (o < nn) cst[o] = first;
        bc_own(first, k, (int)o, owner, cap, err);
    }
}

__global__ void k_bc_to_float(const double *bc, int n, float *out) {
    for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (long long)gridDim.x * blockDim.x)
        out[i] = (float)bc[i];
}

// expansion workgroups per CU (8: +2 % per call, 4: +26 %)
constexpr int BC_EXPAND_WGS = 16;
static int bc_grid(long long work, int cap) {
    long long g = (work + 255) / 256;
    return (int)(g < 1 ? 1 : (g > cap ? cap : g));
}

hipError_t launch_bc_reset(const BcDev &b, hipStream_t s) {
    hipLaunchKernelGGL(k_bc_reset, dim3(bc_grid((long long)b.n << b.ks, 8192)), dim3(256), 0, s, b);
    return hipGetLastError();
}
hipError_t launch_bc_sources(const BcDev &b, const int *srcs, int nsrc, hipStream_t s) {
    hipLaunchKernelGGL(k_bc_sources, dim3(1), dim3(64), 0, s, b, srcs, nsrc);
    return hipGetLastError();
}
hipError_t launch_bc_compact(const BcDev &b, int *ent_v, unsigned *ent_m, int2 *lv, int d, long long *cst,
                             unsigned long long *ctot, int *owner, long long cap, int *err, hipStream_t s) {
    hipLaunchKernelGGL(k_bc_compact, dim3(bc_grid(b.n, 4096)), dim3(256), 0, s, b, ent_v, ent_m, lv, d, cst, ctot, owner,
                       cap, err);
    return hipGetLastError();
}
hipError_t launch_bc_expand(const BcDev &b, bool fwd, const int *ent_v, const unsigned *ent_m, int2 *lv,
                            const long long *cst, const int *owner, const unsigned long long *ctot, long long cap,
                            int d, int num_cus, hipStream_t s) {
    const int grid = num_cus * BC_EXPAND_WGS;  // grid-stride over the chunks (their count is on the device)
    if (fwd)
        hipLaunchKernelGGL(k_bc_expand<true>, dim3(grid), dim3(256), 0, s, b, ent_v, ent_m, lv, cst, owner, ctot, cap, d);
    else
        hipLaunchKernelGGL(k_bc_expand<false>, dim3(grid), dim3(256), 0, s, b, ent_v, ent_m, lv, cst, owner, ctot, cap,
                           d);
    return hipGetLastError();
}
hipError_t launch_bc_finish(const BcDev &b, const int *ent_v, const unsigned *ent_m, int ne, double *bc,
                            const int *nxt_v, const unsigned *nxt_m, int nn, long long *cst, unsigned long long *ctot,
                            int *owner, long long cap, int *err, hipStream_t s) {
    const long long work = std::max((long long)ne * 32, (long long)nn);
    hipLaunchKernelGGL(k_bc_finish, dim3(bc_grid(work, 4096)), dim3(256), 0, s, b, ent_v, ent_m, ne, bc, nxt_v, nxt_m, nn,
                       cst, ctot, owner, cap, err);
    return hipGetLastError();
}
hipError_t launch_bc_to_float(const double *bc, int n, float *out, hipStream_t s) {
    hipLaunchKernelGGL(k_bc_to_float, dim3(bc_grid(n, 4096)), dim3(256), 0, s, bc, n, out);
    return hipGetLastError();
}

}  // namespace np
