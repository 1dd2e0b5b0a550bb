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
// the source-packed SSSP does: sigma and delta (double: path counts stay exact integers up to
// 2^53).  No level is stored: st[v] = {seen, next} has one bit per source.  While level d is
// expanded, seen holds the sources that reached v on a level <= d, so an edge v -> w of an entry
// (v, mask of the sources with v on level d) is a predecessor edge for exactly mask & ~seen[w]: one
// 8-byte gather per edge answers for all sources, where a level per slot was a 128-byte row.  The
// forward sweep collects those bits in next[w]; the compaction turns them into level d + 1's
// entries, after the previous levels' ones, and adds them to seen.  The backward sweep replays the
// entries deepest level first and takes each finished level's bits out of seen again, so the same
// expression gives the same edges (an edge leads at most one level down).
//
// Work split: an entry's edges are cut into chunks of 64, one wavefront each, a lane per edge for
// the gather; the edges with a predecessor bit are then packed (LDS) and taken by groups of P'
// lanes, a lane per source slot, P' = popc(mask) rounded up to a power of two: the forward adds of
// one edge are one row segment, and the lanes of one source are lane, lane ^ P', ..., which the
// backward sweep sums with xor-shuffles.  A chunk is a 16-byte record {v, mask, first edge, edges},
// written by the compaction, so a wavefront starts with one load.  A row of one chunk is finished
// in its own sweep (factor and centrality, plain stores); longer rows add per chunk and are
// finished by the launch between two levels.  Two launches per level each way.
//
// 256 sources of R-MAT s16 (65,536 / 1 M), one call (before: a level per slot, a lane per (edge,
// source), two atomics on one line per wavefront of vertices): forward sweeps 2.26 ms (2.27: the
// float64 adds of the path counts, 4 lines per predecessor edge, at the 27 G lines/s that atomics
// reach), backward 0.72 (1.52), compactions 0.33 (0.90), finish 0.44 (0.77); the call 4.36 (5.93).
#include <hip/hip_runtime.h>
#include <algorithm>
#include "np_internal.h"

namespace np {

__device__ __forceinline__ int bc_lane() { return threadIdx.x & 63; }

constexpr int BC_CHUNK = 64;  // edges per chunk: one per lane
constexpr int BC_UNR = 4;     // edges a group of the backward sweep has in flight
constexpr int BC_WG = 1024;   // workgroup of the launches that reserve

// Every thread of the workgroup calls it: `cnt` entries (0 or 1) with k chunks in all are reserved
// on *ctl (entries in the low half, chunks in the high half); returns the thread's first of each.
// One atomic per workgroup: atomics on one line take 30 ns each, whoever issues them, and two per
// wavefront were most of a pass over the vertices.
__device__ __forceinline__ unsigned long long bc_reserve(unsigned cnt, unsigned k, unsigned long long *ctl) {
    __shared__ unsigned long long s_tot[BC_WG / 64];
    __shared__ unsigned long long s_base;
    const int lane = bc_lane(), wave = threadIdx.x >> 6;
    const unsigned long long mine = ((unsigned long long)k << 32) | cnt;
    unsigned long long incl = mine;
    for (int o = 1; o < 64; o <<= 1) {
        const unsigned long long t = __shfl_up(incl, o);
        if (lane >= o) incl += t;
    }
    if (lane == 63) s_tot[wave] = incl;
    __syncthreads();
    if (threadIdx.x == 0) {
        unsigned long long tot = 0;
        for (int i = 0; i < BC_WG / 64; ++i) {
            const unsigned long long t = s_tot[i];
            s_tot[i] = tot;
            tot += t;
        }
        s_base = tot ? atomicAdd(ctl, tot) : 0ull;
    }
    __syncthreads();
    const unsigned long long r = s_base + s_tot[wave] + incl - mine;
    __syncthreads();  // the next call writes both
    return r;
}

// The records of this lane's k chunks, `first` on (every lane of the wave calls it): the first by
// the lane itself, a longer row's others by the whole wave.  A level has at most m / 64 + ne chunks;
// a range past cap sets *err and nothing is written past it.
__device__ __forceinline__ void bc_chunks(long long first, int k, int v, unsigned m, int e0, int deg, int4 *rec,
                                          long long cap, int *err) {
    const int lane = bc_lane();
    if (k > 0) {
        if (first + k > cap) *err = 1;
        if (first < cap) rec[first] = int4{v, (int)m, e0, deg};
    }
    unsigned long long todo = __ballot(k > 1);
    while (todo) {
        const int l = __ffsll((long long)todo) - 1;
        todo &= todo - 1;
        const long long f = __shfl(first, l);
        const int kl = __shfl(k, l), vl = __shfl(v, l), el = __shfl(e0, l), dl = __shfl(deg, l);
        const int ml = __shfl((int)m, l);
        for (long long c = 1 + lane; c < kl && f + c < cap; c += 64)
            rec[f + c] = int4{vl, ml, el + (int)c * BC_CHUNK, dl - (int)c * BC_CHUNK};
    }
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
        b.sig[i] = 0.0;
        b.del[i] = 0.0;
        if (i < b.n) b.st[i] = uint2{0u, 0u};
    }
}

__global__ void k_bc_sources(BcDev b, const int *srcs, int nsrc) {
    const int j = threadIdx.x;
    if (blockIdx.x != 0 || j >= nsrc) return;
    const int s = srcs[j];
    b.sig[((long long)s << b.ks) + j] = 1.0;
    atomicOr(&b.st[s].y, 1u << j);
}

// Vertices with next bits -> the entries of level d (v, mask) at ent_v/ent_m + lv[d].first, counted
// with their chunks in lv[d].ctl, and the chunks' records.  Entries of all levels fit in n x
// sources: every (vertex, source) pair is in one level's entry and every entry holds at least one.
__global__ __launch_bounds__(BC_WG) void k_bc_compact(BcDev b, int *ent_v, unsigned *ent_m, BcLevel *lv, int4 *rec,
                                                      long long cap, int *err) {
    const long long E = lv->first;
    for (long long base = (long long)blockIdx.x * BC_WG; base < b.n; base += (long long)gridDim.x * BC_WG) {
        const long long v = base + threadIdx.x;  // the trip count is uniform over the workgroup
        const uint2 st = v < b.n ? b.st[v] : uint2{0u, 0u};
        const unsigned m = st.y;
        const int e0 = m ? b.row[v] : 0;
        const int deg = m ? b.row[v + 1] - e0 : 0;
        const int k = (int)(((long long)deg + BC_CHUNK - 1) / BC_CHUNK);
        const unsigned long long at = bc_reserve(m ? 1u : 0u, (unsigned)k, &lv->ctl);
        if (m) {
            b.st[v] = uint2{st.x | m, 0u};
            ent_v[E + (unsigned)at] = (int)v;
            ent_m[E + (unsigned)at] = m;
        }
        bc_chunks((long long)(at >> 32), k, (int)v, m, e0, deg, rec, cap, err);
    }
}

// One chunk per wavefront.  FWD: path counts and next bits of the level after lv's, and that
// level's first entry; else the dependencies of lv's level from the level after it.
template <bool FWD>
__global__ __launch_bounds__(256) void k_bc_expand(BcDev b, BcLevel *lv, const int4 *rec, long long cap, double *bc) {
    __shared__ int2 s_edge[4][BC_CHUNK];
    const unsigned long long ctl = lv->ctl;
    if (FWD && blockIdx.x == 0 && threadIdx.x == 0) lv[1].first = lv->first + (unsigned)ctl;
    const int lane = bc_lane();
    int2 *edge = s_edge[threadIdx.x >> 6];
    const long long tot = (long long)(ctl >> 32);
    const long long nchunks = tot < cap ? tot : cap;
    const long long nw = (long long)gridDim.x * (blockDim.x >> 6);
    for (long long c = (long long)blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6); c < nchunks; c += nw) {
        const int4 r = rec[c];  // {v, mask, first edge, edges of the row from there on}
        const int v = r.x;
        const unsigned m = (unsigned)r.y;
        int w = -1;
        unsigned pm = 0u;
        if (lane < r.w) {
            w = b.col[r.z + lane];
            const uint2 sw = b.st[w];
            pm = m & ~sw.x;
            // a stale next only costs an atomic that changes nothing
            if (FWD && (pm & ~sw.y)) atomicOr(&b.st[w].y, pm);
        }
        const int p = __popc(m);
        const int lp = p <= 1 ? 0 : 32 - __clz(p - 1);
        const int j = lane & ((1 << lp) - 1);
        const int src = j < p ? bc_nth_bit(m, j) : 0;
        const unsigned bit = j < p ? 1u << src : 0u;
        const long long own = ((long long)v << b.ks) + src;
        const double sv = j < p ? b.sig[own] : 0.0;
        const unsigned long long act = __ballot(pm != 0);
        const int cnt = __popcll(act);
        if (pm) edge[__popcll(act & ((1ull << lane) - 1))] = int2{w, (int)pm};
        wave_lds_order();
        const int step = 64 >> lp;  // groups in the wave
        if (FWD) {
            for (int i = lane >> lp; i < cnt; i += step) {
                const int2 e = edge[i];
                if ((unsigned)e.y & bit) atomicAdd(&b.sig[((long long)e.x << b.ks) + src], sv);
            }
        } else {
            // the next level's slots hold (1 + delta) / sigma
            double x = 0.0;
            for (int i = lane >> lp; i < cnt; i += step * BC_UNR) {
                double f[BC_UNR];
                bool on[BC_UNR];
#pragma unroll
                for (int k = 0; k < BC_UNR; ++k) {
                    const int ik = i + k * step;
                    const int2 e = edge[ik < cnt ? ik : i];
                    on[k] = ik < cnt && ((unsigned)e.y & bit);
                    f[k] = on[k] ? b.sig[((long long)e.x << b.ks) + src] : 0.0;
                }
                // not sv * 0 for the others: a path count past float64 is infinite
#pragma unroll
                for (int k = 0; k < BC_UNR; ++k) x += on[k] ? sv * f[k] : 0.0;
            }
            for (int off = 32; off >= (1 << lp); off >>= 1) x += __shfl_xor(x, off);
            const bool whole = r.w <= BC_CHUNK && r.z == b.row[v];  // the row's only chunk
            if (whole) {
                if (lane < p) b.sig[own] = (1.0 + x) / sv;
                double sum = lane < p ? x : 0.0;
                for (int off = 1; off < (1 << lp); off <<= 1) sum += __shfl_xor(sum, off);
                if (lane == 0 && sum != 0.0) bc[v] += sum;  // one entry per vertex per level
            } else if (lane < p && x != 0.0) {
                atomicAdd(&b.del[own], x);
            }
        }
        wave_lds_order();  // the next chunk's edges overwrite the list
    }
}

// Between two backward levels.  The finished level's ne entries (ent_v, ent_m) leave seen; those
// that the sweep has not finished (rows of several chunks, rows without edges, every row of the
// deepest level: `all`) are finished here: bc[v] += delta of v for every source of the entry, and
// the slot's sigma is replaced by (1 + delta) / sigma, the factor the level above needs from it.
// Each (vertex, source) slot is in exactly one level's entries, so it is transformed once.  Half a
// wavefront per entry, lane j on the j-th source of its mask.
// The next level's nn entries (nxt_v, nxt_m), replayed: their chunks, counted in lv->ctl.
__global__ __launch_bounds__(BC_WG) void k_bc_finish(BcDev b, const int *ent_v, const unsigned *ent_m, int ne, int all,
                                                     double *bc, const int *nxt_v, const unsigned *nxt_m, int nn,
                                                     BcLevel *lv, int4 *rec, long long cap, int *err) {
    const int j = threadIdx.x & 31;
    const long long per = (long long)gridDim.x * (BC_WG / 32);
    const long long half = ((long long)ne + 1) / 2 * 2;  // whole waves: both halves make the same trips
    for (long long o = ((long long)blockIdx.x * BC_WG + threadIdx.x) / 32; o < half; o += per) {
        double dl = 0.0;
        int v = 0;
        bool mine = false;
        if (o < ne) {
            v = ent_v[o];
            const unsigned m = ent_m[o];
            const int deg = b.row[v + 1] - b.row[v];
            mine = all || deg == 0 || deg > BC_CHUNK;
            if (j == 0) b.st[v].x &= ~m;  // one entry per vertex per level
            if (mine && j < __popc(m)) {
                const long long k = ((long long)v << b.ks) + bc_nth_bit(m, j);
                dl = b.del[k];
                b.sig[k] = (1.0 + dl) / b.sig[k];
            }
        }
        if (__ballot(mine) == 0) continue;
        for (int off = 16; off > 0; off >>= 1) dl += __shfl_xor(dl, off);
        if (mine && j == 0 && dl != 0.0) bc[v] += dl;
    }
    for (long long base = (long long)blockIdx.x * BC_WG; base < nn; base += (long long)gridDim.x * BC_WG) {
        const long long o = base + threadIdx.x;  // the trip count is uniform over the workgroup
        const int v = o < nn ? nxt_v[o] : 0;
        const unsigned m = o < nn ? nxt_m[o] : 0u;
        const int e0 = o < nn ? b.row[v] : 0;
        const int deg = o < nn ? b.row[v + 1] - e0 : 0;
        const int k = (int)(((long long)deg + BC_CHUNK - 1) / BC_CHUNK);
        const unsigned long long at = bc_reserve(0u, (unsigned)k, &lv->ctl);
        bc_chunks((long long)(at >> 32), k, v, m, e0, deg, rec, cap, err);
    }
}

__global__ void k_bc_to_float(const double *bc, int n, float *out) {
    for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (long long)gridDim.x * blockDim.x)
        out[i] = (float)bc[i];
}

// expansion workgroups per CU (8: +2 % per call, 4: +26 %)
constexpr int BC_EXPAND_WGS = 16;
static int bc_grid(long long work, int wg, int cap) {
    long long g = (work + wg - 1) / wg;
    return (int)(g < 1 ? 1 : (g > cap ? cap : g));
}

hipError_t launch_bc_reset(const BcDev &b, hipStream_t s) {
    hipLaunchKernelGGL(k_bc_reset, dim3(bc_grid((long long)b.n << b.ks, 256, 8192)), dim3(256), 0, s, b);
    return hipGetLastError();
}
hipError_t launch_bc_sources(const BcDev &b, const int *srcs, int nsrc, hipStream_t s) {
    hipLaunchKernelGGL(k_bc_sources, dim3(1), dim3(64), 0, s, b, srcs, nsrc);
    return hipGetLastError();
}
hipError_t launch_bc_compact(const BcDev &b, int *ent_v, unsigned *ent_m, BcLevel *lv, int4 *rec, long long cap,
                             int *err, hipStream_t s) {
    hipLaunchKernelGGL(k_bc_compact, dim3(bc_grid(b.n, BC_WG, 1024)), dim3(BC_WG), 0, s, b, ent_v, ent_m, lv, rec, cap,
                       err);
    return hipGetLastError();
}
hipError_t launch_bc_expand(const BcDev &b, bool fwd, BcLevel *lv, const int4 *rec, long long cap, double *bc,
                            int num_cus, hipStream_t s) {
    const int grid = num_cus * BC_EXPAND_WGS;  // grid-stride over the chunks (their count is on the device)
    if (fwd)
        hipLaunchKernelGGL(k_bc_expand<true>, dim3(grid), dim3(256), 0, s, b, lv, rec, cap, bc);
    else
        hipLaunchKernelGGL(k_bc_expand<false>, dim3(grid), dim3(256), 0, s, b, lv, rec, cap, bc);
    return hipGetLastError();
}
hipError_t launch_bc_finish(const BcDev &b, const int *ent_v, const unsigned *ent_m, int ne, bool all, double *bc,
                            const int *nxt_v, const unsigned *nxt_m, int nn, BcLevel *lv, int4 *rec, long long cap,
                            int *err, hipStream_t s) {
    const long long work = std::max((long long)ne * 32, (long long)nn);
    hipLaunchKernelGGL(k_bc_finish, dim3(bc_grid(work, BC_WG, 1024)), dim3(BC_WG), 0, s, b, ent_v, ent_m, ne, all ? 1 : 0,
                       bc, nxt_v, nxt_m, nn, lv, rec, cap, err);
    return hipGetLastError();
}
hipError_t launch_bc_to_float(const double *bc, int n, float *out, hipStream_t s) {
    hipLaunchKernelGGL(k_bc_to_float, dim3(bc_grid(n, 256, 4096)), dim3(256), 0, s, bc, n, out);
    return hipGetLastError();
}

}  // namespace np
