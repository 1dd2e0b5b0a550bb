// np_kernels.hip -- gfx950 kernels of the SSSP / recursive-BFS nested-parallelism path.
//
// The reference (apps/sssp/src/gpu/sssp_kernel.cu) expands each frontier vertex in a
// thread and hands vertices of out-degree >= THRESHOLD to child grids launched from
// the device, consolidated per warp (consolidate_warp_dp_kernel, :330-404), per block
// (consolidate_block_dp_kernel, :407-481) or per grid (consolidate_grid_dp_kernel,
// :484-541).  HIP has no device-side launch, so here the frontier is kept as a queue
// segmented by out-degree class and every scope of consolidation is a mapping of those
// segments onto workers of the same launch:
//   lane bin       64 frontier vertices per wavefront, their edges spread evenly over the
//                  64 lanes (prefix sum of degrees + owner search), coalesced CSR reads
//   wavefront bin  one vertex per 64-lane wavefront (the reference's 64-thread child block)
//   workgroup bin  one vertex per 256-thread workgroup (block-level consolidation)
//   grid bin       a vertex split into 2048-edge chunks spread over every wavefront of
//                  the grid (grid-level consolidation)
// The relaxation is the reference's, bit for bit (sssp_kernel.cu:46-52):
//   alt = dist[u] + w;  if (dist[v] > alt) atomicMin(&dist[v], alt)  -- int32.
// A vertex whose distance improved is flagged in an update bitmap (the reference's
// update[] byte array, one bit per vertex) and, for the next iteration, either compacted
// from the bitmap (scan frontier, unorder_generateQueue_kernel :648-658) or appended by
// the relaxing wavefront (push frontier).  Batches of up to 32 sources of one graph run
// the same bins over (vertex, pending sources) work items ("source-packed batch" below).
#include <hip/hip_runtime.h>
#include "np_internal.h"

namespace np {

#define NP_AGENT __HIP_MEMORY_SCOPE_AGENT
static constexpr int WG = 256;
static constexpr int WAVES = WG / 64;
static constexpr unsigned long long SPIN_LIMIT = 1ull << 24;

// ------------------------------------------------------------------------------------
// small helpers
// ------------------------------------------------------------------------------------
// threadIdx.x for one phase of a persistent kernel.  What a phase derives from it is the same in every
// iteration, so the compiler would compute it once, before the loop, and hold it in registers through
// all other phases; behind this it is computed again where it is used.  k_persistent 130 (with the
// small-frontier path 150) -> 93 (116) VGPRs, 3 -> 5 (4) workgroups per CU; k_pk_persistent without a
// window 156 -> 124, 3 -> 4; k_pk_expand (64 at most) no longer spills.  A limit on the registers alone (waves_per_eu)
// gave the same count and lost it again: every wavefront had fewer loads in flight.
__device__ __forceinline__ int phase_tid() {
    int t = threadIdx.x;
    asm volatile("" : "+v"(t));
    return t;
}
__device__ __forceinline__ int lane_id() { return phase_tid() & 63; }
__device__ __forceinline__ unsigned long long lanes_below(int lane) { return (1ull << lane) - 1; }

// Data that one workgroup writes and another reads inside a persistent launch (queue
// entries, bitmap words, counters, distances) only moves through device-coherent
// accesses: relaxed agent-scope atomics, loads and stores (sc1 on gfx950: they bypass
// the per-CU cache and the non-coherent L2 state of the other XCDs).  The grid barrier
// then needs no L2 writeback or invalidate, which would also evict the read-only CSR.
__device__ __forceinline__ int ld_coherent(const int *p) {
    return __hip_atomic_load(const_cast<int *>(p), __ATOMIC_RELAXED, NP_AGENT);
}
__device__ __forceinline__ unsigned ld_coherent_u(const unsigned *p) {
    return __hip_atomic_load(const_cast<unsigned *>(p), __ATOMIC_RELAXED, NP_AGENT);
}
__device__ __forceinline__ void st_coherent(int *p, int v) {
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, NP_AGENT);
}
__device__ __forceinline__ void st_coherent_b(unsigned char *p, unsigned char v) {
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, NP_AGENT);
}
__device__ __forceinline__ void st_coherent_u(unsigned *p, unsigned v) {
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, NP_AGENT);
}

#ifndef NP_BOUNDS_CHECK
#define NP_BOUNDS_CHECK 0
#endif
// Bounds-checked build (NP_BOUNDS_CHECK=1, libnpsssp_bounds.so): every write into a frontier
// queue, its source masks or a scheme's delayed buffer checks its index against the segment it
// belongs to, [lo, hi); an index outside is not written and the solve fails with NP_ERR_BOUNDS.
// The normal build compiles the check out.
__device__ __forceinline__ bool seg_ok(Ctrl *ctrl, long long idx, long long lo, long long hi) {
#if NP_BOUNDS_CHECK
    if (idx >= lo && idx < hi) return true;
    atomicCAS(&ctrl->error, 0, (int)NP_ERR_BOUNDS);
    return false;
#else
    (void)ctrl; (void)idx; (void)lo; (void)hi;
    return true;
#endif
}

__device__ __forceinline__ int wave_incl_scan(int x) {
    const int lane = lane_id();
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        int t = __shfl_up(x, o);
        if (lane >= o) x += t;
    }
    return x;
}

template <bool BATCH>
__device__ __forceinline__ void decode(const DevState &st, int slot, int &B, int &VB) {
    if (BATCH) {
        int i = st.lut[slot >> LUT_SHIFT];
        int2 d = st.inst[i];
        B = d.x; VB = d.y;
    } else {
        B = 0; VB = 0;
    }
}

// Grid-wide barrier of a cooperative launch.  Every wave first waits for its own
// outstanding memory operations (s_waitcnt 0: its coherent stores and atomics have
// completed), the workgroup meets at s_barrier, then one lane arrives.  Arrivals form a
// two-level tree of cumulative 64-bit counters (no reset): workgroup b counts on leaf
// b % 32 (each on its own cache line), the last arrival of a leaf counts on the root,
// and every workgroup spins on the root with relaxed coherent loads.  The spin is
// bounded: on expiry the block raises NP_ERR_TIMEOUT and every block leaves its loop at
// the next barrier, so the grid always drains.
__device__ bool grid_sync(Ctrl *ctrl, unsigned nblocks, unsigned long long &gen) {
    __shared__ int s_ok;
    stores_done();
    __syncthreads();
    if (threadIdx.x == 0) {
        gen += 1;
        const unsigned nleaves = nblocks < (unsigned)BAR_LEAVES ? nblocks : (unsigned)BAR_LEAVES;
        const unsigned l = blockIdx.x % nleaves;
        const unsigned long long lsize = nblocks / nleaves + (l < nblocks % nleaves ? 1u : 0u);
        unsigned long long la =
            __hip_atomic_fetch_add(&ctrl->leaf[l].n, 1ull, __ATOMIC_RELAXED, NP_AGENT) + 1ull;
        const unsigned long long target = gen * (unsigned long long)nleaves;
        unsigned long long arrived = 0;
        if (la == gen * lsize)
            arrived = __hip_atomic_fetch_add(&ctrl->bar, 1ull, __ATOMIC_RELAXED, NP_AGENT) + 1ull;
        int ok = 1;
        if (arrived < target) {
            unsigned long long spins = 0;
            while (__hip_atomic_load(&ctrl->bar, __ATOMIC_RELAXED, NP_AGENT) < target) {
                __builtin_amdgcn_s_sleep(1);
                if (++spins > SPIN_LIMIT) { ok = 0; break; }
                if ((spins & 1023) == 0 && __hip_atomic_load(&ctrl->error, __ATOMIC_RELAXED, NP_AGENT)) {
                    ok = 0; break;
                }
            }
        }
        if (!ok) {
            int expected = 0;
            __hip_atomic_compare_exchange_strong(&ctrl->error, &expected, (int)NP_ERR_TIMEOUT,
                                                 __ATOMIC_RELAXED, __ATOMIC_RELAXED, NP_AGENT);
        }
        if (__hip_atomic_load(&ctrl->error, __ATOMIC_RELAXED, NP_AGENT)) ok = 0;
        s_ok = ok;
    }
    __syncthreads();
    return s_ok != 0;
}

// ------------------------------------------------------------------------------------
// relaxation
// ------------------------------------------------------------------------------------
struct PushCtx {
    unsigned *bm_next;  // bitmap receiving "improved" marks
    unsigned *bm_cur;   // push: bitmap of the frontier being consumed (cleared here)
    int *cnt_next;      // push: class counters of the next frontier
    int *q_next;        // push: next frontier queue
};

// Tail of one relaxation after the cheap check (alt < dist[tslot]) passed: the atomicMin of the
// reference, issued without a return value, and the update mark.  Marking on the check alone
// marks exactly the slots the atomic's old value would: when a concurrent atomicMin has already
// stored less than alt, that writer passed its own check in this same launch and marks the slot
// itself (every earlier store is visible to the check).  With a scanned frontier the mark is one
// more atomic without a return, so no lane waits on either; the compaction drops vertices without
// out-edges.  Pushing relaxers need the class of the slot and the bit's old value to append it
// once.  Returns true when the caller must append tslot (push only).
template <bool PUSH>
__device__ __forceinline__ bool relax_tail(const DevState &st, const PushCtx &pc, int tslot,
                                           int alt, int &c_out) {
    atomicMin(&st.dist[tslot], alt);
    const unsigned bit = 1u << (tslot & 31);
    if (!PUSH) {
        atomicOr(&pc.bm_next[tslot >> 5], bit);
        return false;
    }
    const int c = st.cls[tslot];
    if (c == 0) return false;  // no out-edges: nothing to propagate
    const unsigned prev = atomicOr(&pc.bm_next[tslot >> 5], bit);
    c_out = c;
    return (prev & bit) == 0;
}

// Wavefront-aggregated append into the class-segmented next frontier: one counter
// atomic per (wavefront, class) group.
__device__ __forceinline__ void push_wave(const DevState &st, const PushCtx &pc, bool want,
                                          int slot, int c) {
    unsigned long long mask = __ballot(want);
    while (mask) {
        int leader = __ffsll((long long)mask) - 1;
        int cl = __shfl(c, leader);
        unsigned long long same = __ballot(want && c == cl);
        int base = 0;
        if (lane_id() == leader) base = atomicAdd(&pc.cnt_next[cl], __popcll(same));
        base = __shfl(base, leader);
        if (want && c == cl) {
            int pos = base + __popcll(same & __lanemask_lt());
            if (seg_ok(st.ctrl, (long long)st.seg_off[cl] + pos, st.seg_off[cl], st.seg_off[cl + 1]))
                st_coherent(pc.q_next + st.seg_off[cl] + pos, slot);
            want = false;
        }
        mask &= ~same;
    }
}

constexpr int UNR = 4;

// GUARD: lanes past the end of their range issue no loads (per-iteration kernels, eight
// waves per SIMD: enough loads in flight already); otherwise every load is issued and only
// the atomics are guarded, so the unrolled items' loads are all in flight together
// (persistent kernels, four to five waves per SIMD).  Dead lanes then read a valid address.

// Edges [e0, e1) of one vertex (slot base B, distance du), worker t of `stride`.
// The loop trip count is uniform across the wavefront.
template <bool UNIT, bool PUSH, bool GUARD>
__device__ __forceinline__ void relax_range(const DevState &st, const PushCtx &pc, int B, int e0,
                                            int e1, int du, int t, int stride) {
    for (int base = e0; base < e1; base += UNR * stride) {
        int tv[UNR], alt[UNR], cur[UNR];
        bool ok[UNR];
#pragma unroll
        for (int k = 0; k < UNR; ++k) {
            int e = base + t + k * stride;
            ok[k] = e < e1;
            int ec = ok[k] ? e : e0;
            tv[k] = B + st.col[ec];
            alt[k] = du + (UNIT ? 1 : st.w[ec]);
        }
#pragma unroll
        for (int k = 0; k < UNR; ++k) cur[k] = (GUARD && !ok[k]) ? 0 : ld_coherent(st.dist + tv[k]);
#pragma unroll
        for (int k = 0; k < UNR; ++k) {
            bool want = false;
            int c = 0;
            if (ok[k] && alt[k] < cur[k]) want = relax_tail<PUSH>(st, pc, tv[k], alt[k], c);
            if (PUSH) push_wave(st, pc, want, tv[k], c);
        }
    }
}

// Lane bin: 64 frontier vertices (queue[qidx .. qidx+nvalid)), edges balanced over lanes.
template <bool BATCH, bool UNIT, bool PUSH, bool GUARD>
__device__ __forceinline__ void lane_tile(const DevState &st, const PushCtx &pc, const int *q,
                                          long long qidx, int nvalid) {
    const int lane = lane_id();
    const bool valid = lane < nvalid;
    int slot = valid ? ld_coherent(q + qidx + lane) : 0;
    int B = 0, VB = 0, s = 0, d = 0, du = 0;
    if (valid) {
        decode<BATCH>(st, slot, B, VB);
        int v = slot - B;
        s = st.row[VB + v];
        d = st.row[VB + v + 1] - s;
        du = ld_coherent(st.dist + slot);
        if (PUSH) st_coherent_u(pc.bm_cur + (slot >> 5), 0u);
    }
    const int incl = wave_incl_scan(d);
    const int total = __shfl(incl, 63);
    const int excl = incl - d;
    if (total == 0) return;
    // First edge of the tile (owner of index 0 = first lane with d > 0) and that lane's slot
    // base: the address the lanes whose index runs past the end read.  Edge and base come
    // from the same lane, so the target slot lies inside that lane's instance.
    const int first_lane = __ffsll((long long)__ballot(d > 0)) - 1;
    const int e_safe = __shfl(s, first_lane);
    const int b_safe = BATCH ? __shfl(B, first_lane) : 0;
    for (int base = 0; base < total; base += UNR * 64) {
        int tv[UNR], alt[UNR], cur[UNR];
        bool ok[UNR];
#pragma unroll
        for (int k = 0; k < UNR; ++k) {
            const int kk = base + lane + k * 64;
            ok[k] = kk < total;
            // owner: the last lane whose exclusive offset is <= kk
            int o = 0;
#pragma unroll
            for (int step = 32; step > 0; step >>= 1) {
                int t = __shfl(excl, o + step);
                if (t <= kk) o += step;
            }
            const int e = __shfl(s, o) + (kk - __shfl(excl, o));
            const int ou = __shfl(du, o);
            const int ob = BATCH ? __shfl(B, o) : 0;
            const int ec = ok[k] ? e : e_safe;
            tv[k] = (ok[k] ? ob : b_safe) + st.col[ec];
            alt[k] = ou + (UNIT ? 1 : st.w[ec]);
        }
#pragma unroll
        for (int k = 0; k < UNR; ++k) cur[k] = (GUARD && !ok[k]) ? 0 : ld_coherent(st.dist + tv[k]);
#pragma unroll
        for (int k = 0; k < UNR; ++k) {
            bool want = false;
            int c = 0;
            if (ok[k] && alt[k] < cur[k]) want = relax_tail<PUSH>(st, pc, tv[k], alt[k], c);
            if (PUSH) push_wave(st, pc, want, tv[k], c);
        }
    }
}

// Shortest rows: a lane per queued vertex walks its edges, UNR loads in flight.  No owner search;
// the rows of neighbouring vertices share cache lines.  Not for pushed distances: the vertices would be
// appended in an order that keeps neighbours apart, and the next frontier's reads with them (grid 3200^2
// 36.4 -> 38.2 ms, 2048^2 16.1 -> 16.8); levels settle at once and gain (grid 1200^2 1.81 -> 1.72).
template <bool BATCH, bool UNIT, bool PUSH>
__device__ __forceinline__ void lane_serial(const DevState &st, const PushCtx &pc, const int *q, long long qidx,
                                            int nvalid) {
    const int lane = lane_id();
    int B = 0, VB = 0, s = 0, d = 0, du = 0;
    if (lane < nvalid) {
        const int slot = ld_coherent(q + qidx + lane);
        decode<BATCH>(st, slot, B, VB);
        const int v = slot - B;
        s = st.row[VB + v];
        d = st.row[VB + v + 1] - s;
        du = ld_coherent(st.dist + slot);
        if (PUSH) st_coherent_u(pc.bm_cur + (slot >> 5), 0u);
    }
    for (int i = 0; __ballot(i < d) != 0; i += UNR) {
        int tv[UNR], alt[UNR], cur[UNR];
#pragma unroll
        for (int k = 0; k < UNR; ++k) {
            const bool ok = i + k < d;
            tv[k] = ok ? B + st.col[s + i + k] : 0;
            alt[k] = ok ? du + (UNIT ? 1 : st.w[s + i + k]) : 0;
        }
#pragma unroll
        for (int k = 0; k < UNR; ++k) cur[k] = i + k < d ? ld_coherent(st.dist + tv[k]) : 0;
#pragma unroll
        for (int k = 0; k < UNR; ++k) {
            bool want = false;
            int c = 0;
            if (alt[k] < cur[k]) want = relax_tail<PUSH>(st, pc, tv[k], alt[k], c);
            if (PUSH) push_wave(st, pc, want, tv[k], c);
        }
    }
}

// ------------------------------------------------------------------------------------
// one expansion (all threads of every workgroup call it)
// ------------------------------------------------------------------------------------
// Per-workgroup item tables: exclusive prefix, by class, of the work items of each scope.
struct ItemTables {
    long long pre[4][NCLS + 1];  // 0 grid chunks, 1 workgroup items, 2 wavefront items, 3 lane tiles
    int cnt[NCLS];
    int seg[NCLS];
    int tv;                      // single source: vertices per lane tile
};

__device__ __forceinline__ int find_class(const long long *pre, long long idx) {
    int c = 0;
#pragma unroll
    for (int step = 16; step > 0; step >>= 1)
        if (c + step <= NCLS - 1 && pre[c + step] <= idx) c += step;
    return c;
}

// Filtered packed expansions (pk_edge_tile): vertices of class c per tile, about 768 edges, for the
// classes below PK_TILE_CLS.
__device__ __forceinline__ int pk_tile_vertices(int c) { return c <= 4 ? 64 : 1024 >> c; }
constexpr int PK_TILE_CLS = 11;

// Single-source work items.
// Lane bin: vertices of degree below 2^SERIAL_CLS are walked one per lane; longer rows go to tiles
// whose edges are spread over the lanes, of as many vertices (8 to 64) as give every wavefront a
// tile (64 always: the widest ER 65,536 / 1 M frontier, 43 K vertices, filled 670 of 4,096
// wavefronts; the tables, tiles and serial rows together: 0.82 -> 0.63 ms).
// Workgroup bin: a row of more than 2^WG_CHUNK_SHIFT edges goes to several workgroups in chunks; one
// workgroup on a hub of 160 K edges was the iteration's tail (R-MAT s22, block level, one solve: 3.81
// -> 3.18 ms).  Shorter chunks make the block level itself 3 to 7 % faster still (2^14 3.09, 2^13
// 3.02, 2^12 2.96 ms), but it is the reference's fixed heuristic, one workgroup per heavy vertex,
// that the learned schedule is trained against and measured by (R-MAT s20, learned over block level:
// 1.54 without chunks, 1.42 with 2^15, 1.29 with 2^13), so only the longest rows are cut.
constexpr int SERIAL_CLS = 3;
constexpr int WG_CHUNK_SHIFT = 15;
__device__ __forceinline__ int wg_chunks(int c) { return c > WG_CHUNK_SHIFT ? 1 << (c - WG_CHUNK_SHIFT) : 1; }

enum TableKind { TABLES_SINGLE = 0, TABLES_PACKED = 1, TABLES_FILTERED = 2 };

// The first wavefront builds the tables from the frontier's class counts (already in tb.cnt),
// lane c for class c; nwaves = wavefronts of the expansion.
__device__ __forceinline__ void build_tables(ItemTables &tb, const Cfg &cfg, TableKind kind, long long nwaves) {
    const int c = lane_id();
    const long long n = c >= 1 && c < NCLS ? tb.cnt[c] : 0;
    int tv = 64;
    if (kind == TABLES_SINGLE) {
        long long lanes = c > SERIAL_CLS && c < cfg.b1 ? n : 0;
#pragma unroll
        for (int o = 16; o > 0; o >>= 1) lanes += __shfl_xor(lanes, o);
        lanes = __shfl(lanes, 0);
        while (tv > 8 && lanes <= (tv >> 1) * nwaves) tv >>= 1;
        if (c == 0) tb.tv = tv;
        if (c <= SERIAL_CLS) tv = 64;
    } else if (kind == TABLES_FILTERED) {
        tv = c < PK_TILE_CLS ? pk_tile_vertices(c) : 1;
    }
    long long item[4];
    item[0] = c >= cfg.b3 ? n * grid_chunks(c & 31) : 0;
    item[1] = c >= cfg.b2 && c < cfg.b3 ? (kind == TABLES_SINGLE ? n * wg_chunks(c & 31) : n) : 0;
    item[2] = c >= cfg.b1 && c < cfg.b2 ? n : 0;
    item[3] = c < cfg.b1 ? (n + tv - 1) / tv : 0;
#pragma unroll
    for (int t = 0; t < 4; ++t) {
        long long x = item[t];
#pragma unroll
        for (int o = 1; o < 32; o <<= 1) {
            const long long y = __shfl_up(x, o);
            if (c >= o) x += y;
        }
        if (c < NCLS) tb.pre[t][c] = x - item[t];
        if (c == NCLS - 1) tb.pre[t][NCLS] = x;
    }
}

// Vertices of a frontier from its class counts (the first wavefront; the result in every lane).
__device__ __forceinline__ long long frontier_size(const int *cnt) {
    const int c = lane_id();
    long long x = c >= 1 && c < NCLS ? cnt[c] : 0;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) x += __shfl_xor(x, o);
    return x;
}

template <bool BATCH, bool UNIT, bool PUSH, bool GUARD>
__device__ void expansion(const DevState &st, const PushCtx &pc, const int *q, ItemTables &tb) {
    const long long G = tb.pre[0][NCLS], K = tb.pre[1][NCLS], W = tb.pre[2][NCLS],
                    T = tb.pre[3][NCLS];
    const int tid = phase_tid(), lane = tid & 63;
    // workgroup items: the whole workgroup strides one vertex's edges
    for (long long k = blockIdx.x; k < K; k += gridDim.x) {
        int c = find_class(tb.pre[1], k);
        long long r = k - tb.pre[1][c];
        int sh = c > WG_CHUNK_SHIFT ? c - WG_CHUNK_SHIFT : 0;
        int j = (int)(r & ((1ll << sh) - 1));
        int slot = ld_coherent(q + tb.seg[c] + (r >> sh));
        int B, VB;
        decode<BATCH>(st, slot, B, VB);
        int v = slot - B;
        int s = st.row[VB + v], e = st.row[VB + v + 1];
        int du = ld_coherent(st.dist + slot);
        if (PUSH && j == 0 && tid == 0) st_coherent_u(pc.bm_cur + (slot >> 5), 0u);
        if (j > (e - s - 1) >> WG_CHUNK_SHIFT) continue;  // a class's rows have half to all of its chunks
        int e0 = s + (j << WG_CHUNK_SHIFT);
        int e1 = e - e0 > (1 << WG_CHUNK_SHIFT) ? e0 + (1 << WG_CHUNK_SHIFT) : e;
        relax_range<UNIT, PUSH, GUARD>(st, pc, B, e0, e1, du, tid, WG);
    }
    // wavefront-granular items: grid chunks, wavefront items, lane tiles, round-robin
    const long long NW = (long long)gridDim.x * WAVES;
    const long long gw = (long long)blockIdx.x * WAVES + (tid >> 6);
    const long long U = G + W + T;
    for (long long u = gw; u < U; u += NW) {
        if (u < G) {
            int c = find_class(tb.pre[0], u);
            long long r = u - tb.pre[0][c];
            int sh = c > GRID_CHUNK_SHIFT ? c - GRID_CHUNK_SHIFT : 0;
            long long qi = tb.seg[c] + (r >> sh);
            int j = (int)(r & ((1ll << sh) - 1));
            int slot = ld_coherent(q + qi);
            int B, VB;
            decode<BATCH>(st, slot, B, VB);
            int v = slot - B;
            int s = st.row[VB + v], e = st.row[VB + v + 1];
            int e0 = s + (j << GRID_CHUNK_SHIFT);
            int e1 = e0 + (1 << GRID_CHUNK_SHIFT);
            if (e1 > e) e1 = e;
            if (PUSH && j == 0 && lane == 0) st_coherent_u(pc.bm_cur + (slot >> 5), 0u);
            if (e0 < e1) {
                int du = ld_coherent(st.dist + slot);
                relax_range<UNIT, PUSH, GUARD>(st, pc, B, e0, e1, du, lane, 64);
            }
        } else if (u < G + W) {
            long long i = u - G;
            int c = find_class(tb.pre[2], i);
            long long qi = tb.seg[c] + (i - tb.pre[2][c]);
            int slot = ld_coherent(q + qi);
            int B, VB;
            decode<BATCH>(st, slot, B, VB);
            int v = slot - B;
            int e0 = st.row[VB + v], e1 = st.row[VB + v + 1];
            int du = ld_coherent(st.dist + slot);
            if (PUSH && lane == 0) st_coherent_u(pc.bm_cur + (slot >> 5), 0u);
            relax_range<UNIT, PUSH, GUARD>(st, pc, B, e0, e1, du, lane, 64);
        } else {
            long long t = u - G - W;
            int c = find_class(tb.pre[3], t);
            long long ti = t - tb.pre[3][c];
            const int tv = c <= SERIAL_CLS ? 64 : tb.tv;
            long long first = ti * tv;
            int nvalid = (int)((long long)tb.cnt[c] - first < tv ? (long long)tb.cnt[c] - first : tv);
            if ((UNIT || !PUSH) && c <= SERIAL_CLS) lane_serial<BATCH, UNIT, PUSH>(st, pc, q, tb.seg[c] + first, nvalid);
            else lane_tile<BATCH, UNIT, PUSH, GUARD>(st, pc, q, tb.seg[c] + first, nvalid);
        }
    }
}

// ------------------------------------------------------------------------------------
// compaction (scan frontier): update bitmap -> class-segmented queue
// ------------------------------------------------------------------------------------
// With a priority window (T < INT_MAX) only flagged vertices with dist < T are queued and
// unflagged; the others keep their flag, and the pass adds how many were kept and the
// least distance among them to the pass's deferral sums (BarLeaf).  T = INT_MAX queues every flag.
constexpr int NO_WINDOW = 0x7FFFFFFF;

// The waves' class counters of this tile -> global reservation: s_wc[w][c] becomes wave w's first
// place of class c, so that a wave's vertices stay together in the queue.
__device__ __forceinline__ void reserve_classes(int (*s_wc)[NCLS], int *cnt_out) {
    __syncthreads();
    if (threadIdx.x < NCLS) {
        int k = 0;
        for (int w = 0; w < WAVES; ++w) k += s_wc[w][threadIdx.x];
        int at = k ? atomicAdd(&cnt_out[threadIdx.x], k) : 0;
        for (int w = 0; w < WAVES; ++w) {
            const int t = s_wc[w][threadIdx.x];
            s_wc[w][threadIdx.x] = at;
            at += t;
        }
    }
    __syncthreads();
}

// Deferred-pair statistics of the workgroup -> its line's sums of the pass.  One line for all took
// turns for longer than the pass: 2,048 workgroups, 0.12 ms (32 sources of a 2048^2 grid).
__device__ __forceinline__ void flush_deferred(Ctrl *ctrl, int slot, int my_dc, int my_dm, int *s_dc, int *s_dm) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        my_dc += __shfl_xor(my_dc, o);
        const int x = __shfl_xor(my_dm, o);
        my_dm = x < my_dm ? x : my_dm;
    }
    if (lane_id() == 0 && my_dc) { atomicAdd(s_dc, my_dc); atomicMin(s_dm, my_dm); }
    __syncthreads();
    if (threadIdx.x == 0 && *s_dc) {
        BarLeaf &l = ctrl->leaf[blockIdx.x % BAR_LEAVES];
        atomicAdd(&l.dcnt[slot], *s_dc);
        atomicMin(&l.dmin[slot], *s_dm);
    }
}
// The sums of a pass over all lines (a whole wavefront; the result in every lane).
__device__ __forceinline__ void deferred_sums(const Ctrl *ctrl, int slot, int *cnt, int *least) {
    const BarLeaf &l = ctrl->leaf[lane_id() % BAR_LEAVES];
    int c = lane_id() < BAR_LEAVES ? ld_coherent(&l.dcnt[slot]) : 0;
    int m = ld_coherent(&l.dmin[slot]);
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        c += __shfl_xor(c, o);
        const int x = __shfl_xor(m, o);
        m = x < m ? x : m;
    }
    *cnt = c;
    *least = m;
}
// Clears a pass's sums (threads 0 .. BAR_LEAVES of one workgroup).
__device__ __forceinline__ void deferred_clear(Ctrl *ctrl, int slot) {
    if (threadIdx.x < BAR_LEAVES) {
        st_coherent(&ctrl->leaf[threadIdx.x].dcnt[slot], 0);
        st_coherent(&ctrl->leaf[threadIdx.x].dmin[slot], NO_WINDOW);
    }
}

// A wave loads up to 64 words at once and takes the nonzero ones two at a time, a lane per vertex,
// COMPACT_UNR pairs in flight (one fewer in the persistent kernel without the small-frontier path, which
// then fits 5 workgroups on a CU; grid 3200^2 on 3: 6.58 ms with 4 or 3, 6.72 with 2); the vertices to queue gather in LDS as (offset, class).  A thread
// per word, walking its bits, left all but n / 8192 workgroups idle and waited for every class: one
// solve on the persistent drive, ER 65,536 / 1 M 0.94 -> 0.82 ms, grid 2048^2 5.12 -> 4.13.
constexpr int COMPACT_UNR = 4;
// Words a wavefront takes at once, 8 to 64: about 512 workgroups get a tile, because every tile
// reserves its classes' queue slots on the same cache lines, where atomics take turns (a tile for
// each of 2,048 workgroups made the heaviest compactions of 4.2 M vertices 75 -> 95 us).  A windowed
// pack reads a row of distances per vertex: from 4 words on, and 1,024 workgroups where 512 would
// take more than 32 (persistent drive, 16 sources of ER 65,536 2.95 ms with 8, 1.97 with 4; 3 sources
// of a 2048^2 grid, window 8,000: 6.56 ms with 512, 6.21 with 1,024; of 1200^2, 22 words each, launches 5.94 and 6.23).
__host__ __device__ __forceinline__ int compact_words(long long nwords, int grid, bool windowed) {
    auto share = [&](long long most) {
        const long long waves = (grid < most ? grid : most) * WAVES;
        return (nwords + waves - 1) / waves;
    };
    long long w = share(512);
    if (windowed && w > 32) w = share(1024) > 32 ? share(1024) : 32;
    const long long least = windowed ? 4 : 8;
    return (int)(w < least ? least : w < 64 ? w : 64);
}
template <int UNROLL>
__device__ __forceinline__ void compaction_impl(Ctrl *ctrl, unsigned *bm, const unsigned char *cls, const int *seg_off,
                                                long long nwords, int *cnt_out, int *q_out, const int *dist,
                                                int T, int slot) {
    __shared__ unsigned short s_list[WAVES][64 * 32];
    __shared__ int s_lc[NCLS], s_lb[NCLS];
    __shared__ int s_dc, s_dm;
    static_assert(NCLS <= 32, "an entry holds 11 bits of offset and 5 of class");
    const int tid = phase_tid();
    if (tid == 0) { s_dc = 0; s_dm = NO_WINDOW; }
    int my_dc = 0, my_dm = NO_WINDOW;
    const int lane = tid & 63, half = lane & 31;
    unsigned short *list = s_list[tid >> 6];
    const int wt = compact_words(nwords, gridDim.x, false);
    const long long tile = (long long)WAVES * wt;
    for (long long wb = (long long)blockIdx.x * tile; wb < nwords; wb += (long long)gridDim.x * tile) {
        if (tid < NCLS) s_lc[tid] = 0;
        const long long w0 = wb + (tid >> 6) * wt;
        const unsigned word = lane < wt && w0 + lane < nwords ? ld_coherent_u(bm + w0 + lane) : 0u;
        unsigned long long nz = __ballot(word != 0);
        int n = 0;
        while (nz) {
            int idx[UNROLL], c[UNROLL], d[UNROLL];
            unsigned x[UNROLL];
#pragma unroll
            for (int k = 0; k < UNROLL; ++k) {
                const int ia = __ffsll((long long)nz) - 1;
                nz &= nz - 1;
                const int ib = __ffsll((long long)nz) - 1;
                nz &= nz - 1;
                idx[k] = lane < 32 ? ia : ib;  // -1: none left
                x[k] = __shfl(word, idx[k] < 0 ? 0 : idx[k]);
                if (idx[k] < 0) x[k] = 0u;
                c[k] = (x[k] >> half) & 1u ? (int)cls[(w0 + idx[k]) * 32 + half] : 0;
            }
            if (T != NO_WINDOW) {
#pragma unroll
                for (int k = 0; k < UNROLL; ++k)
                    d[k] = c[k] ? ld_coherent(dist + (w0 + idx[k]) * 32 + half) : 0;
            }
#pragma unroll
            for (int k = 0; k < UNROLL; ++k) {
                const bool defer = T != NO_WINDOW && c[k] && d[k] >= T;
                if (defer) { my_dc++; my_dm = d[k] < my_dm ? d[k] : my_dm; }
                const bool take = c[k] && !defer;  // no out-edges (class 0): dropped
                const unsigned long long m = __ballot(take), kept = __ballot(defer);
                if (take) list[n + __popcll(m & lanes_below(lane))] = (unsigned short)((c[k] << 11) | (idx[k] * 32 + half));
                n += __popcll(m);
                const unsigned nw = (unsigned)(kept >> (lane & 32));
                if (half == 0 && nw != x[k]) st_coherent_u(bm + w0 + idx[k], nw);
            }
        }
        if (!__syncthreads_or(n)) continue;  // s_lc is clear, nothing was counted
        for (int i = lane; i < n; i += 64) atomicAdd(&s_lc[list[i] >> 11], 1);
        __syncthreads();
        if (tid < NCLS) {
            const int k = s_lc[tid];
            s_lb[tid] = k ? seg_off[tid] + atomicAdd(&cnt_out[tid], k) : 0;
            s_lc[tid] = 0;
        }
        __syncthreads();
        for (int i = lane; i < n; i += 64) {
            const int e = list[i], c = e >> 11;
            const int at = s_lb[c] + atomicAdd(&s_lc[c], 1);
            if (seg_ok(ctrl, at, seg_off[c], seg_off[c + 1])) st_coherent(q_out + at, (int)(w0 * 32) + (e & 2047));
        }
        __syncthreads();
    }
    if (T != NO_WINDOW) flush_deferred(ctrl, slot, my_dc, my_dm, &s_dc, &s_dm);
}

// ------------------------------------------------------------------------------------
// schedule decision (all threads of a workgroup; the MLP is evaluated redundantly per
// workgroup so every workgroup reaches the same decision without another barrier)
// ------------------------------------------------------------------------------------
// features() by one wavefront: lane c holds class c's count, the sums are butterflies and lane i
// finishes feature i (one thread walking the classes took 0.9 us of every iteration).  Counts below
// 2^24 add without rounding, so the features are the host's but for the last bit of larger sums.
__device__ __forceinline__ void wave_features(const int *count, int it, int n, float *x) {
    const int c = lane_id();
    const float k = c >= 1 && c < NCLS ? (float)count[c] : 0.f;
    const int g = c <= 2 ? 0 : c <= 4 ? 1 : c <= 6 ? 2 : c <= 8 ? 3 : c <= 12 ? 4 : 5;
    float sum[8] = {k, c >= 1 && c < NCLS ? k * 0.75f * (float)(1u << c) : 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < 6; ++i) sum[2 + i] = g == i ? k : 0.f;
#pragma unroll
    for (int o = 1; o < 32; o <<= 1) {
#pragma unroll
        for (int i = 0; i < 8; ++i) sum[i] += __shfl_xor(sum[i], o);
    }
    const float tot = sum[0];
    float v = c == 8 ? (float)(it < 256 ? it : 256) / 64.f : 0.f;
#pragma unroll
    for (int i = 0; i < 6; ++i)
        if (c == 2 + i) v = tot > 0.f ? sum[2 + i] / tot : 0.f;
    if (c == 0 || c == 1 || c == 9) {
        const float y = c == 0 ? 1.f + tot : c == 1 ? 1.f + sum[1] : (float)(n > 1 ? n : 1);
        v = log2f(y) / (c == 0 ? 24.f : 32.f);
    }
    if (c < NP_MLP_NIN) x[c] = v;
}

// The MLP's decision, or the fixed schedule (level, klo, khi) when its output is unusable.
// Called with scalars, not the SchedDev: a struct passed by reference to a function that is not
// inlined is first stored to scratch memory by every caller.
__device__ __noinline__ Cfg decide_mlp(const float *mlp, int n_feat, int flevel, int fklo, int fkhi,
                                       const int *cnt, int it) {
    static_assert(WG == 256 && NP_MLP_NIN <= 16, "decide() maps 32 outputs x 8 parts onto the workgroup");
    __shared__ float s_x[NP_MLP_NIN], s_h1[32], s_h2[32], s_o[5];
    const Cfg fixed = make_cfg(flevel, fklo, fkhi);
    const float *W1 = mlp, *b1 = W1 + 32 * NP_MLP_NIN, *W2 = b1 + 32, *b2 = W2 + 32 * 32;
    const float *W3 = b2 + 32, *b3 = W3 + 5 * 32;
    // Thread t computes part p = t % 8 of output j = t / 8 of each layer; the 8 parts of an output
    // are adjacent lanes, summed with three shuffles.  Every weight is loaded before the first
    // layer (W2 and W3 rows as float4, thread t at float 4t: one coalesced 4 KB read), so the
    // forward pass waits for global memory once, not once per weight.
    const int t = threadIdx.x, j = t >> 3, p = t & 7;
    const float w1a = W1[j * NP_MLP_NIN + p];
    const float w1b = p + 8 < NP_MLP_NIN ? W1[j * NP_MLP_NIN + p + 8] : 0.f;
    const float4 w2 = *(const float4 *)(W2 + 4 * t);
    const float4 w3 = t < 40 ? *(const float4 *)(W3 + 4 * t) : make_float4(0.f, 0.f, 0.f, 0.f);
    const float b1j = b1[j], b2j = b2[j], b3j = t < 40 ? b3[j] : 0.f;
    if (t < 64) wave_features(cnt, it, n_feat, s_x);
    __syncthreads();
    float a = w1a * s_x[p] + (p + 8 < NP_MLP_NIN ? w1b * s_x[p + 8] : 0.f);
    a += __shfl_xor(a, 1);
    a += __shfl_xor(a, 2);
    a += __shfl_xor(a, 4);
    if (p == 0) s_h1[j] = a + b1j > 0.f ? a + b1j : 0.f;
    __syncthreads();
    a = w2.x * s_h1[4 * p] + w2.y * s_h1[4 * p + 1] + w2.z * s_h1[4 * p + 2] + w2.w * s_h1[4 * p + 3];
    a += __shfl_xor(a, 1);
    a += __shfl_xor(a, 2);
    a += __shfl_xor(a, 4);
    if (p == 0) s_h2[j] = a + b2j > 0.f ? a + b2j : 0.f;
    __syncthreads();
    a = w3.x * s_h2[4 * p] + w3.y * s_h2[4 * p + 1] + w3.z * s_h2[4 * p + 2] + w3.w * s_h2[4 * p + 3];
    a += __shfl_xor(a, 1);
    a += __shfl_xor(a, 2);
    a += __shfl_xor(a, 4);
    if (t < 40 && p == 0) s_o[j] = a + b3j;
    __syncthreads();
    float o0 = s_o[0], o1 = s_o[1], o2 = s_o[2], o3 = s_o[3], o4 = s_o[4];
    __syncthreads();
    if (!(isfinite(o0) && isfinite(o1) && isfinite(o2) && isfinite(o3) && isfinite(o4)) ||
        fabsf(o3) > 1e6f || fabsf(o4) > 1e6f)
        return fixed;  // fallback: the fixed-threshold heuristic
    int level = (o1 > o0) ? ((o2 > o1) ? 2 : 1) : ((o2 > o0) ? 2 : 0);
    return make_cfg(level, (int)rintf(o3), (int)rintf(o4));
}

__device__ __forceinline__ Cfg decide(const SchedDev &sp, const int *cnt, int it) {
    if (!sp.learned || !sp.mlp) return make_cfg(sp.level, sp.klo, sp.khi);
    return decide_mlp(sp.mlp, sp.n_feat, sp.level, sp.klo, sp.khi, cnt, it);
}

// The first wavefront records an iteration (lane c holds class c; t0 is lane 0's).
__device__ __forceinline__ void record_trace(const SchedDev &sp, int it, const Cfg &cfg, const int *cnt,
                                             long long t0, Ctrl *ctrl) {
    if (!sp.trace || it >= sp.trace_cap) return;
    np_trace_rec *r = sp.trace + it;
    const int lane = lane_id();
    long long pairs = lane < BAR_LEAVES ? __hip_atomic_load(&ctrl->leaf[lane].pairs, __ATOMIC_RELAXED, NP_AGENT) : 0;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) pairs += __shfl_xor(pairs, o);
    if (lane < NCLS) r->count[lane] = cnt[lane];
    if (lane == 0) {
        r->pairs = pairs;
        r->edges = __hip_atomic_load(&ctrl->edges_total, __ATOMIC_RELAXED, NP_AGENT);
        r->iteration = it;
        r->level = cfg.level;
        r->log2_t_lo = cfg.klo;
        r->log2_t_hi = cfg.khi;
        r->t_begin = t0;
        r->t_end = t0;
    }
}

// ------------------------------------------------------------------------------------
// small frontiers of the persistent drive
// ------------------------------------------------------------------------------------
// A frontier of a few hundred vertices costs a whole iteration's two grid barriers, a scan of the
// bitmap and the work tables (14-18 us) for a few microseconds of work, and road-like graphs start
// and end with dozens of them.  One workgroup runs such iterations alone, the frontier in LDS, while
// the others wait at the next grid barrier: about 4 us each (one solve, grid 512^2 1.20 -> 1.03 ms,
// 2048^2 3.88 -> 3.66; ER 65,536 / 1 M, with few small frontiers, 0.563 -> 0.552).  An improved vertex is appended once
// (the returned bitmap word decides), so when the frontier outgrows the limits the bitmap holds
// exactly the vertices pending, and the next compaction takes over.
constexpr int SOLO_V = 512;        // vertices of a solo frontier
constexpr int SOLO_E = 4096;       // edges of one
constexpr int SOLO_ITERS = 256;    // iterations per visit (the other workgroups' wait is bounded)

struct SoloBufs {
    int list[2][SOLO_V];
    int pre[SOLO_V + 1];  // exclusive prefix of the degrees
    int start[SOLO_V];    // first edge - prefix
    int base[SOLO_V];     // slot base of the vertex's instance
    int du[SOLO_V];
    int wsum[WAVES], live, next;
};

__device__ __forceinline__ bool solo_fits(const ItemTables &tb, int total) {
    if (total > SOLO_V) return false;
    const int c = threadIdx.x & 31;  // every half-wave for itself
    int e = c >= 1 && tb.cnt[c] ? (c >= 13 ? SOLO_E + 1 : tb.cnt[c] << c) : 0;
#pragma unroll
    for (int o = 16; o > 0; o >>= 1) e += __shfl_xor(e, o);
    return e <= SOLO_E;
}

// Iterations of the queued frontier (classes in tb) until it is empty or outgrows the limits, at
// most `most`; returns how many.  Called by one whole workgroup.
template <bool BATCH, bool UNIT>
__device__ __forceinline__ int solo_iterations(const DevState &st, const ItemTables &tb, const int *q, SoloBufs &sb,
                                               int total, int most) {
    const int t = phase_tid(), lane = t & 63, wave = t >> 6;
    unsigned *bm = st.bm[0];
    // the queue's class segments -> list[0]
    for (int i = t; i < total; i += WG) {
        int c = 1, k = i;
        while (k >= tb.cnt[c]) { k -= tb.cnt[c]; ++c; }
        sb.list[0][i] = ld_coherent(q + tb.seg[c] + k);
    }
    int n = total, iters = 0;
    long long sum = 0;
    for (;;) {
        __syncthreads();
        if (t == 0) { sb.next = 0; sb.live = 0; }
        const int *cur = sb.list[iters & 1];
        int *nxt = sb.list[(iters & 1) ^ 1];
        // vertices 2t, 2t + 1: flags of an appended vertex are cleared before it is expanded
        int d[2] = {0, 0}, s[2] = {0, 0};
        static_assert(SOLO_V == 2 * WG, "two vertices per thread");
#pragma unroll
        for (int k = 0; k < 2; ++k) {
            const int i = 2 * t + k;
            if (i >= n) continue;
            const int slot = cur[i];
            if (iters > 0) atomicAnd(&bm[slot >> 5], ~(1u << (slot & 31)));
            int B, VB;
            decode<BATCH>(st, slot, B, VB);
            s[k] = st.row[VB + slot - B];
            d[k] = st.row[VB + slot - B + 1] - s[k];
            sb.base[i] = B;
            sb.du[i] = ld_coherent(st.dist + slot);
        }
        __syncthreads();  // next and live are zero
        const unsigned long long m0 = __ballot(d[0] > 0), m1 = __ballot(d[1] > 0);
        const int incl = wave_incl_scan(d[0] + d[1]);
        if (lane == 63) {
            sb.wsum[wave] = incl;
            atomicAdd(&sb.live, __popcll(m0) + __popcll(m1));
        }
        stores_done();  // the cleared flags are in memory
        __syncthreads();
        int before = 0, edges = 0;
#pragma unroll
        for (int w = 0; w < WAVES; ++w) {
            before += w < wave ? sb.wsum[w] : 0;
            edges += sb.wsum[w];
        }
        const int x0 = before + incl - d[0] - d[1], x1 = x0 + d[0];
        if (2 * t < n) { sb.pre[2 * t] = x0; sb.start[2 * t] = s[0] - x0; }
        if (2 * t + 1 < n) { sb.pre[2 * t + 1] = x1; sb.start[2 * t + 1] = s[1] - x1; }
        const int live = sb.live;
        // empty, or a frontier that the grid should expand: from the second iteration on its flags
        // were cleared just now, so they are set again for the next compaction
        if (edges == 0 || iters >= most || (iters > 0 && edges > SOLO_E)) {
            if (iters > 0 && edges > 0) {
#pragma unroll
                for (int k = 0; k < 2; ++k)
                    if (2 * t + k < n && d[k] > 0) {
                        const int slot = cur[2 * t + k];
                        atomicOr(&bm[slot >> 5], 1u << (slot & 31));
                    }
            }
            break;
        }
        __syncthreads();
        sum += live;
        ++iters;
        for (int b0 = 0; b0 < edges; b0 += UNR * WG) {
            int tv[UNR], alt[UNR], cv[UNR];
#pragma unroll
            for (int k = 0; k < UNR; ++k) {
                const int i = b0 + k * WG + t;
                int o = 0;  // owner: the last vertex whose prefix is <= i
#pragma unroll
                for (int step = SOLO_V / 2; step > 0; step >>= 1)
                    if (o + step < n && sb.pre[o + step] <= i) o += step;
                const bool ok = i < edges;
                const int e = ok ? i + sb.start[o] : 0;
                tv[k] = ok ? sb.base[o] + st.col[e] : -1;
                alt[k] = ok ? sb.du[o] + (UNIT ? 1 : st.w[e]) : 0;
            }
#pragma unroll
            for (int k = 0; k < UNR; ++k) cv[k] = tv[k] >= 0 ? ld_coherent(st.dist + tv[k]) : 0;
            unsigned prev[UNR];
#pragma unroll
            for (int k = 0; k < UNR; ++k) {
                prev[k] = ~0u;
                if (alt[k] >= cv[k]) continue;
                atomicMin(&st.dist[tv[k]], alt[k]);
                prev[k] = atomicOr(&bm[tv[k] >> 5], 1u << (tv[k] & 31));
            }
#pragma unroll
            for (int k = 0; k < UNR; ++k) {
                if (tv[k] < 0 || (prev[k] >> (tv[k] & 31)) & 1u) continue;
                const int at = atomicAdd(&sb.next, 1);
                if (at < SOLO_V) nxt[at] = tv[k];
            }
        }
        stores_done();  // the distances are in memory
        __syncthreads();
        n = sb.next;
        if (n > SOLO_V) break;  // the bitmap has them all
        if (n == 0) break;
    }
    if (t == 0) st.ctrl->frontier_total += sum;
    return iters;
}

// ------------------------------------------------------------------------------------
// persistent drive
// ------------------------------------------------------------------------------------
// SOLO: small frontiers run on one workgroup.  The registers of that (116 against 93) cost a workgroup
// per CU, 4 instead of 5, so graphs that want more go without (persistent_wgs in np_api.cpp).
template <bool BATCH, bool UNIT, bool PUSH, bool SOLO>
__global__ __launch_bounds__(WG) void k_persistent(DevState st, SchedDev sp) {
    __shared__ ItemTables tb;
    __shared__ int s_total;
    Ctrl *ctrl = st.ctrl;
    unsigned long long gen = 0;
    const unsigned nb = gridDim.x;
    long long t_prev = 0;
    // priority window: every workgroup computes the same sequence of thresholds
    int T = (!PUSH && sp.delta > 0) ? sp.delta : NO_WINDOW;
    int next = 0;  // counters and sums of the next compaction pass
    for (int it = 0;; ++it) {
        int *q_cur = st.queue[it & 1];
        if (blockIdx.x == 0 && phase_tid() == 0) {
            long long now = (long long)wall_clock64();
            if (it > 0 && sp.trace && it - 1 < sp.trace_cap) sp.trace[it - 1].t_end = now;
            t_prev = now;
        }
        if (PUSH && blockIdx.x == 0 && threadIdx.x < NCLS) st_coherent(st.cnt + ((it + 2) % 3) * NCLS + threadIdx.x, 0);
        for (;;) {
            const int slot = next;
            // every pass has counters of its own: one that queues nothing is followed by the next without
            // a barrier, while slower workgroups are still reading its zeros
            const int *cnt_cur = st.cnt + (PUSH ? it % 3 : slot) * NCLS;
            if (!PUSH) {
                // the counters and the statistics slot of the next pass were last read before the previous barrier
                next = slot == 2 ? 0 : slot + 1;
                if (blockIdx.x == 0 && phase_tid() < NCLS) st_coherent(st.cnt + next * NCLS + phase_tid(), 0);
                if (blockIdx.x == 0 && T != NO_WINDOW) deferred_clear(ctrl, next);
                compaction_impl<SOLO ? COMPACT_UNR : COMPACT_UNR - 1>(st.ctrl, st.bm[0], st.cls, st.seg_off, st.nwords, st.cnt + slot * NCLS, q_cur, st.dist, T, slot);
                if (!grid_sync(ctrl, nb, gen)) return;
            }
            const int tid = phase_tid();
            if (tid < NCLS) {
                tb.cnt[tid] = ld_coherent(cnt_cur + tid);
                tb.seg[tid] = st.seg_off[tid];
            }
            __syncthreads();
            if (tid < 64) {
                const long long tot = frontier_size(tb.cnt);
                if (tid == 0) s_total = tot > 0x7FFFFFFF ? 0x7FFFFFFF : (int)tot;
            }
            __syncthreads();
            if (s_total > 0 || T == NO_WINDOW) break;
            // nothing below the window: raise it to the least pending distance + delta
            int kept, mn;
            deferred_sums(ctrl, slot, &kept, &mn);
            if (kept == 0) break;
            T = __builtin_amdgcn_readfirstlane(mn > NO_WINDOW - sp.delta ? NO_WINDOW : mn + sp.delta);
        }
        const int tid = phase_tid();
        const int total = __builtin_amdgcn_readfirstlane(s_total);
        if (total == 0 || (sp.max_iters > 0 && it >= sp.max_iters)) {
            if (blockIdx.x == 0 && tid == 0) {
                ctrl->iters = it;
                ctrl->done = total == 0 ? 1 : 0;
                if (total != 0) ctrl->error = NP_ERR_NOT_CONVERGED;
            }
            return;
        }
        if (SOLO && T == NO_WINDOW && !sp.trace && solo_fits(tb, total)) {
            __shared__ SoloBufs s_solo;
            int most = SOLO_ITERS;
            if (sp.max_iters > 0 && sp.max_iters - it < most) most = sp.max_iters - it;
            if (blockIdx.x == 0) {
                const int k = solo_iterations<BATCH, UNIT>(st, tb, q_cur, s_solo, total, most);
                if (tid == 0) st_coherent(&ctrl->solo, k);
            }
            if (!grid_sync(ctrl, nb, gen)) return;
            it += __builtin_amdgcn_readfirstlane(ld_coherent(&ctrl->solo)) - 1;
            continue;
        }
        Cfg cfg = decide(sp, tb.cnt, it);
        if (tid < 64) build_tables(tb, cfg, TABLES_SINGLE, (long long)nb * WAVES);
        if (blockIdx.x == 0 && tid < 64) {
            if (tid == 0) ctrl->frontier_total += total;
            record_trace(sp, it, cfg, tb.cnt, t_prev, ctrl);
        }
        __syncthreads();
        PushCtx pc;
        pc.bm_next = PUSH ? st.bm[(it + 1) & 1] : st.bm[0];
        pc.bm_cur = st.bm[it & 1];
        pc.cnt_next = st.cnt + ((it + 1) % 3) * NCLS;
        pc.q_next = st.queue[(it + 1) & 1];
        expansion<BATCH, UNIT, PUSH, false>(st, pc, q_cur, tb);
        if (!grid_sync(ctrl, nb, gen)) return;
    }
}

// ------------------------------------------------------------------------------------
// host-loop / graph drive kernels
// ------------------------------------------------------------------------------------
__global__ __launch_bounds__(WG) void k_compact(DevState st, int it_off) {
    Ctrl *ctrl = st.ctrl;
    if (ld_coherent(&ctrl->done) || ld_coherent(&ctrl->error)) return;
    const int it = ld_coherent(&ctrl->it_base) + it_off;
    const int pass = ld_coherent(&ctrl->pass);
    const int T = ld_coherent(&ctrl->thresh);
    if (blockIdx.x == 0 && threadIdx.x < NCLS) st.cnt[((it + 2) % 3) * NCLS + threadIdx.x] = 0;
    if (blockIdx.x == 0) deferred_clear(ctrl, (pass + 1) % 3);
    compaction_impl<COMPACT_UNR>(st.ctrl, st.bm[0], st.cls, st.seg_off, st.nwords, st.cnt + (it % 3) * NCLS, st.queue[it & 1],
                    st.dist, T, pass % 3);
}

__global__ __launch_bounds__(WG) void k_decide(DevState st, SchedDev sp, int it_off) {
    __shared__ int s_cnt[NCLS];
    Ctrl *ctrl = st.ctrl;
    if (ld_coherent(&ctrl->done) || ld_coherent(&ctrl->error)) return;
    const int it = ld_coherent(&ctrl->it_base) + it_off;
    if (threadIdx.x < NCLS) s_cnt[threadIdx.x] = ld_coherent(st.cnt + (it % 3) * NCLS + threadIdx.x);
    __syncthreads();
    const long long tot = frontier_size(s_cnt);  // every wavefront for itself
    const int pass = ld_coherent(&ctrl->pass);  // the compaction of this slot
    if (tot == 0 && !sp.push) {
        const int T = ld_coherent(&ctrl->thresh);
        const int win = ld_coherent(&ctrl->win);
        int kept, mn;
        deferred_sums(ctrl, (st.deferred ? win : pass) % 3, &kept, &mn);
        if (T != NO_WINDOW ? mn != NO_WINDOW : st.hold_cls && kept != 0) {
            // nothing queued but pairs kept back: raise the window (held vertices need only the
            // next pass); this slot's expansion is skipped
            if (threadIdx.x == 0) {
                if (T != NO_WINDOW) {
                    ctrl->thresh = mn > NO_WINDOW - sp.delta ? NO_WINDOW : mn + sp.delta;
                    ctrl->full = 1;  // a pack's next pass looks at its deferred pairs
                    ctrl->win = win + 1;
                }
                ctrl->skip = 1;
                ctrl->pass = pass + 1;
            }
            return;
        }
    }
    if (tot == 0 || (sp.max_iters > 0 && ctrl->iters >= sp.max_iters)) {
        if (threadIdx.x == 0) {
            if (tot == 0) ctrl->done = 1;
            else ctrl->error = NP_ERR_NOT_CONVERGED;
        }
        return;
    }
    if (st.bound && threadIdx.x < 64) {
        // bound filter: one iteration after enough of the sources reached the hub (their first
        // distances there are far from final) the bounds are computed and switched on
        const int f = ld_coherent(&ctrl->filt);
        const int j = threadIdx.x;
        const int d = f < 2 && j < (1 << st.kshift) ? ld_coherent(st.dist + j) : st.inf;
        const unsigned m = (unsigned)__ballot(d < st.inf);
        if (f == 1) {
            if (j < PACK_MAX) ctrl->foff[j] = d < st.inf ? d : 0;
            if (j == 0) { ctrl->fmask = m; ctrl->filt = 2; }
        } else if (f == 0 && j == 0 && __popc(m) >= st.fmin) {
            ctrl->filt = 1;
        }
    }
    Cfg cfg = decide(sp, s_cnt, ctrl->iters);
    if (threadIdx.x < 64) {
        if (ctrl->cfg_pad != 0) cfg = make_cfg(ctrl->cfg_level, ctrl->cfg_klo, ctrl->cfg_khi);  // forced (stepping)
        record_trace(sp, ctrl->iters, cfg, s_cnt, (long long)wall_clock64(), ctrl);
    }
    if (threadIdx.x == 0) {
        ctrl->cfg_level = cfg.level;
        ctrl->cfg_klo = cfg.klo;
        ctrl->cfg_khi = cfg.khi;
        ctrl->frontier_total += tot;
        ctrl->iters += 1;
        ctrl->skip = 0;
        ctrl->full = 0;
        if (!sp.push) ctrl->pass = pass + 1;
    }
}

template <bool BATCH, bool UNIT, bool PUSH>
__global__ __launch_bounds__(WG) void k_expand(DevState st, int it_off) {
    __shared__ ItemTables tb;
    Ctrl *ctrl = st.ctrl;
    if (ld_coherent(&ctrl->done) || ld_coherent(&ctrl->error) || ld_coherent(&ctrl->skip)) return;
    const int it = ld_coherent(&ctrl->it_base) + it_off;
    if (threadIdx.x < NCLS) {
        tb.cnt[threadIdx.x] = ld_coherent(st.cnt + (it % 3) * NCLS + threadIdx.x);
        tb.seg[threadIdx.x] = st.seg_off[threadIdx.x];
    }
    if (PUSH && blockIdx.x == 0 && threadIdx.x < NCLS) st.cnt[((it + 2) % 3) * NCLS + threadIdx.x] = 0;
    __syncthreads();
    if (threadIdx.x < 64) {
        Cfg cfg = make_cfg(ld_coherent(&ctrl->cfg_level), ld_coherent(&ctrl->cfg_klo),
                           ld_coherent(&ctrl->cfg_khi));
        build_tables(tb, cfg, TABLES_SINGLE, (long long)gridDim.x * WAVES);
    }
    __syncthreads();
    PushCtx pc;
    pc.bm_next = PUSH ? st.bm[(it + 1) & 1] : st.bm[0];
    pc.bm_cur = st.bm[it & 1];
    pc.cnt_next = st.cnt + ((it + 1) % 3) * NCLS;
    pc.q_next = st.queue[(it + 1) & 1];
    expansion<BATCH, UNIT, PUSH, true>(st, pc, st.queue[it & 1], tb);
}

__global__ void k_advance(DevState st, int k) {
    if (threadIdx.x == 0 && blockIdx.x == 0) st.ctrl->it_base += k;
}

__global__ void k_set_cfg(DevState st, int level, int klo, int khi) {
    if (threadIdx.x == 0 && blockIdx.x == 0) {
        st.ctrl->cfg_level = level;
        st.ctrl->cfg_klo = klo;
        st.ctrl->cfg_khi = khi;
        st.ctrl->cfg_pad = 1;
    }
}

// ------------------------------------------------------------------------------------
// the reference's other schedules (SSSP_GPU solutions 0-5, BFS_REC_GPU solutions 0 and 2)
// ------------------------------------------------------------------------------------
// They run on the host-loop and graph drives after the scan compaction and k_decide of the
// consolidated path, over the same class-segmented queue; they differ from it, and from one
// another, only in how queued vertices are mapped to workers (sssp_wrapper.cu:151-473,
// sssp_kernel.cu:34-327; bfs_rec_kernel.cu:41-140).  A vertex is heavy when its out-degree is
// at least 2^cfg_klo (THRESHOLD 64 = 2^6, sssp_kernel.cu:7), i.e. its class is >= cfg_klo + 1.
// Every relaxation is the reference's: alt = dist[u] + w; if (dist[v] > alt) atomicMin.

// One lane walks all edges of one vertex (the thread loop of unorder_threadQueue_kernel,
// sssp_kernel.cu:34-55), UNR edges' loads in flight at a time.
template <bool UNIT>
__device__ __forceinline__ void relax_serial(const DevState &st, const PushCtx &pc, int slot) {
    const int e0 = st.row[slot], e1 = st.row[slot + 1];
    const int du = ld_coherent(st.dist + slot);
    for (int base = e0; base < e1; base += UNR) {
        int tv[UNR], alt[UNR], cur[UNR];
#pragma unroll
        for (int k = 0; k < UNR; ++k) {
            const int e = base + k < e1 ? base + k : e0;
            tv[k] = st.col[e];
            alt[k] = du + (UNIT ? 1 : st.w[e]);
        }
#pragma unroll
        for (int k = 0; k < UNR; ++k) cur[k] = base + k < e1 ? ld_coherent(st.dist + tv[k]) : 0;
#pragma unroll
        for (int k = 0; k < UNR; ++k) {
            int c = 0;
            if (base + k < e1 && alt[k] < cur[k]) relax_tail<false>(st, pc, tv[k], alt[k], c);
        }
    }
}

// All lanes of `stride` workers (t = this one's index) walk the edges of one vertex.
template <bool UNIT>
__device__ __forceinline__ void relax_vertex(const DevState &st, const PushCtx &pc, int slot, int t, int stride) {
    const int e0 = st.row[slot], e1 = st.row[slot + 1];
    relax_range<UNIT, false, true>(st, pc, 0, e0, e1, ld_coherent(st.dist + slot), t, stride);
}

// Class prefix of the queued vertices of classes [c0, c1) into pre[0..NCLS] (thread 0).
__device__ __forceinline__ void sol_prefix(const int *cnt, int c0, int c1, long long *pre) {
    long long acc = 0;
    for (int c = 0; c < NCLS; ++c) {
        pre[c] = acc;
        if (c >= c0 && c < c1) acc += cnt[c];
    }
    pre[NCLS] = acc;
}

struct SolBufs {
    int *buf;  // global delayed buffer (solution 3): heavy vertices of one expansion
    int *bcnt; // [3] its fill counters, rotating by iteration
};

enum SolMode { SOL_THREAD = 0, SOL_DUAL = 1, SOL_LDS = 2, SOL_GLOBAL = 3, SOL_WAVE = 4, SOL_WGLIST = 5 };

// The parent kernel of solutions 0-5: one lane per queued vertex.
//   SOL_THREAD  every vertex walked by its lane (solution 0, unorder_threadQueue_kernel)
//   SOL_DUAL    light classes only; the heavy ones are the second queue (solution 1)
//   SOL_LDS     heavy vertices of the workgroup's 256 into an LDS buffer, then the whole
//               workgroup walks each one's edges (solution 2,
//               unorder_threadQueue_shared_delaybuffer_kernel, sssp_kernel.cu:112-172)
//   SOL_GLOBAL  heavy vertices appended to a global buffer (one atomic per wavefront),
//               drained by k_sol_drain (solution 3, sssp_kernel.cu:179-209)
//   SOL_WAVE    each wavefront then walks its own heavy vertices one by one with 64 lanes
//               (solution 4: a 64-thread nested launch per heavy vertex, sssp_kernel.cu:237-286)
//   SOL_WGLIST  heavy vertices of the workgroup into an LDS list; its four wavefronts take
//               them in turn, 64 lanes per vertex (solution 5: one nested launch per block
//               over the block's buffer, 64 threads per vertex, sssp_kernel.cu:289-327)
template <int MODE, bool UNIT>
__global__ __launch_bounds__(WG) void k_sol_parent(DevState st, SolBufs sb, int it_off) {
    __shared__ long long s_pre[NCLS + 1];
    __shared__ int s_seg[NCLS];
    __shared__ int s_list[WG];
    __shared__ int s_nlist;
    Ctrl *ctrl = st.ctrl;
    if (ld_coherent(&ctrl->done) || ld_coherent(&ctrl->error) || ld_coherent(&ctrl->skip)) return;
    const int it = ld_coherent(&ctrl->it_base) + it_off;
    const int hc = ld_coherent(&ctrl->cfg_klo) + 1;  // first heavy class
    const int *cnt = st.cnt + (it % 3) * NCLS;
    if (MODE == SOL_GLOBAL && blockIdx.x == 0 && threadIdx.x == 0) st_coherent(sb.bcnt + (it + 1) % 3, 0);
    if (threadIdx.x < NCLS) s_seg[threadIdx.x] = st.seg_off[threadIdx.x];
    if (threadIdx.x == 0) {
        int lc[NCLS];
        for (int c = 0; c < NCLS; ++c) lc[c] = ld_coherent(cnt + c);
        sol_prefix(lc, 1, MODE == SOL_DUAL ? hc : NCLS, s_pre);
        s_nlist = 0;
    }
    __syncthreads();
    const long long total = s_pre[NCLS];
    const int *q = st.queue[it & 1];
    PushCtx pc;
    pc.bm_next = st.bm[0];
    const int lane = lane_id(), wave = threadIdx.x >> 6;
    for (long long base = (long long)blockIdx.x * WG; base < total; base += (long long)gridDim.x * WG) {
        const long long i = base + threadIdx.x;
        int slot = 0, c = 0;
        const bool valid = i < total;
        if (valid) {
            c = find_class(s_pre, i);
            slot = ld_coherent(q + s_seg[c] + (i - s_pre[c]));
        }
        const bool heavy = valid && MODE != SOL_THREAD && MODE != SOL_DUAL && c >= hc;
        if (valid && !heavy) relax_serial<UNIT>(st, pc, slot);
        if (MODE == SOL_LDS || MODE == SOL_WGLIST) {
            if (heavy) s_list[atomicAdd(&s_nlist, 1)] = slot;
            __syncthreads();
            const int nl = s_nlist;
            if (MODE == SOL_LDS) {
                for (int k = 0; k < nl; ++k) relax_vertex<UNIT>(st, pc, s_list[k], threadIdx.x, WG);
            } else {
                for (int k = wave; k < nl; k += WAVES) relax_vertex<UNIT>(st, pc, s_list[k], lane, 64);
            }
            __syncthreads();
            if (threadIdx.x == 0) s_nlist = 0;
            __syncthreads();
        } else if (MODE == SOL_WAVE) {
            unsigned long long m = __ballot(heavy);
            while (m) {
                const int l = __ffsll((long long)m) - 1;
                m &= m - 1;
                relax_vertex<UNIT>(st, pc, __shfl(slot, l), lane, 64);
            }
        } else if (MODE == SOL_GLOBAL) {
            const unsigned long long m = __ballot(heavy);
            if (m) {
                int at = 0;
                if (lane == 0) at = atomicAdd(sb.bcnt + it % 3, __popcll(m));
                at = __shfl(at, 0);
                const long long bi = (long long)at + __popcll(m & __lanemask_lt());
                if (heavy && seg_ok(ctrl, bi, 0, st.seg_off[NCLS])) st_coherent(sb.buf + bi, slot);
            }
        }
    }
}

// Second launch of solution 1: one workgroup per heavy vertex (unorder_blockQueue_kernel,
// sssp_kernel.cu:57-78, over the heavy queue).
template <bool UNIT>
__global__ __launch_bounds__(WG) void k_sol_heavy(DevState st, int it_off) {
    __shared__ long long s_pre[NCLS + 1];
    __shared__ int s_seg[NCLS];
    Ctrl *ctrl = st.ctrl;
    if (ld_coherent(&ctrl->done) || ld_coherent(&ctrl->error) || ld_coherent(&ctrl->skip)) return;
    const int it = ld_coherent(&ctrl->it_base) + it_off;
    const int hc = ld_coherent(&ctrl->cfg_klo) + 1;
    const int *cnt = st.cnt + (it % 3) * NCLS;
    if (threadIdx.x < NCLS) s_seg[threadIdx.x] = st.seg_off[threadIdx.x];
    if (threadIdx.x == 0) {
        int lc[NCLS];
        for (int c = 0; c < NCLS; ++c) lc[c] = ld_coherent(cnt + c);
        sol_prefix(lc, hc, NCLS, s_pre);
    }
    __syncthreads();
    const long long total = s_pre[NCLS];
    const int *q = st.queue[it & 1];
    PushCtx pc;
    pc.bm_next = st.bm[0];
    for (long long k = blockIdx.x; k < total; k += gridDim.x) {
        const int c = find_class(s_pre, k);
        relax_vertex<UNIT>(st, pc, ld_coherent(q + s_seg[c] + (k - s_pre[c])), threadIdx.x, WG);
    }
}

// Second launch of solution 3: one wavefront per buffered vertex (NESTED_BLOCK_SIZE 64 threads
// of sssp_process_buffer / unorder_blockQueue_kernel).
template <bool UNIT>
__global__ __launch_bounds__(WG) void k_sol_drain(DevState st, SolBufs sb, int it_off) {
    Ctrl *ctrl = st.ctrl;
    if (ld_coherent(&ctrl->done) || ld_coherent(&ctrl->error) || ld_coherent(&ctrl->skip)) return;
    const int it = ld_coherent(&ctrl->it_base) + it_off;
    const int nb = ld_coherent(sb.bcnt + it % 3);
    PushCtx pc;
    pc.bm_next = st.bm[0];
    const long long nw = (long long)gridDim.x * WAVES;
    for (long long k = (long long)blockIdx.x * WAVES + (threadIdx.x >> 6); k < nb; k += nw)
        relax_vertex<UNIT>(st, pc, ld_coherent(sb.buf + k), lane_id(), 64);
}

// BFS_REC_GPU solution 0 (bfs_kernel_flat, bfs_rec_kernel.cu:41-58): level-synchronous and
// topology-driven -- every vertex is inspected at every level; those at `level` set their
// unreached or deeper children to level + 1 (plain stores: every writer of a level writes the
// same value) and raise *changed.
__global__ __launch_bounds__(WG) void k_bfs_flat(const int *row, const int *col, int *lvl, int n, int level,
                                                 int *changed) {
    int any = 0;
    for (long long v = (long long)blockIdx.x * WG + threadIdx.x; v < n; v += (long long)gridDim.x * WG) {
        if (lvl[v] != level) continue;
        for (int e = row[v], e1 = row[v + 1]; e < e1; ++e) {
            const int t = col[e];
            if (lvl[t] > level + 1) { lvl[t] = level + 1; any = 1; }
        }
    }
    if (__ballot(any) && lane_id() == 0) st_coherent(changed, 1);
}

// BFS_REC_GPU solution 2 (bfs_kernel_dp_hier, bfs_rec_kernel.cu:95-140): two levels per
// expansion.  A queued vertex u's children are taken 64 at a time by one wavefront, a lane
// per child (the reference's block per child); each child whose level this lane lowered to
// level(u) + 1 is expanded at once by the whole wavefront (the reference's threads over the
// grandchildren), and the grandchildren it lowers to level(u) + 2 are flagged for the next
// expansion (the reference's nested launch per grandchild).  Levels are exact: a vertex is
// expanded after every lowering of its level, as in the consolidated path.
__device__ __forceinline__ int hier_chunks(int c) { return c <= 6 ? 1 : 1 << (c - 6); }

__global__ __launch_bounds__(WG) void k_bfs_hier(DevState st, int it_off) {
    __shared__ long long s_pre[NCLS + 1];
    __shared__ int s_seg[NCLS];
    Ctrl *ctrl = st.ctrl;
    if (ld_coherent(&ctrl->done) || ld_coherent(&ctrl->error) || ld_coherent(&ctrl->skip)) return;
    const int it = ld_coherent(&ctrl->it_base) + it_off;
    const int *cnt = st.cnt + (it % 3) * NCLS;
    if (threadIdx.x < NCLS) s_seg[threadIdx.x] = st.seg_off[threadIdx.x];
    if (threadIdx.x == 0) {
        long long acc = 0;
        for (int c = 0; c < NCLS; ++c) {
            s_pre[c] = acc;
            if (c >= 1) acc += (long long)ld_coherent(cnt + c) * hier_chunks(c);
        }
        s_pre[NCLS] = acc;
    }
    __syncthreads();
    const long long total = s_pre[NCLS];
    const int *q = st.queue[it & 1];
    PushCtx pc;
    pc.bm_next = st.bm[0];
    const int lane = lane_id();
    const long long nw = (long long)gridDim.x * WAVES;
    for (long long k = (long long)blockIdx.x * WAVES + (threadIdx.x >> 6); k < total; k += nw) {
        const int c = find_class(s_pre, k);
        const long long r = k - s_pre[c];
        const int sh = c <= 6 ? 0 : c - 6;
        const int u = ld_coherent(q + s_seg[c] + (r >> sh));
        const int j = (int)(r & ((1ll << sh) - 1));
        const long long e = (long long)st.row[u] + (long long)j * 64 + lane;
        const int e1 = st.row[u + 1];
        const int du = ld_coherent(st.dist + u);
        bool won = false;
        int child = 0;
        if (e < e1) {
            child = st.col[e];
            const int alt = du + 1;
            if (alt < ld_coherent(st.dist + child)) won = alt < atomicMin(&st.dist[child], alt);
        }
        unsigned long long m = __ballot(won);
        while (m) {
            const int l = __ffsll((long long)m) - 1;
            m &= m - 1;
            const int ch = __shfl(child, l);
            relax_range<true, false, true>(st, pc, 0, st.row[ch], st.row[ch + 1], du + 1, lane, 64);
        }
    }
}

// ------------------------------------------------------------------------------------
// source-packed batch: up to 32 sources of one graph solved together
// ------------------------------------------------------------------------------------
// Distances are vertex-major, 2^kshift sources per vertex row: dist[(v << kshift) + i].
// The distances of every source at one vertex share a cache line (64 B for 16 sources),
// so one read of an edge's col/w serves every source pending at its tail, and the check
// of dist[v][*] is one coalesced line instead of one random sector per source.
// mflag[v] collects the sources whose distance at v improved since v was last queued;
// the relaxation that made it nonzero also stores 1 to a byte that 8 vertices share (pk_mark, in
// bm[0]), so the compaction scans n/8 bytes and reads mflag only where work is pending.
// A queue entry carries the source mask it was queued with (qmask).  The work of a
// queued vertex is out-degree x pending sources; its items are numbered edge-major,
// item t = (edge t / P, t % P-th pending source), so the P lanes of one edge are adjacent.
// The relaxation per (edge, source) is the reference's: alt = dist[u][i] + w;
// if (dist[v][i] > alt) atomicMin -- int32, as in the single-source kernels.

// Position of the k-th (0-based) set bit of m (k < popcount(m)).
__device__ __forceinline__ int nth_set_bit(unsigned m, int k) {
    int pos = 0, c;
    c = __popc(m & 0xFFFFu); if (k >= c) { k -= c; m >>= 16; pos += 16; }
    c = __popc(m & 0xFFu);   if (k >= c) { k -= c; m >>= 8;  pos += 8; }
    c = __popc(m & 0xFu);    if (k >= c) { k -= c; m >>= 4;  pos += 4; }
    c = __popc(m & 0x3u);    if (k >= c) { k -= c; m >>= 2;  pos += 2; }
    c = (int)(m & 1u);       if (k >= c) { pos += 1; }
    return pos;
}

// Lane-bin vertices of a packed expansion have out-degree < 2^(PACK_LANE_CLS - 1): each lane
// of a lane tile walks the edges of one vertex in sequence (pk_lane_tile), so the bin is kept to
// short rows; longer ones go to the wavefront and wider bins whatever the schedule says.
constexpr int PACK_LANE_CLS = 10;

// The mark of v and its 7 neighbours.  A byte, set by a plain store: as a bit set by an atomicOr it
// was a third of the atomics of a sparse graph's expansion (27 G lines/s whatever they do), 32
// sources of a 2048^2 grid 26.5 -> 22.1 ms per solve, of 1024^2 9.3 -> 7.7 (ER 1 M and R-MAT within
// 3 % either way).  A byte per 32 vertices made ER 65,536 25 to 30 % slower: stores to one line take
// turns too.
__device__ __forceinline__ unsigned char *pk_mark(const DevState &st, long long v) {
    return (unsigned char *)st.bm[0] + (v >> 3);
}

// UNR packed relaxation steps of a wavefront: in step k every lane holds one (edge, source)
// item -- target tv[k], pending source s, candidate alt[k] = dist[u][s] + w, loaded dist[v][s]
// cur[k] -- or none (ok[k] false).  The lanes of one edge form a run of consecutive lanes (rs =
// the run's first lane inside this wavefront, last = this lane ends its run), so they share v.
// The reference's relaxation per item (sssp_kernel.cu:46-52): if (dist[v][s] > alt) atomicMin,
// issued without a return value; each source that passed the check sets its bit in mflag[v],
// OR-ed across the run first so that one lane per run updates it, and the first bit of mflag[v]
// marks v (pk_mark).  Flagging on the check alone flags exactly the (v, s) the atomic's old
// value would: when alt < cur but a concurrent atomicMin has already stored less, that writer
// passed its own check in this same launch and flags (v, s) itself (every earlier store is
// visible to the check).  So no lane waits for an atomic's return before the next step.
// Vertices without out-edges are flagged too and dropped by the compaction.  Every lane of the
// wavefront calls it together.
__device__ __forceinline__ void pk_relax_steps(const DevState &st, int lane, const bool *ok, const int *tv, int s,
                                               const int *alt, const int *cur, int rs, bool last) {
#pragma unroll
    for (int k = 0; k < UNR; ++k) {
        if (ok[k] && alt[k] < cur[k])
            atomicMin(st.dist + (((unsigned)tv[k] << st.kshift) + (unsigned)s), alt[k]);
    }
    // every step's mflag OR is issued before any old value is tested: one wait for all UNR
    unsigned prev[UNR];
#pragma unroll
    for (int k = 0; k < UNR; ++k) {
        prev[k] = 1u;
        const unsigned bit = (ok[k] && alt[k] < cur[k]) ? 1u << s : 0u;
        if (__ballot(bit != 0) == 0) continue;
        unsigned acc = bit;
#pragma unroll
        for (int d = 1; d < 32; d <<= 1) {  // runs are at most 32 lanes long (one per source)
            const unsigned y = __shfl_up(acc, d);
            if (lane - d >= rs) acc |= y;
        }
        if (last && ok[k] && acc) prev[k] = atomicOr(&st.mflag[tv[k]], acc);
    }
#pragma unroll
    for (int k = 0; k < UNR; ++k)
        if (prev[k] == 0) st_coherent_b(pk_mark(st, tv[k]), 1);
}

// Items of one queued vertex u -- edges [e0, e1) x the P pending sources of M -- on `stride`
// workers (t = this worker's index; M, e0, e1 are the same for all of them).  Worker t takes
// source j = t mod P, whose distance at u it reads once, and the edges e0 + t / P + k q,
// q = stride / P: the P workers of an edge are adjacent and share its col/w read and the cache
// line of dist[v][*]; the last stride mod P workers idle.
template <bool UNIT>
__device__ __forceinline__ void pk_relax_vertex(const DevState &st, int u, unsigned M, int e0, int e1, int t,
                                                int stride) {
    M = (unsigned)__builtin_amdgcn_readfirstlane((int)M);
    const int P = __popc(M);
    if (P == 0 || e0 >= e1) return;
    const int ks = st.kshift;
    const int q = stride / P;
    const int eo = t / P, j = t - eo * P;
    const bool on = eo < q;
    const int s = on ? nth_set_bit(M, j) : 0;
    const int du = on ? ld_coherent(st.dist + (((unsigned)u << ks) + (unsigned)s)) : 0;
    const int lane = lane_id();
    const int rs = lane - j > 0 ? lane - j : 0;
    const bool last = j == P - 1 || lane == 63;
    for (int e = e0 + eo; __ballot(on && e < e1) != 0; e += UNR * q) {
        int tv[UNR], alt[UNR], cur[UNR];
        bool ok[UNR];
#pragma unroll
        for (int k = 0; k < UNR; ++k) {
            const int ek = e + k * q;
            ok[k] = on && ek < e1;
            const unsigned ec = ok[k] ? ek : e0;
            tv[k] = st.col[ec];
            alt[k] = du + (UNIT ? 1 : st.w[ec]);
        }
#pragma unroll
        for (int k = 0; k < UNR; ++k)
            cur[k] = ok[k] ? ld_coherent(st.dist + (((unsigned)tv[k] << ks) + (unsigned)s)) : 0;
        pk_relax_steps(st, lane, ok, tv, s, alt, cur, rs, last);
    }
}

// Bound filter of a pack on a skewed graph.  Once every source has reached the core, most edges a
// packed expansion reads improve nothing (R-MAT s18, 16 sources, CPU model: 0.40 of 4.8 x m edge
// rows improve), yet each costs a random row of distances and a lane per pending source.  The
// sources' distances at a vertex differ mostly by one offset per source, its distance off[s] at the
// hub: max over s of (dist[v][s] - off[s]) is a bound within a few units of every source's own
// value.  An edge (u, v) with min over u's pending s of (dist[u][s] - off[s]) + w >= bound[v] can
// improve no source, so it is dropped after reading one byte.  The bounds are upper bounds whatever
// off[] is (any constants would do) and stay valid without upkeep, because distances only fall; a
// vertex's bound is refreshed when it is expanded, as a tile, by a wavefront or by the whole grid.
// Rows in the workgroup bin (level 1, from class PK_TILE_CLS on) are neither filtered nor refreshed.
// Sources that had not reached the hub when off[] was taken (fmask clear) have no part in the bounds,
// and edges of a vertex pending for one of them are never dropped.  16 sources of R-MAT s24, one solve: the four heaviest filtered expansions
// 5.2 / 4.8 / 3.7 / 1.6 -> 4.1 / 3.2 / 2.4 / 1.1 ms, for 0.29 ms of bounds; what is left of them is
// the stream of the rows themselves.
// A byte holds ceil((bound - FBASE) / 2^fshift) with FBASE = -64 steps, 255 = no bound.
constexpr int FBASE_STEPS = 64;
constexpr int FNONE = 255;
constexpr int FLOW = -(1 << 30), FHIGH = 1 << 30;  // below / above every normalised distance in use

__device__ __forceinline__ int pk_bound_code(int b, int fshift) {
    if (b >= FHIGH) return FNONE;
    const int x = b + (FBASE_STEPS << fshift);
    const int q = x <= 0 ? 0 : (x + (1 << fshift) - 1) >> fshift;
    return q < FNONE ? q : FNONE;
}
// true when an edge with candidate value thr + w (relative to FBASE) may improve a source of the
// vertex with bound code q
__device__ __forceinline__ bool pk_may_improve(int q, int thr, int w, int fshift) {
    return q == FNONE || thr + w < (q << fshift);
}
// One thread over vertex v's whole row: its bound (*hi) over the sources in `mask`, and the least
// normalised distance (*lo) of the sources pending in m, FLOW when one of them is not in mask.
__device__ __forceinline__ void pk_row_bound(const DevState &st, long long v, const int *off, unsigned mask, unsigned m,
                                             int *hi, int *lo) {
    const int *row = st.dist + (v << st.kshift);
    int h = FLOW, l = (m & ~mask) ? FLOW : FHIGH;
    for (int q = 0; q < (1 << st.kshift) / 4; ++q) {
        const int4 x = ((const int4 *)row)[q];
        const int d[4] = {x.x, x.y, x.z, x.w};
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const int y = d[k] >= st.inf ? FHIGH : d[k] - off[4 * q + k];
            const bool in = (mask >> (4 * q + k)) & 1u;
            h = in && y > h ? y : h;
            l = in && ((m >> (4 * q + k)) & 1u) && y < l ? y : l;
        }
    }
    *hi = h;
    *lo = l;
}
// What an expansion needs of the filter, per lane: source lane & (row length - 1).
struct PkFilt {
    const int *off;   // [PACK_MAX] in LDS
    unsigned mask;
};

// Wavefront-scope form of pk_relax_vertex (stride 64) with the neighbour tile staged in LDS: the
// wavefront copies up to PK_TILE consecutive edges' col (and w) into its own LDS slice with
// coalesced loads, one edge per lane per load, then takes the edges of its relaxation steps from
// there.  Without staging every step re-reads col/w from global memory, q = 64 / P distinct edges
// per load, and waits for them before its distance gathers.  tcol / tw: the wavefront's slice.
constexpr int PK_TILE = 256;
// a group of UNR steps spans up to UNR * 64 edges (one pending source): a tile must hold one,
// or the rounded tile below would be empty and its loop would not advance
static_assert(PK_TILE >= UNR * 64 && PK_TILE % 64 == 0, "PK_TILE must hold a step group of one source");
constexpr int PK_SLICE = 2 * PK_TILE;  // LDS entries per wavefront
template <bool UNIT, bool FILT>
__device__ __forceinline__ void pk_relax_vertex_staged(const DevState &st, const PkFilt &pf, int u, unsigned M, int e0,
                                                       int e1, bool first, int *tcol, int *tw) {
    M = (unsigned)__builtin_amdgcn_readfirstlane((int)M);
    const int P = __popc(M);
    if (P == 0 || e0 >= e1) return;
    const int ks = st.kshift;
    const int lane = lane_id();
    const int q = 64 / P;
    const int eo = lane / P, j = lane - eo * P;
    const bool on = eo < q;
    const int s = on ? nth_set_bit(M, j) : 0;
    int du, thr = 0;
    if (FILT) {
        // u's whole row: its bound, the least pending normalised distance and every lane's du
        const int sl = lane & ((1 << ks) - 1);
        const int d = ld_coherent(st.dist + (((unsigned)u << ks) + (unsigned)sl));
        const bool in = (pf.mask >> sl) & 1u;
        const int nd = d >= st.inf ? FHIGH : d - pf.off[sl];
        int hi = in ? nd : FLOW;
        int lo = !((M >> sl) & 1u) ? FHIGH : in ? nd : FLOW;
        for (int o = 1; o < (1 << ks); o <<= 1) {
            const int x = __shfl_xor(hi, o), y = __shfl_xor(lo, o);
            hi = x > hi ? x : hi;
            lo = y < lo ? y : lo;
        }
        if (first && lane == 0) st.bound[u] = (unsigned char)pk_bound_code(hi, st.fshift);
        thr = lo + (FBASE_STEPS << st.fshift);
        du = __shfl(d, s);
    } else {
        du = on ? ld_coherent(st.dist + (((unsigned)u << ks) + (unsigned)s)) : 0;
    }
    const int rs = lane - j > 0 ? lane - j : 0;
    const bool last = j == P - 1 || lane == 63;
    const int span = UNR * q;                  // edges of one group of UNR steps (<= PK_TILE)
    // unfiltered: whole groups per tile, so that no group straddles two tiles; filtered: the edges
    // that may improve gather in the slice until another tile might not fit
    const int tile = FILT ? PK_TILE : (PK_TILE / span) * span;
    int have = 0;
    for (int tb = e0; tb < e1; tb += tile) {
        int nt = e1 - tb < tile ? e1 - tb : tile;
        wave_lds_order();       // the previous tile's reads come first
        int c[PK_TILE / 64], wv[PK_TILE / 64];
#pragma unroll
        for (int r = 0; r < PK_TILE / 64; ++r) {
            const int i = lane + 64 * r;
            const int ic = tb + (i < nt ? i : nt - 1);  // lanes past the tile re-read its last edge
            c[r] = st.col[ic];
            wv[r] = UNIT ? 1 : st.w[ic];
        }
        if (FILT) {
            int b[PK_TILE / 64];
#pragma unroll
            for (int r = 0; r < PK_TILE / 64; ++r) b[r] = 64 * r < nt ? (int)st.bound[c[r]] : 0;
#pragma unroll
            for (int r = 0; r < PK_TILE / 64; ++r) {
                const bool keep = lane + 64 * r < nt && pk_may_improve(b[r], thr, wv[r], st.fshift);
                const unsigned long long m = __ballot(keep);
                if (keep) {
                    const int at = have + __popcll(m & __lanemask_lt());
                    tcol[at] = c[r];
                    if (!UNIT) tw[at] = wv[r];
                }
                have += __popcll(m);
            }
            if (have <= PK_SLICE - PK_TILE && tb + tile < e1) continue;
            nt = have;
            have = 0;
        } else {
#pragma unroll
            for (int r = 0; r < PK_TILE / 64; ++r) {
                tcol[lane + 64 * r] = c[r];
                if (!UNIT) tw[lane + 64 * r] = wv[r];
            }
        }
        wave_lds_order();
        for (int e = eo; __ballot(on && e < nt) != 0; e += span) {
            int tv[UNR], alt[UNR], cur[UNR];
            bool ok[UNR];
#pragma unroll
            for (int k = 0; k < UNR; ++k) {
                const int ek = e + k * q;
                ok[k] = on && ek < nt;
                const int ec = ok[k] ? ek : 0;
                tv[k] = tcol[ec];
                alt[k] = du + (UNIT ? 1 : tw[ec]);
            }
#pragma unroll
            for (int k = 0; k < UNR; ++k)
                cur[k] = ok[k] ? ld_coherent(st.dist + (((unsigned)tv[k] << ks) + (unsigned)s)) : 0;
            pk_relax_steps(st, lane, ok, tv, s, alt, cur, rs, last);
        }
    }
}

// Lane bin: 64 queued vertices (queue[qidx .. qidx+nvalid)) of one out-degree class.  Their
// (vertex, pending source) pairs go to the lanes, 64 at a time, the pairs of one vertex adjacent;
// each lane walks its vertex's edges in order for its source, so the lanes of one vertex read the
// same edge (one col/w address, one dist[v][*] line) at every step.
template <bool UNIT>
__device__ __forceinline__ void pk_lane_tile(const DevState &st, const int *q, const unsigned *qm,
                                             long long qidx, int nvalid) {
    const int lane = lane_id();
    const int ks = st.kshift;
    int u = 0, s0 = 0, d = 0, P = 0;
    unsigned M = 0;
    if (lane < nvalid) {
        u = ld_coherent(q + qidx + lane);
        M = ld_coherent_u(qm + qidx + lane);
        s0 = st.row[u];
        d = st.row[u + 1] - s0;
        P = d > 0 ? __popc(M) : 0;
    }
    const int incl = wave_incl_scan(P);
    const int total = __shfl(incl, 63);
    const int excl = incl - P;
    if (total == 0) return;
    // lanes past the last pair read the first edge of the first vertex with pairs (a valid edge)
    const int e_safe = __shfl(s0, __ffsll((long long)__ballot(P > 0)) - 1);
    for (int base = 0; base < total; base += 64) {
        const int k = base + lane;
        const bool on = k < total;
        int o = 0;  // owner: the last lane whose exclusive offset is <= k
#pragma unroll
        for (int step = 32; step > 0; step >>= 1) {
            const int x = __shfl(excl, o + step);
            if (x <= k) o += step;
        }
        const int j = k - __shfl(excl, o);
        const int Po = __shfl(P, o);
        const unsigned Mo = __shfl(M, o);
        const int uo = __shfl(u, o);
        // every lane takes part in each shuffle: a lane left out would return 0 to its readers
        const int so = __shfl(s0, o);
        const int dso = __shfl(d, o);
        const int e0 = on ? so : e_safe;
        const int deg = on ? dso : 0;
        const int s = on ? nth_set_bit(Mo, j) : 0;
        const int du = on ? ld_coherent(st.dist + (((unsigned)uo << ks) + (unsigned)s)) : 0;
        const int rs = lane - j > 0 ? lane - j : 0;
        const bool last = j == Po - 1 || lane == 63;
        for (int i = 0; __ballot(i < deg) != 0; i += UNR) {
            int tv[UNR], alt[UNR], cur[UNR];
            bool ok[UNR];
#pragma unroll
            for (int kk = 0; kk < UNR; ++kk) {
                ok[kk] = i + kk < deg;
                const unsigned ec = e0 + (ok[kk] ? i + kk : 0);  // a lane with deg 0 reads a valid edge of its tile
                tv[kk] = st.col[ec];
                alt[kk] = du + (UNIT ? 1 : st.w[ec]);
            }
#pragma unroll
            for (int kk = 0; kk < UNR; ++kk)
                cur[kk] = ok[kk] ? ld_coherent(st.dist + (((unsigned)tv[kk] << ks) + (unsigned)s)) : 0;
            pk_relax_steps(st, lane, ok, tv, s, alt, cur, rs, last);
        }
    }
}

// Filtered tile: up to 64 queued vertices of one out-degree class (pk_tile_vertices), about 768
// edges in all (cl = the class: degrees below 2^cl).  A lane reads one vertex's row (bound, least
// pending value); then the tile's edges are spread over the lanes, one lane per edge, and those that may improve are listed in LDS; a
// listed edge gets one lane per source of the row (2^kshift), so the sources that improve are one
// ballot.  One vertex per wavefront spent a chain of seven dependent accesses on about 40 edges.
// The listed edges 0 .. nt of the wave's slice; u, M: lane i holds the tile's vertex i.
__device__ __forceinline__ void pk_relax_listed(const DevState &st, int u, unsigned M, const int *tcol, const int *tw,
                                                const unsigned char *town, int nt) {
    const int ks = st.kshift;
    const int lane = lane_id();
    const int s = lane & ((1 << ks) - 1), rs = lane - s;
    const int per = 64 >> ks;  // edges per step
    const unsigned rowmask = ks == 5 ? ~0u : (1u << (1 << ks)) - 1u;
    for (int base = 0; base < nt; base += UNR * per) {
        int tv[UNR], alt[UNR], cur[UNR];
#pragma unroll
        for (int k = 0; k < UNR; ++k) {
            const int i = base + k * per + (lane >> ks);
            const int ic = i < nt ? i : 0;
            const int o = town[ic];
            const unsigned uo = (unsigned)__shfl(u, o);
            const unsigned Mo = (unsigned)__shfl((int)M, o);
            tv[k] = tcol[ic];
            const bool pend = i < nt && ((Mo >> s) & 1u);
            // cached: a value older than the vertex's last improvement only repeats what its next
            // expansion does again
            alt[k] = pend ? st.dist[(uo << ks) + (unsigned)s] + tw[ic] : 0;
            cur[k] = pend ? ld_coherent(st.dist + (((unsigned)tv[k] << ks) + (unsigned)s)) : 0;
        }
        unsigned prev[UNR];
#pragma unroll
        for (int k = 0; k < UNR; ++k) {
            prev[k] = 1u;
            const bool imp = alt[k] < cur[k];
            if (imp) atomicMin(st.dist + (((unsigned)tv[k] << ks) + (unsigned)s), alt[k]);
            const unsigned mine = (unsigned)(__ballot(imp) >> rs) & rowmask;
            if (s == 0 && mine) prev[k] = atomicOr(&st.mflag[tv[k]], mine);
        }
#pragma unroll
        for (int k = 0; k < UNR; ++k)
            if (prev[k] == 0) st_coherent_b(pk_mark(st, tv[k]), 1);
    }
}

__device__ __forceinline__ void pk_edge_tile(const DevState &st, const PkFilt &pf, const int *q, const unsigned *qm,
                                             long long qidx, int nvalid, int cl, int *tcol, int *tw, unsigned char *town) {
    const int lane = lane_id();
    int u = 0, s0 = 0, d = 0, thr = 0;
    unsigned M = 0;
    if (lane < nvalid) {
        u = ld_coherent(q + qidx + lane);
        M = ld_coherent_u(qm + qidx + lane);
        s0 = st.row[u];
        d = M ? st.row[u + 1] - s0 : 0;
        int hi, lo;
        pk_row_bound(st, u, pf.off, pf.mask, M, &hi, &lo);
        st.bound[u] = (unsigned char)pk_bound_code(hi, st.fshift);
        thr = lo + (FBASE_STEPS << st.fshift);
    }
    // 2^cl slots per vertex (its degree is at least half of that): a slot's vertex and edge are its
    // bits, where a prefix sum of the degrees needs a search of six dependent shuffles per edge
    const int total = nvalid << cl;
    int have = 0;
    for (int base = 0; base < total; base += UNR * 64) {
        int o[UNR], c[UNR], wv[UNR], b[UNR];
#pragma unroll
        for (int k = 0; k < UNR; ++k) {
            const int kk = base + k * 64 + lane;
            o[k] = (kk >> cl) & 63;
            const int i = kk & ((1 << cl) - 1);
            const int e = __shfl(s0, o[k]) + i;
            const bool ok = i < __shfl(d, o[k]) && kk < total;
            c[k] = ok ? st.col[e] : -1;
            wv[k] = ok ? st.w[e] : 0;
        }
#pragma unroll
        for (int k = 0; k < UNR; ++k) b[k] = c[k] >= 0 ? (int)st.bound[c[k]] : 0;
        wave_lds_order();  // the list's previous reads come first
#pragma unroll
        for (int k = 0; k < UNR; ++k) {
            const int t = __shfl(thr, o[k]);
            const bool keep = c[k] >= 0 && pk_may_improve(b[k], t, wv[k], st.fshift);
            const unsigned long long m = __ballot(keep);
            if (keep) {
                const int at = have + __popcll(m & __lanemask_lt());
                tcol[at] = c[k];
                tw[at] = wv[k];
                town[at] = (unsigned char)o[k];
            }
            have += __popcll(m);
        }
        wave_lds_order();
        if (have > PK_SLICE - UNR * 64 || base + UNR * 64 >= total) {
            pk_relax_listed(st, u, M, tcol, tw, town, have);
            have = 0;
        }
    }
}

template <bool UNIT, bool FILT>
__device__ void pk_expansion(const DevState &st, const PkFilt &pf, const int *q, const unsigned *qm, ItemTables &tb,
                             int *tcol, int *tw, unsigned char *town) {
    const int tid = phase_tid();
    const long long G = tb.pre[0][NCLS], K = tb.pre[1][NCLS], W = tb.pre[2][NCLS],
                    T = tb.pre[3][NCLS];
    for (long long k = blockIdx.x; k < K; k += gridDim.x) {
        int c = find_class(tb.pre[1], k);
        long long qi = tb.seg[c] + (k - tb.pre[1][c]);
        int u = ld_coherent(q + qi);
        unsigned M = ld_coherent_u(qm + qi);
        pk_relax_vertex<UNIT>(st, u, M, st.row[u], st.row[u + 1], tid, WG);
    }
    const long long NW = (long long)gridDim.x * WAVES;
    const long long gw = (long long)blockIdx.x * WAVES + (tid >> 6);
    const long long U = G + W + T;
    for (long long x = gw; x < U; x += NW) {
        if (x < G) {
            int c = find_class(tb.pre[0], x);
            long long r = x - tb.pre[0][c];
            int sh = c > GRID_CHUNK_SHIFT ? c - GRID_CHUNK_SHIFT : 0;
            long long qi = tb.seg[c] + (r >> sh);
            int j = (int)(r & ((1ll << sh) - 1));
            int u = ld_coherent(q + qi);
            unsigned M = ld_coherent_u(qm + qi);
            int s = st.row[u], e = st.row[u + 1];
            int e0 = s + (j << GRID_CHUNK_SHIFT);
            int e1 = e0 + (1 << GRID_CHUNK_SHIFT);
            if (e1 > e) e1 = e;
            pk_relax_vertex_staged<UNIT, FILT>(st, pf, u, M, e0, e1, j == 0, tcol, tw);
        } else if (x < G + W) {
            long long i = x - G;
            int c = find_class(tb.pre[2], i);
            long long qi = tb.seg[c] + (i - tb.pre[2][c]);
            int u = ld_coherent(q + qi);
            unsigned M = ld_coherent_u(qm + qi);
            pk_relax_vertex_staged<UNIT, FILT>(st, pf, u, M, st.row[u], st.row[u + 1], true, tcol, tw);
        } else {
            long long t = x - G - W;
            int c = find_class(tb.pre[3], t);
            long long ti = t - tb.pre[3][c];
            const int tv = FILT ? pk_tile_vertices(c) : 64;
            long long first = ti * tv;
            int nvalid = (int)((long long)tb.cnt[c] - first < tv ? (long long)tb.cnt[c] - first : tv);
            if (FILT) pk_edge_tile(st, pf, q, qm, tb.seg[c] + first, nvalid, c, tcol, tw, town);
            else pk_lane_tile<UNIT>(st, q, qm, tb.seg[c] + first, nvalid);
        }
    }
}

// Number of the pack's sources that have reached v (finite entries of its distance row; the
// row's unused entries stay at inf).
__device__ __forceinline__ int pk_reached(const DevState &st, long long v) {
    const int *row = st.dist + (v << st.kshift);
    int r = 0;
    if (st.kshift < 2) {
        for (int i = 0; i < (1 << st.kshift); ++i) r += ld_coherent(row + i) < st.inf;
        return r;
    }
    const int4 *row4 = (const int4 *)row;
    for (int q = 0; q < (1 << (st.kshift - 2)); ++q) {
        const int4 x = row4[q];
        r += (x.x < st.inf) + (x.y < st.inf) + (x.z < st.inf) + (x.w < st.inf);
    }
    return r;
}

// Lane q of a group of 8 has vertex v's distances of sources 4q .. 4q + 3 (rows of 1 or 2: source q).
// Through the caches in a launch of its own, which starts with none of them.  Inside the persistent
// kernel a cached row can be many iterations old, and only larger: pairs below the window were
// deferred, and the window rose above distances that were long passed (3 sources of a 2048^2 grid,
// window 2000: 339 iterations against 146 of launches), so there the loads are coherent.
template <bool COHERENT>
__device__ __forceinline__ int4 pk_row_part(const DevState &st, long long v, int q, bool ok) {
    const int *row = st.dist + (v << st.kshift);
    if (st.kshift < 2) {
        const bool in = ok && q < (1 << st.kshift);
        return int4{!in ? 0 : COHERENT ? ld_coherent(row + q) : row[q], 0, 0, 0};
    }
    if (!ok || q >= (1 << (st.kshift - 2))) return int4{0, 0, 0, 0};
    if (!COHERENT) return ((const int4 *)row)[q];
    const unsigned long long *p = (const unsigned long long *)row + 2 * q;
    const unsigned long long a = __hip_atomic_load(p, __ATOMIC_RELAXED, NP_AGENT);
    const unsigned long long b = __hip_atomic_load(p + 1, __ATOMIC_RELAXED, NP_AGENT);
    return int4{(int)a, (int)(a >> 32), (int)b, (int)(b >> 32)};
}
// The group's sources of mask m whose distance is below the window T, and the least distance among
// its others (both in every lane of the group).
__device__ __forceinline__ unsigned pk_take(const DevState &st, int4 x, int q, unsigned m, int T, int *dmin) {
    const int d[4] = {x.x, x.y, x.z, x.w};
    const int per = st.kshift < 2 ? 1 : 4;
    unsigned take = 0;
    int dm = NO_WINDOW;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        if (k >= per || !((m >> (per * q + k)) & 1u)) continue;
        if (d[k] < T || T == NO_WINDOW) take |= 1u << (per * q + k);
        else dm = d[k] < dm ? d[k] : dm;
    }
#pragma unroll
    for (int o = 1; o < 8; o <<= 1) {
        take |= (unsigned)__shfl_xor((int)take, o);
        const int y = __shfl_xor(dm, o);
        dm = y < dm ? y : dm;
    }
    *dmin = dm;
    return take;
}

// Vertices with pending sources -> class-segmented queue with their source masks.  With a
// priority window (T < NO_WINDOW) only the (vertex, source) pairs with dist < T are queued; the
// others move from mflag[v] to deferred[v].  A deferred pair is below the window only after a
// relaxation, which flags it again, or after the window has risen: so the passes of one window look at
// the flagged pairs alone, and only a `full` pass, the first one after the window has risen, looks at
// every deferred one.  Every pass adds the pairs it defers to the window's sums (`slot`), so the least
// of them bounds all that are pending from below when the window has to rise; the bound may belong to
// a pair taken since, then the window rises once more.  Kept flagged and re-read in every pass by a
// lane per row, the rows of the deferred were most of the compaction: 32 sources of a 2048^2 grid
// 16.5 -> 7.4 ms of it per solve (13.4 with a lane per row still), the solve 33.2 -> 26.5 ms.  A second
// full pass, to find the least pending distance before the window rises, cost small packs more than
// that saved (persistent drive, 3 sources of a 300^2 grid 6.2 -> 8.0 ms).
template <int WIN_UNR, bool COHERENT>
__device__ __forceinline__ void pk_compaction(const DevState &st, int *cnt_out, int *q_out, unsigned *qm_out,
                                              int T, bool full, int slot) {
    __shared__ int s_wc[WAVES][NCLS];
    static_assert(WAVES * NCLS <= WG, "cleared by one store each");
    __shared__ int s_dc, s_dm, s_pairs;
    const int tid = phase_tid();
    if (tid == 0) { s_dc = 0; s_dm = NO_WINDOW; s_pairs = 0; }
    if (tid < WAVES * NCLS) s_wc[0][tid] = 0;
    __syncthreads();
    int pairs = 0, my_dc = 0, my_dm = NO_WINDOW;
    const bool windowed = T != NO_WINDOW || full;
    // The marks are scanned as compaction_impl scans its words (a thread per word took 0.24 ms where this takes
    // 0.1, R-MAT s24, 16 sources, 8 M vertices queued); then the hubs held for one pass (hold_cls) or
    // the vertices without a pair below the window leave the list.
    __shared__ unsigned short s_list[WAVES][64 * 32];
    __shared__ unsigned s_held[WG];  // per word of the wave: held vertices, and whether it has hubs
    __shared__ int s_heavy[WG];
    const int lane = tid & 63, half = lane & 31;
    unsigned short *list = s_list[tid >> 6];
    int *wc = s_wc[tid >> 6];
    const int wt = compact_words(st.nwords, gridDim.x, st.deferred != nullptr);
    const long long tile = (long long)WAVES * wt;
    for (long long wb = (long long)blockIdx.x * tile; wb < st.nwords; wb += (long long)gridDim.x * tile) {
        const long long w0 = wb + (tid >> 6) * wt;
        const bool in = lane < wt && w0 + lane < st.nwords;
        const unsigned marks = in ? ld_coherent_u(st.bm[0] + w0 + lane) : 0u;  // of 32 vertices
        unsigned long long nz = __ballot(in && (full || marks));
        int n = 0;
        while (nz) {
            int idx[COMPACT_UNR], c[COMPACT_UNR];
            unsigned f[COMPACT_UNR];
#pragma unroll
            for (int k = 0; k < COMPACT_UNR; ++k) {
                const int ia = __ffsll((long long)nz) - 1;
                nz &= nz - 1;
                const int ib = __ffsll((long long)nz) - 1;
                nz &= nz - 1;
                idx[k] = lane < 32 ? ia : ib;  // -1: none left
                const long long v = (w0 + idx[k]) * 32 + half;
                const unsigned mk = full ? ~0u : __shfl(marks, idx[k] < 0 ? 0 : idx[k]);
                const bool ok = idx[k] >= 0 && (mk >> (half & 24) & 0xFFu) && v < st.nslots;
                c[k] = ok ? (int)st.cls[v] : 0;
                f[k] = ok ? ld_coherent_u(st.mflag + v) : 0u;
                if (full && ok) f[k] |= ld_coherent_u(st.deferred + v);
            }
            // no out-edges (class 0): dropped
#pragma unroll
            for (int k = 0; k < COMPACT_UNR; ++k) c[k] = f[k] ? c[k] : 0;
#pragma unroll
            for (int k = 0; k < COMPACT_UNR; ++k) {
                const unsigned long long m = __ballot(c[k] != 0);
                if (c[k]) list[n + __popcll(m & lanes_below(lane))] = (unsigned short)((c[k] << 11) | (idx[k] * 32 + half));
                n += __popcll(m);
            }
        }
        wave_lds_order();   // the list, written by all lanes, is read from here on
        unsigned stay = 0;  // vertices of this lane's word that stay pending
        if (windowed) {
            // 8 lanes per vertex read its row; a vertex with a pair below the window keeps its
            // mask for the queue in mflag, the others leave the list
            const int g = lane >> 3, q = lane & 7;
            int left = 0;
            for (int base = 0; base < n; base += 8 * WIN_UNR) {
                int e[WIN_UNR];
                unsigned f[WIN_UNR], old[WIN_UNR];
                int4 x[WIN_UNR];
#pragma unroll
                for (int k = 0; k < WIN_UNR; ++k) {
                    const int i = base + 8 * k + g;
                    e[k] = i < n ? (int)list[i] : 0;  // class 0: none
                    const long long v = w0 * 32 + (e[k] & 2047);
                    f[k] = e[k] ? ld_coherent_u(st.mflag + v) : 0u;
                    old[k] = e[k] ? ld_coherent_u(st.deferred + v) : 0u;
                    x[k] = pk_row_part<COHERENT>(st, v, q, e[k] != 0);
                }
                wave_lds_order();
#pragma unroll
                for (int k = 0; k < WIN_UNR; ++k) {
                    const long long v = w0 * 32 + (e[k] & 2047);
                    int dmin;
                    const unsigned m = full ? f[k] | old[k] : f[k];
                    const unsigned t = pk_take(st, x[k], q, m, T, &dmin);
                    const unsigned rest = (old[k] | f[k]) & ~t;
                    const bool take = q == 0 && t != 0;
                    if (q == 0 && e[k]) {
                        if (f[k] != t) st_coherent_u(st.mflag + v, t);
                        if (rest != old[k]) st_coherent_u(st.deferred + v, rest);
                        if (m & ~t) {
                            my_dc += __popc(m & ~t);
                            my_dm = dmin < my_dm ? dmin : my_dm;
                        }
                    }
                    const unsigned long long queued = __ballot(take);
                    if (take) list[left + __popcll(queued & lanes_below(lane))] = (unsigned short)e[k];
                    left += __popcll(queued);
                }
            }
            n = left;
            wave_lds_order();
        }
        if (st.hold_cls) {
            // hubs that more sources are on their way to wait one pass and keep their flag; a held
            // vertex stays flagged, so the held bits are always a subset of the flags: they become
            // exactly this pass's held vertices (the ones held before are queued).  Renumbered hubs
            // share a wavefront's words, so their rows are read COMPACT_UNR x 64 at a time.
            s_held[tid] = 0u;
            s_heavy[tid] = 0;
            unsigned *held_w = s_held + (tid & ~63);
            int *heavy_w = s_heavy + (tid & ~63);
            wave_lds_order();
            int left = 0;
            for (int base = 0; base < n; base += 64 * COMPACT_UNR) {
                int e[COMPACT_UNR], reached[COMPACT_UNR];
                unsigned hw[COMPACT_UNR];
#pragma unroll
                for (int k = 0; k < COMPACT_UNR; ++k) {
                    const int i = base + 64 * k + lane;
                    e[k] = i < n ? (int)list[i] : 0;
                    const bool heavy = (e[k] >> 11) >= st.hold_cls;
                    hw[k] = heavy ? ld_coherent_u(st.bm[1] + w0 + ((e[k] & 2047) >> 5)) : 0u;
                    reached[k] = heavy ? pk_reached(st, w0 * 32 + (e[k] & 2047)) : st.hold_min;
                }
                wave_lds_order();
#pragma unroll
                for (int k = 0; k < COMPACT_UNR; ++k) {
                    const int wi = (e[k] & 2047) >> 5, bit = e[k] & 31;
                    const bool heavy = (e[k] >> 11) >= st.hold_cls;
                    const bool held = heavy && !((hw[k] >> bit) & 1u) && reached[k] < st.hold_min;
                    if (heavy) heavy_w[wi] = 1;
                    if (held) atomicOr(&held_w[wi], 1u << bit);
                    my_dc += held;
                    const bool take = e[k] != 0 && !held;
                    const unsigned long long m = __ballot(take);
                    if (take) list[left + __popcll(m & lanes_below(lane))] = (unsigned short)e[k];
                    left += __popcll(m);
                }
            }
            n = left;
            wave_lds_order();
            stay = s_held[tid];
            if (s_heavy[tid]) st_coherent_u(st.bm[1] + w0 + lane, stay);
        }
        if (marks && !stay) st_coherent_u(st.bm[0] + w0 + lane, 0u);
        if (!__syncthreads_or(n)) continue;  // s_wc is clear, nothing was counted
        for (int i = lane; i < n; i += 64) atomicAdd(&wc[list[i] >> 11], 1);
        reserve_classes(s_wc, cnt_out);
        for (int i = lane; i < n; i += 64) {
            const int e = list[i], c = e >> 11;
            const long long v = w0 * 32 + (e & 2047);
            const unsigned t = ld_coherent_u(st.mflag + v);
            st_coherent_u(st.mflag + v, 0u);
            const long long qi = st.seg_off[c] + atomicAdd(&wc[c], 1);
            if (seg_ok(st.ctrl, qi, st.seg_off[c], st.seg_off[c + 1])) {
                st_coherent(q_out + qi, (int)v);
                st_coherent_u(qm_out + qi, t);
            }
            pairs += __popc(t);
        }
        __syncthreads();
        if (tid < WAVES * NCLS) s_wc[0][tid] = 0;  // the last loop counted in s_wc
        __syncthreads();
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) pairs += __shfl_xor(pairs, o);
    if (lane == 0 && pairs) atomicAdd(&s_pairs, pairs);
    __syncthreads();
    if (tid == 0 && s_pairs)
        atomicAdd((unsigned long long *)&st.ctrl->leaf[blockIdx.x % BAR_LEAVES].pairs, (unsigned long long)s_pairs);
    if (windowed || st.hold_cls) flush_deferred(st.ctrl, slot, my_dc, my_dm, &s_dc, &s_dm);
}

// Lane-bin bound of a packed expansion (see PACK_LANE_CLS); the other bins keep theirs.  A filtered
// expansion takes every class below PK_TILE_CLS as tiles.
__device__ __forceinline__ Cfg pk_cfg(Cfg c, bool filt) {
    if (filt) {
        c.b1 = PK_TILE_CLS;
        if (c.b2 < c.b1) c.b2 = c.b1;
        if (c.b3 < c.b1) c.b3 = c.b1;
    } else if (c.b1 > PACK_LANE_CLS) {
        c.b1 = PACK_LANE_CLS;
    }
    return c;
}

// WINDOW: a priority window is on.  Its compaction keeps 4 rows per lane group in flight, for which 3
// workgroups fit on a CU; without a window 2 are enough for code that is not reached, and 4 fit (with 2
// the window itself, 32 sources of a 2048^2 grid: 23.1 -> 24.0 ms; with 3 workgroups on a CU the packs
// without one, 32 sources of R-MAT s20: 5.0 -> 6.1 ms).
template <bool UNIT, bool WINDOW>
__global__ __launch_bounds__(WG) void k_pk_persistent(DevState st, SchedDev sp) {
    __shared__ ItemTables tb;
    __shared__ int s_tcol[WAVES][PK_TILE], s_tw[WAVES][PK_TILE];
    __shared__ int s_total;
    Ctrl *ctrl = st.ctrl;
    unsigned long long gen = 0;
    const unsigned nb = gridDim.x;
    long long t_prev = 0;
    // priority window: every workgroup computes the same sequence of thresholds
    int T = sp.delta > 0 ? sp.delta : NO_WINDOW;
    bool full = false;
    int pass = 0, win = 0;
    for (int it = 0;; ++it) {
        const int tid = phase_tid();
        int *q_cur = st.queue[it & 1];
        unsigned *qm_cur = st.qmask[it & 1];
        if (blockIdx.x == 0 && tid == 0) {
            long long now = (long long)wall_clock64();
            if (it > 0 && sp.trace && it - 1 < sp.trace_cap) sp.trace[it - 1].t_end = now;
            t_prev = now;
        }
        for (;;) {
            // every pass has counters of its own, as in k_persistent
            int *cnt_cur = st.cnt + (pass % 3) * NCLS;
            if (blockIdx.x == 0 && tid < NCLS) st_coherent(st.cnt + ((pass + 1) % 3) * NCLS + tid, 0);
            // the sums of a window, or of a pass (held vertices); the next ones' were last read before
            // the previous barrier
            const int sums = st.deferred ? win : pass;
            if (blockIdx.x == 0) deferred_clear(ctrl, (sums + 1) % 3);
            pk_compaction<WINDOW ? 4 : 2, true>(st, cnt_cur, q_cur, qm_cur, T, full, sums % 3);
            if (!grid_sync(ctrl, nb, gen)) return;
            pass++;
            if (tid < NCLS) {
                tb.cnt[tid] = ld_coherent(cnt_cur + tid);
                tb.seg[tid] = st.seg_off[tid];
            }
            __syncthreads();
            if (tid < 64) {
                const long long tot = frontier_size(tb.cnt);
                if (tid == 0) s_total = tot > 0x7FFFFFFF ? 0x7FFFFFFF : (int)tot;
            }
            __syncthreads();
            if (s_total > 0) {
                full = false;
                break;
            }
            // nothing queued: done unless pairs are kept back (by the window, which rises to the least
            // of them + delta, or held vertices, which the next pass takes)
            if (st.deferred && T == NO_WINDOW) break;
            int kept, mn;
            deferred_sums(ctrl, sums % 3, &kept, &mn);
            if (T == NO_WINDOW ? kept == 0 : mn == NO_WINDOW) break;
            if (T != NO_WINDOW) {
                T = mn > NO_WINDOW - sp.delta ? NO_WINDOW : mn + sp.delta;
                full = true;
                win++;
            }
        }
        const int total = s_total;
        if (total == 0 || (sp.max_iters > 0 && it >= sp.max_iters)) {
            if (blockIdx.x == 0 && tid == 0) {
                ctrl->iters = it;
                ctrl->done = total == 0 ? 1 : 0;
                if (total != 0) ctrl->error = NP_ERR_NOT_CONVERGED;
            }
            return;
        }
        Cfg cfg = decide(sp, tb.cnt, it);
        if (tid < 64) build_tables(tb, pk_cfg(cfg, false), TABLES_PACKED, (long long)nb * WAVES);
        if (blockIdx.x == 0 && tid < 64) {
            if (tid == 0) ctrl->frontier_total += total;
            record_trace(sp, it, cfg, tb.cnt, t_prev, ctrl);
        }
        __syncthreads();
        pk_expansion<UNIT, false>(st, PkFilt{}, q_cur, qm_cur, tb, s_tcol[tid >> 6], s_tw[tid >> 6], nullptr);
        if (!grid_sync(ctrl, nb, gen)) return;
    }
}

__global__ __launch_bounds__(WG) void k_pk_compact(DevState st, int it_off) {
    Ctrl *ctrl = st.ctrl;
    if (ld_coherent(&ctrl->done) || ld_coherent(&ctrl->error)) return;
    const int it = ld_coherent(&ctrl->it_base) + it_off;
    const int pass = ld_coherent(&ctrl->pass);
    const int T = ld_coherent(&ctrl->thresh);
    if (blockIdx.x == 0 && threadIdx.x < NCLS) st.cnt[((it + 2) % 3) * NCLS + threadIdx.x] = 0;
    const int sums = st.deferred ? ld_coherent(&ctrl->win) : pass;  // as in k_pk_persistent
    if (blockIdx.x == 0) deferred_clear(ctrl, (sums + 1) % 3);
    pk_compaction<4, false>(st, st.cnt + (it % 3) * NCLS, st.queue[it & 1], st.qmask[it & 1], T, ld_coherent(&ctrl->full) != 0,
                  sums % 3);
}

// Every vertex's bound, once: between the compaction and the decision that records the offsets (no
// distance changes in between, so every workgroup sees those offsets).  A launch of its own: inside
// the compaction, behind an untaken branch, it cost every compaction about 65 us on 16.8 M vertices.
__global__ __launch_bounds__(WG) void k_pk_bounds(DevState st) {
    __shared__ int s_off[PACK_MAX];
    __shared__ unsigned s_mask;
    Ctrl *ctrl = st.ctrl;
    if (ld_coherent(&ctrl->done) || ld_coherent(&ctrl->error) || ld_coherent(&ctrl->filt) != 1) return;
    if (threadIdx.x < 64) {
        const int j = threadIdx.x;
        const int d = j < (1 << st.kshift) ? ld_coherent(st.dist + j) : st.inf;  // the hub's row
        const unsigned m = (unsigned)__ballot(d < st.inf);
        if (j < PACK_MAX) s_off[j] = d < st.inf ? d : 0;
        if (j == 0) s_mask = m;
    }
    __syncthreads();
    for (long long v = (long long)blockIdx.x * WG + threadIdx.x; v < st.nslots; v += (long long)gridDim.x * WG)
    {
        int hi, lo;
        pk_row_bound(st, v, s_off, s_mask, 0u, &hi, &lo);
        st.bound[v] = (unsigned char)pk_bound_code(hi, st.fshift);
    }
}

// The packed expansion is a latency-bound gather: it is held to 64 VGPRs so that eight waves share
// each SIMD (C3 packed, graph drive: 41.7 -> 31.3 ms per solve, a few registers spilled).  The
// persistent kernel keeps the compiler's allocation: held to 64 it spills its compaction and
// window code, which made C3 faster (42.2 -> 37.2 ms) but the grid with a window slower
// (125 -> 155 ms), and the graph drive is the faster drive for both.
// Work of the queue the last compaction built (traced solves on the host-loop and graph drives):
// out-degrees of the queued vertices into Ctrl::edges_total, out-degree x queued sources into
// Ctrl::items_total.  Kept out of the compaction, where even the untaken counting branch cost
// the windowed grid 20 %.
__global__ __launch_bounds__(WG) void k_pk_count(DevState st, int it_off) {
    __shared__ long long s_pre[NCLS + 1];
    __shared__ int s_seg[NCLS];
    Ctrl *ctrl = st.ctrl;
    if (ld_coherent(&ctrl->done) || ld_coherent(&ctrl->error)) return;
    const int it = ld_coherent(&ctrl->it_base) + it_off;
    if (threadIdx.x < NCLS) s_seg[threadIdx.x] = st.seg_off[threadIdx.x];
    if (threadIdx.x == 0) {
        int lc[NCLS];
        for (int c = 0; c < NCLS; ++c) lc[c] = ld_coherent(st.cnt + (it % 3) * NCLS + c);
        sol_prefix(lc, 1, NCLS, s_pre);
    }
    __syncthreads();
    const long long total = s_pre[NCLS];
    const int *q = st.queue[it & 1];
    const unsigned *qm = st.qmask[it & 1];
    unsigned long long edges = 0, items = 0;
    for (long long i = (long long)blockIdx.x * WG + threadIdx.x; i < total; i += (long long)gridDim.x * WG) {
        const int c = find_class(s_pre, i);
        const long long qi = s_seg[c] + (i - s_pre[c]);
        const int u = ld_coherent(q + qi);
        const unsigned d = (unsigned)(st.row[u + 1] - st.row[u]);
        edges += d;
        items += (unsigned long long)d * __popc(ld_coherent_u(qm + qi));
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        edges += __shfl_xor(edges, o);
        items += __shfl_xor(items, o);
    }
    if (lane_id() == 0 && edges) {
        atomicAdd((unsigned long long *)&ctrl->edges_total, edges);
        atomicAdd((unsigned long long *)&ctrl->items_total, items);
    }
}

// BOUND: the state has a bound filter (one more set of bodies; without it the kernel stays as small
// as it was, which the windowed grid's expansion shows: 2 % of its solve).
template <bool UNIT, bool BOUND>
__global__ __launch_bounds__(WG) __attribute__((amdgpu_waves_per_eu(8))) void k_pk_expand(DevState st, int it_off) {
    __shared__ ItemTables tb;
    constexpr int SLICE = BOUND ? PK_SLICE : PK_TILE;
    __shared__ int s_tcol[WAVES][SLICE], s_tw[WAVES][SLICE];
    __shared__ unsigned char s_town[BOUND ? WAVES : 1][BOUND ? PK_SLICE : 1];
    __shared__ int s_off[PACK_MAX];
    Ctrl *ctrl = st.ctrl;
    if (ld_coherent(&ctrl->done) || ld_coherent(&ctrl->error) || ld_coherent(&ctrl->skip)) return;
    const int it = ld_coherent(&ctrl->it_base) + it_off;
    const bool filt = BOUND && ld_coherent(&ctrl->filt) == 2;
    if (threadIdx.x < NCLS) {
        tb.cnt[threadIdx.x] = ld_coherent(st.cnt + (it % 3) * NCLS + threadIdx.x);
        tb.seg[threadIdx.x] = st.seg_off[threadIdx.x];
    }
    __syncthreads();
    if (threadIdx.x < 64) {
        Cfg cfg = make_cfg(ld_coherent(&ctrl->cfg_level), ld_coherent(&ctrl->cfg_klo),
                           ld_coherent(&ctrl->cfg_khi));
        build_tables(tb, pk_cfg(cfg, filt), filt ? TABLES_FILTERED : TABLES_PACKED, (long long)gridDim.x * WAVES);
    }
    if (filt && threadIdx.x < PACK_MAX) s_off[threadIdx.x] = ld_coherent(ctrl->foff + threadIdx.x);
    __syncthreads();
    const PkFilt pf{s_off, filt ? ld_coherent_u(&ctrl->fmask) : 0u};
    int *tcol = s_tcol[threadIdx.x >> 6], *tw = s_tw[threadIdx.x >> 6];
    unsigned char *town = s_town[BOUND ? threadIdx.x >> 6 : 0];
    if (BOUND && filt) pk_expansion<UNIT, BOUND>(st, pf, st.queue[it & 1], st.qmask[it & 1], tb, tcol, tw, town);
    else pk_expansion<UNIT, false>(st, pf, st.queue[it & 1], st.qmask[it & 1], tb, tcol, tw, town);
}

__global__ void k_pk_init_sources(DevState st, const int *srcs, int nsrc, int T0) {
    if (blockIdx.x != 0) return;
    if (threadIdx.x == 0) {
        st.ctrl->thresh = T0;
    }
    for (int k = 0; k < 3; ++k) deferred_clear(st.ctrl, k);
    __syncthreads();
    for (int i = threadIdx.x; i < nsrc; i += blockDim.x) {
        const int v = srcs[i];
        st.dist[((long long)v << st.kshift) + i] = 0;
        if (st.cls[v] == 0) continue;
        atomicOr(&st.mflag[v], 1u << i);
        st_coherent_b(pk_mark(st, v), 1);
    }
}

// Every source's distances of a pack, in original vertex ids, in one pass over the rows: a thread
// reads one vertex's row (2^KS consecutive distances, a random row when renumbered) and the wave
// stores 64 consecutive vertices of one source after another.  One source at a time re-read every
// row per source.  16 sources of 16.8 M vertices (1 GB of rows), solve and all results: 29.5 ms with
// a pass per source, 26.5 with this one; 32 sources of 4.2 M vertices 39.0 -> 35.6.
template <int KS>
__global__ __launch_bounds__(WG) void k_unpack(const int *dist, UnpackTo to, const int *old2new, int n, int *out) {
    for (long long v = (long long)blockIdx.x * WG + threadIdx.x; v < n; v += (long long)gridDim.x * WG) {
        const long long r = old2new ? old2new[v] : v;
        const int *row = dist + (r << KS);
        int d[1 << KS];
        if (KS >= 2) {
#pragma unroll
            for (int q = 0; q < (1 << KS) / 4; ++q) {
                const int4 x = ((const int4 *)row)[q];
                d[4 * q] = x.x; d[4 * q + 1] = x.y; d[4 * q + 2] = x.z; d[4 * q + 3] = x.w;
            }
        } else {
#pragma unroll
            for (int j = 0; j < (1 << KS); ++j) d[j] = row[j];
        }
#pragma unroll
        for (int j = 0; j < (1 << KS); ++j)
            if (j < to.count && to.off[j] >= 0) out[to.off[j] + v] = d[j];
    }
}

// Results of a concatenated part's renumbered instances, in original vertex ids, in one launch (a
// launch and a wait per instance cost more than small graphs' results): a workgroup's slots belong
// to one instance (slots are padded to 2^LUT_SHIFT per instance).
__global__ __launch_bounds__(WG) void k_unpermute_parts(const int *dist, const int *lut, const ConcatOut *parts,
                                                        long long nslots, int *out) {
    static_assert((1 << LUT_SHIFT) % WG == 0, "a workgroup must lie in one instance");
    for (long long base = (long long)blockIdx.x * WG; base < nslots; base += (long long)gridDim.x * WG) {
        const ConcatOut p = parts[lut[base >> LUT_SHIFT]];
        const long long v = base + threadIdx.x - p.base;
        if (p.old2new && v < p.n) out[p.off + v] = dist[p.base + p.old2new[v]];
    }
}

// ------------------------------------------------------------------------------------
// setup kernels
// ------------------------------------------------------------------------------------
__global__ void k_fill_i32(int *p, long long n, int v) {
    for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n;
         i += (long long)gridDim.x * blockDim.x)
        p[i] = v;
}
__global__ void k_fill_u32(unsigned *p, long long n, unsigned v) {
    for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n;
         i += (long long)gridDim.x * blockDim.x)
        p[i] = v;
}

__global__ __launch_bounds__(WG) void k_degree_class(const int *row, int n, unsigned char *cls,
                                                     int *hist) {
    __shared__ int h[NCLS];
    if (threadIdx.x < NCLS) h[threadIdx.x] = 0;
    __syncthreads();
    for (long long v = (long long)blockIdx.x * WG + threadIdx.x; v < n; v += (long long)gridDim.x * WG) {
        int c = deg_class(row[v + 1] - row[v]);
        cls[v] = (unsigned char)c;
        atomicAdd(&h[c], 1);
    }
    __syncthreads();
    if (threadIdx.x < NCLS && h[threadIdx.x]) atomicAdd(&hist[threadIdx.x], h[threadIdx.x]);
}

// CSR well-formedness, so that no kernel can index outside the arrays:
// row[0] == 0, row non-decreasing, row[n] == m, 0 <= col < n.  out[0] counts violations;
// with weights (w non-null) out[1] counts negative weights and out[2] receives the largest
// weight (out[] starts at 0).
__global__ void k_validate_csr(const int *row, const int *col, const int *w, int n, long long m, int *out) {
    int local = 0, neg = 0, wmax = 0;
    const long long stride = (long long)gridDim.x * blockDim.x;
    for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i <= n; i += stride) {
        int r = row[i];
        if (i == 0 && r != 0) local++;
        if (i == n && (long long)r != m) local++;
        if (i < n && row[i + 1] < r) local++;
    }
    for (long long e = (long long)blockIdx.x * blockDim.x + threadIdx.x; e < m; e += stride) {
        int c = col[e];
        if (c < 0 || c >= n) local++;
        if (w) {
            int x = w[e];
            if (x < 0) neg++;
            wmax = max(wmax, x);
        }
    }
    if (local) atomicAdd(&out[0], local);
    if (neg) atomicAdd(&out[1], neg);
    if (wmax) atomicMax(&out[2], wmax);
}

// Largest finite value of a solve's distance buffer (count entries): atomicMax into *out,
// which starts at 0.  A stream of 16-byte loads, MAXF_UNR in flight per lane (the entries before the
// first aligned address and after the last whole one are workgroup 0's), and one atomic per
// workgroup: 16,384 wavefronts' atomics on *out took turns for longer than the stream.  537 MB:
// 0.28 -> 0.092 ms, 5.8 TB/s; one solve of a 2048^2 grid (16.8 MB) 3.83 -> 3.72.
constexpr int MAXF_UNR = 4;
constexpr int MAXF_WGS = 1024;
__global__ __launch_bounds__(WG) void k_max_finite(const int *dist, long long count, int inf, int *out) {
    __shared__ int s_mx;
    if (threadIdx.x == 0) s_mx = 0;
    __syncthreads();
    int mx = 0;
    auto take = [&](int d) { if (d != inf) mx = max(mx, d); };
    const long long skip = (long long)((16 - ((size_t)dist & 15)) & 15) / 4;
    const long long head = skip < count ? skip : count, n4 = (count - head) / 4;
    const int4 *body = (const int4 *)(dist + head);
    if (blockIdx.x == 0) {
        if (threadIdx.x < head) take(dist[threadIdx.x]);
        const long long t = head + 4 * n4 + threadIdx.x;
        if (t < count) take(dist[t]);
    }
    const long long step = (long long)gridDim.x * WG;
    for (long long i = (long long)blockIdx.x * WG + threadIdx.x; i < n4; i += step * MAXF_UNR) {
        int4 x[MAXF_UNR];
#pragma unroll
        for (int k = 0; k < MAXF_UNR; ++k) x[k] = i + k * step < n4 ? body[i + k * step] : int4{0, 0, 0, 0};
#pragma unroll
        for (int k = 0; k < MAXF_UNR; ++k) { take(x[k].x); take(x[k].y); take(x[k].z); take(x[k].w); }
    }
    for (int o = 32; o > 0; o >>= 1) mx = max(mx, __shfl_xor(mx, o));
    if (lane_id() == 0 && mx) atomicMax(&s_mx, mx);
    __syncthreads();
    if (threadIdx.x == 0 && s_mx) atomicMax(out, s_mx);
}

// Relaxations that int32 distances below inf cannot hold: an edge u -> v whose tail is
// reached, whose target is still at inf and with dist[u] + w >= inf (the relaxation
// alt < dist[v] is false there, so the target stays unreached although a path exists).
// Counts them into *bad.  Every layout: one distance per slot (BATCH: slots of
// concatenated instances) or rows of 2^kshift sources per vertex.
template <bool BATCH>
__global__ __launch_bounds__(WG) void k_dist_escape(DevState st, int *bad) {
    const int ks = st.kshift < 0 ? 0 : st.kshift;
    const long long total = st.nslots << ks;
    int local = 0;
    for (long long i = (long long)blockIdx.x * WG + threadIdx.x; i < total; i += (long long)gridDim.x * WG) {
        const int du = st.dist[i];
        if (du == st.inf) continue;
        const int slot = (int)(i >> ks);
        const int lane = (int)(i & ((1 << ks) - 1));
        int B = 0, VB = 0;
        decode<BATCH>(st, slot, B, VB);
        const int v = slot - B;
        for (int e = st.row[VB + v], e1 = st.row[VB + v + 1]; e < e1; ++e) {
            const long long t = (long long)(B + st.col[e]);
            if (st.dist[(t << ks) + lane] == st.inf && (long long)du + st.w[e] >= (long long)st.inf) local++;
        }
    }
    if (local) atomicAdd(bad, local);
}

template <bool PUSH>
__global__ void k_init_sources(DevState st, const int *srcs, int nsrc, int T0) {
    if (blockIdx.x != 0) return;
    if (threadIdx.x == 0) {
        st.ctrl->thresh = T0;
    }
    for (int k = 0; k < 3; ++k) deferred_clear(st.ctrl, k);
    for (int i = threadIdx.x; i < nsrc; i += blockDim.x) {
        int slot = srcs[i];
        st.dist[slot] = 0;
        int c = st.cls[slot];
        if (c == 0) continue;
        atomicOr(&st.bm[0][slot >> 5], 1u << (slot & 31));
        if (PUSH) {
            int p = atomicAdd(&st.cnt[c], 1);  // counters of iteration 0
            st.queue[0][st.seg_off[c] + p] = slot;
        }
    }
}

__global__ __launch_bounds__(WG) void k_reached_work(const int *row, const int *dist, int n, int inf,
                                                     unsigned long long *out2) {
    __shared__ unsigned long long sa[WG], sb[WG];
    unsigned long long a = 0, b = 0;
    for (long long v = (long long)blockIdx.x * WG + threadIdx.x; v < n; v += (long long)gridDim.x * WG) {
        if (dist[v] != inf) { a++; b += (unsigned long long)(row[v + 1] - row[v]); }
    }
    sa[threadIdx.x] = a; sb[threadIdx.x] = b;
    __syncthreads();
    for (int o = WG / 2; o > 0; o >>= 1) {
        if (threadIdx.x < o) { sa[threadIdx.x] += sa[threadIdx.x + o]; sb[threadIdx.x] += sb[threadIdx.x + o]; }
        __syncthreads();
    }
    if (threadIdx.x == 0) { atomicAdd(&out2[0], sa[0]); atomicAdd(&out2[1], sb[0]); }
}

__global__ void k_rebase_row(const int *row, int n, int add, int *out) {
    for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i <= n;
         i += (long long)gridDim.x * blockDim.x)
        out[i] = row[i] + add;
}
__global__ void k_fill_lut(int *lut, long long first, long long count, int inst) {
    for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < count;
         i += (long long)gridDim.x * blockDim.x)
        lut[first + i] = inst;
}
__global__ void k_copy_u8(const unsigned char *src, unsigned char *dst, long long n) {
    for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n;
         i += (long long)gridDim.x * blockDim.x)
        dst[i] = src[i];
}

// ------------------------------------------------------------------------------------
// scheduler MLP (fp32): forward, per-sample backward, per-parameter reduction, Adam
// ------------------------------------------------------------------------------------
constexpr int H = 32, NO = 5, NI = NP_MLP_NIN;
// per-sample scratch: x copy not needed; h1, h2 (post-ReLU), g1, g2 (pre-activation grads),
// go (output grads), loss
constexpr int PER_SAMPLE = H + H + H + H + NO + 1;

__device__ __forceinline__ void mlp_fwd_sample(const float *p, const float *x, float *a1, float *h1,
                                               float *a2, float *h2, float *o) {
    const float *W1 = p, *b1 = W1 + H * NI, *W2 = b1 + H, *b2 = W2 + H * H, *W3 = b2 + H,
                *b3 = W3 + NO * H;
    for (int j = 0; j < H; ++j) {
        float a = b1[j];
        for (int i = 0; i < NI; ++i) a += W1[j * NI + i] * x[i];
        a1[j] = a; h1[j] = a > 0.f ? a : 0.f;
    }
    for (int j = 0; j < H; ++j) {
        float a = b2[j];
        for (int i = 0; i < H; ++i) a += W2[j * H + i] * h1[i];
        a2[j] = a; h2[j] = a > 0.f ? a : 0.f;
    }
    for (int j = 0; j < NO; ++j) {
        float a = b3[j];
        for (int i = 0; i < H; ++i) a += W3[j * H + i] * h2[i];
        o[j] = a;
    }
}

__global__ void k_mlp_forward(const float *p, const float *x, int batch, float *out) {
    int s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= batch) return;
    float a1[H], h1[H], a2[H], h2[H], o[NO];
    mlp_fwd_sample(p, x + (long long)s * NI, a1, h1, a2, h2, o);
    for (int j = 0; j < NO; ++j) out[(long long)s * NO + j] = o[j];
}

// One thread per sample: forward, softmax-CE + lam * squared error, and the gradients of
// the pre-activations (stored for the reduction).
__global__ void k_mlp_sample_grad(const float *p, const float *x, const int *label,
                                  const float *target, int batch, float lam, float *work) {
    int s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= batch) return;
    const float *W2 = p + H * NI + H, *W3 = W2 + H * H + H;
    float a1[H], h1[H], a2[H], h2[H], o[NO], go[NO];
    mlp_fwd_sample(p, x + (long long)s * NI, a1, h1, a2, h2, o);
    const float inv = 1.0f / (float)batch;
    float mx = fmaxf(o[0], fmaxf(o[1], o[2]));
    float e0 = expf(o[0] - mx), e1 = expf(o[1] - mx), e2 = expf(o[2] - mx);
    float z = e0 + e1 + e2;
    float pr[3] = {e0 / z, e1 / z, e2 / z};
    int lb = label[s];
    float loss = -logf(fmaxf(pr[lb], 1e-30f));
    for (int j = 0; j < 3; ++j) go[j] = (pr[j] - (j == lb ? 1.f : 0.f)) * inv;
    for (int j = 0; j < 2; ++j) {
        float d = o[3 + j] - target[(long long)s * 2 + j];
        loss += lam * d * d;
        go[3 + j] = 2.f * lam * d * inv;
    }
    float *wk = work + (long long)s * PER_SAMPLE;
    float *wh1 = wk, *wh2 = wk + H, *wg1 = wk + 2 * H, *wg2 = wk + 3 * H, *wgo = wk + 4 * H;
    float g2[H];
    for (int i = 0; i < H; ++i) {
        float g = 0.f;
        for (int j = 0; j < NO; ++j) g += W3[j * H + i] * go[j];
        g2[i] = a2[i] > 0.f ? g : 0.f;
    }
    for (int i = 0; i < H; ++i) {
        float g = 0.f;
        for (int j = 0; j < H; ++j) g += W2[j * H + i] * g2[j];
        wg1[i] = a1[i] > 0.f ? g : 0.f;
        wh1[i] = h1[i];
        wh2[i] = h2[i];
        wg2[i] = g2[i];
    }
    for (int j = 0; j < NO; ++j) wgo[j] = go[j];
    wk[4 * H + NO] = loss * inv;
}

// One thread per parameter: sum of the per-sample contributions (deterministic order).
__global__ void k_mlp_reduce(const float *x, int batch, const float *work, float *grad,
                             float *loss) {
    int pidx = blockIdx.x * blockDim.x + threadIdx.x;
    if (pidx > NP_MLP_NPARAM) return;
    if (pidx == NP_MLP_NPARAM) {
        float l = 0.f;
        for (int s = 0; s < batch; ++s) l += work[(long long)s * PER_SAMPLE + 4 * H + NO];
        loss[0] = l;
        return;
    }
    // locate the parameter
    int q = pidx;
    float acc = 0.f;
    if (q < H * NI) {  // W1[j][i] += g1[j] * x[i]
        int j = q / NI, i = q % NI;
        for (int s = 0; s < batch; ++s) acc += work[(long long)s * PER_SAMPLE + 2 * H + j] * x[(long long)s * NI + i];
    } else if ((q -= H * NI) < H) {  // b1
        for (int s = 0; s < batch; ++s) acc += work[(long long)s * PER_SAMPLE + 2 * H + q];
    } else if ((q -= H) < H * H) {  // W2[j][i] += g2[j] * h1[i]
        int j = q / H, i = q % H;
        for (int s = 0; s < batch; ++s) acc += work[(long long)s * PER_SAMPLE + 3 * H + j] * work[(long long)s * PER_SAMPLE + i];
    } else if ((q -= H * H) < H) {  // b2
        for (int s = 0; s < batch; ++s) acc += work[(long long)s * PER_SAMPLE + 3 * H + q];
    } else if ((q -= H) < NO * H) {  // W3[j][i] += go[j] * h2[i]
        int j = q / H, i = q % H;
        for (int s = 0; s < batch; ++s) acc += work[(long long)s * PER_SAMPLE + 4 * H + j] * work[(long long)s * PER_SAMPLE + H + i];
    } else {  // b3
        q -= NO * H;
        for (int s = 0; s < batch; ++s) acc += work[(long long)s * PER_SAMPLE + 4 * H + q];
    }
    grad[pidx] = acc;
}

__global__ void k_adam(float *p, const float *g, float *m, float *v, int n, float lr, float b1,
                       float b2, float eps, float c1, float c2) {
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    float gi = g[i];
    float mi = b1 * m[i] + (1.f - b1) * gi;
    float vi = b2 * v[i] + (1.f - b2) * gi * gi;
    m[i] = mi; v[i] = vi;
    p[i] -= lr * (mi / c1) / (sqrtf(vi / c2) + eps);
}

// ------------------------------------------------------------------------------------
// launchers
// ------------------------------------------------------------------------------------
static int grid_for(long long n, int block) {
    long long g = (n + block - 1) / block;
    if (g < 1) g = 1;
    if (g > 65536) g = 65536;
    return (int)g;
}

hipError_t launch_fill_i32(int *p, long long n, int v, hipStream_t s) {
    if (n <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_fill_i32, dim3(grid_for(n, 256)), dim3(256), 0, s, p, n, v);
    return hipGetLastError();
}
hipError_t launch_fill_u32(unsigned *p, long long n, unsigned v, hipStream_t s) {
    if (n <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_fill_u32, dim3(grid_for(n, 256)), dim3(256), 0, s, p, n, v);
    return hipGetLastError();
}
hipError_t launch_validate_csr(const int *row, const int *col, const int *w, int n, long long m, int *out3,
                               hipStream_t s) {
    long long work = (long long)n + 1 > m ? (long long)n + 1 : m;
    hipLaunchKernelGGL(k_validate_csr, dim3(grid_for(work, 256) > 4096 ? 4096 : grid_for(work, 256)),
                       dim3(256), 0, s, row, col, w, n, m, out3);
    return hipGetLastError();
}

hipError_t launch_max_finite(const DevState &st, int *out, hipStream_t s) {
    const long long count = st.nslots << (st.kshift < 0 ? 0 : st.kshift);
    hipError_t e = launch_fill_i32(out, 1, 0, s);
    if (e != hipSuccess || count <= 0) return e;
    const int g = (int)std::min<long long>(MAXF_WGS, (count / 4 + WG - 1) / WG + 1);
    hipLaunchKernelGGL(k_max_finite, dim3(g), dim3(WG), 0, s, (const int *)st.dist, count, st.inf, out);
    return hipGetLastError();
}

hipError_t launch_dist_escape(const DevState &st, bool batch, int *bad, hipStream_t s) {
    const long long count = st.nslots << (st.kshift < 0 ? 0 : st.kshift);
    hipError_t e = launch_fill_i32(bad, 1, 0, s);
    if (e != hipSuccess || count <= 0) return e;
    const dim3 grid(grid_for(count, WG) > 4096 ? 4096 : grid_for(count, WG));
    if (batch) hipLaunchKernelGGL(k_dist_escape<true>, grid, dim3(WG), 0, s, st, bad);
    else hipLaunchKernelGGL(k_dist_escape<false>, grid, dim3(WG), 0, s, st, bad);
    return hipGetLastError();
}
hipError_t launch_degree_class(const int *row, int n, unsigned char *cls, int *hist, hipStream_t s) {
    if (n <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_degree_class, dim3(grid_for(n, WG)), dim3(WG), 0, s, row, n, cls, hist);
    return hipGetLastError();
}
hipError_t launch_init_solve(const DevState &st, const int *d_src_slots, int nsrc, int push, int delta,
                             hipStream_t s) {
    const int T0 = (!push && delta > 0) ? delta : NO_WINDOW;
    hipError_t e;
    if ((e = launch_fill_i32(st.dist, st.nslots, st.inf, s)) != hipSuccess) return e;
    if ((e = launch_fill_u32(st.bm[0], st.nwords, 0u, s)) != hipSuccess) return e;
    if ((e = launch_fill_u32(st.bm[1], st.nwords, 0u, s)) != hipSuccess) return e;
    if ((e = launch_fill_i32(st.cnt, 3 * NCLS, 0, s)) != hipSuccess) return e;
    if (st.sbcnt && (e = launch_fill_i32(st.sbcnt, 3, 0, s)) != hipSuccess) return e;
    if ((e = launch_fill_i32((int *)st.ctrl, (long long)(sizeof(Ctrl) / sizeof(int)), 0, s)) != hipSuccess)
        return e;
    if (push) hipLaunchKernelGGL(k_init_sources<true>, dim3(1), dim3(256), 0, s, st, d_src_slots, nsrc, T0);
    else hipLaunchKernelGGL(k_init_sources<false>, dim3(1), dim3(256), 0, s, st, d_src_slots, nsrc, T0);
    return hipGetLastError();
}
hipError_t launch_reached_work(const int *row, const int *dist, int n, int inf,
                               unsigned long long *out2, hipStream_t s) {
    hipError_t e = launch_fill_u32((unsigned *)out2, 4, 0u, s);
    if (e != hipSuccess) return e;
    if (n <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_reached_work, dim3(grid_for(n, WG) > 2048 ? 2048 : grid_for(n, WG)), dim3(WG),
                       0, s, row, dist, n, inf, out2);
    return hipGetLastError();
}
hipError_t launch_rebase_row(const int *row, int n, int add, int *out, hipStream_t s) {
    hipLaunchKernelGGL(k_rebase_row, dim3(grid_for((long long)n + 1, 256)), dim3(256), 0, s, row, n, add, out);
    return hipGetLastError();
}
hipError_t launch_fill_lut(int *lut, long long first, long long count, int inst, hipStream_t s) {
    if (count <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_fill_lut, dim3(grid_for(count, 256)), dim3(256), 0, s, lut, first, count, inst);
    return hipGetLastError();
}
hipError_t launch_copy_cls(const unsigned char *src, unsigned char *dst, long long n, hipStream_t s) {
    if (n <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_copy_u8, dim3(grid_for(n, 256)), dim3(256), 0, s, src, dst, n);
    return hipGetLastError();
}

template <bool B, bool U>
static const void *persistent_fn(bool push, bool solo) {
    if (push) return (const void *)&k_persistent<B, U, true, false>;
    return solo ? (const void *)&k_persistent<B, U, false, true> : (const void *)&k_persistent<B, U, false, false>;
}

static const void *pick_persistent(bool batch, bool unit, bool push, bool solo) {
    if (batch) return unit ? persistent_fn<true, true>(push, solo) : persistent_fn<true, false>(push, solo);
    return unit ? persistent_fn<false, true>(push, solo) : persistent_fn<false, false>(push, solo);
}

static const void *pick_packed(bool unit, bool window) {
    if (window) return unit ? (const void *)&k_pk_persistent<true, true> : (const void *)&k_pk_persistent<false, true>;
    return unit ? (const void *)&k_pk_persistent<true, false> : (const void *)&k_pk_persistent<false, false>;
}

int persistent_max_wgs_per_cu(bool batch, bool unit, bool push, bool packed, bool solo, bool window) {
    int nb = 0;
    const void *fn = packed ? pick_packed(unit, window) : pick_persistent(batch, unit, push, solo);
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, fn, WG, 0) != hipSuccess) return 0;
    return nb;
}

hipError_t launch_persistent(const DevState &st, const SchedDev &sp, bool batch, bool unit, int wgs,
                             hipStream_t s) {
    DevState a0 = st;
    SchedDev a1 = sp;
    void *args[] = {&a0, &a1};
    const void *fn = st.kshift >= 0 ? pick_packed(unit, sp.delta > 0) : pick_persistent(batch, unit, sp.push != 0, sp.solo != 0);
    return hipLaunchCooperativeKernel(fn, dim3(wgs), dim3(WG), args, 0, s);
}

hipError_t launch_compact(const DevState &st, int it_off, bool batch, int wgs, hipStream_t s) {
    (void)batch;
    // a workgroup per tile, up to the ones that compact_words has in view (a
    // workgroup per 8,192 vertices left 8 of them on 65,536, each with 8 tiles in turn: 4 sources of
    // R-MAT s16 1.04 -> 0.91 ms, of grid 256^2 1.91 -> 1.41, one of ER 65,536 0.79 -> 0.66)
    const long long tile = (long long)WAVES * compact_words(st.nwords, wgs, st.deferred != nullptr);
    const int g = (int)std::min<long long>(std::max<long long>((st.nwords + tile - 1) / tile, 1), wgs);
    if (st.kshift >= 0) {
        hipLaunchKernelGGL(k_pk_compact, dim3(g), dim3(WG), 0, s, st, it_off);
        if (st.bound) hipLaunchKernelGGL(k_pk_bounds, dim3(wgs), dim3(WG), 0, s, st);
        if (st.count_work) hipLaunchKernelGGL(k_pk_count, dim3(wgs), dim3(WG), 0, s, st, it_off);
    } else {
        hipLaunchKernelGGL(k_compact, dim3(g), dim3(WG), 0, s, st, it_off);
    }
    return hipGetLastError();
}
hipError_t launch_init_packed(const DevState &st, const int *d_srcs, int nsrc, int delta, hipStream_t s) {
    if (st.kshift < 0 || nsrc < 1 || nsrc > (1 << st.kshift) || nsrc > PACK_MAX) return hipErrorInvalidValue;
    hipError_t e;
    if ((e = launch_fill_i32(st.dist, st.nslots << st.kshift, st.inf, s)) != hipSuccess) return e;
    if ((e = launch_fill_u32(st.bm[0], st.nwords, 0u, s)) != hipSuccess) return e;
    if (st.hold_cls && (e = launch_fill_u32(st.bm[1], st.nwords, 0u, s)) != hipSuccess) return e;
    if ((e = launch_fill_u32(st.mflag, st.nslots, 0u, s)) != hipSuccess) return e;
    if (st.deferred && (e = launch_fill_u32(st.deferred, st.nslots, 0u, s)) != hipSuccess) return e;
    if (st.bound && (e = launch_fill_u32((unsigned *)st.bound, (st.nslots + 3) / 4, ~0u, s)) != hipSuccess) return e;
    if ((e = launch_fill_i32(st.cnt, 3 * NCLS, 0, s)) != hipSuccess) return e;
    if (st.sbcnt && (e = launch_fill_i32(st.sbcnt, 3, 0, s)) != hipSuccess) return e;
    if ((e = launch_fill_i32((int *)st.ctrl, (long long)(sizeof(Ctrl) / sizeof(int)), 0, s)) != hipSuccess)
        return e;
    hipLaunchKernelGGL(k_pk_init_sources, dim3(1), dim3(64), 0, s, st, d_srcs, nsrc, delta > 0 ? delta : NO_WINDOW);
    return hipGetLastError();
}
hipError_t launch_unpack(const int *dist, int kshift, const UnpackTo &to, const int *old2new, int n, int *out,
                         hipStream_t s) {
    if (n <= 0) return hipSuccess;
    const dim3 grid(grid_for(n, WG));
#define NP_UNPACK(K) hipLaunchKernelGGL(k_unpack<K>, grid, dim3(WG), 0, s, dist, to, old2new, n, out)
    switch (kshift) {
    case 0: NP_UNPACK(0); break;
    case 1: NP_UNPACK(1); break;
    case 2: NP_UNPACK(2); break;
    case 3: NP_UNPACK(3); break;
    case 4: NP_UNPACK(4); break;
    case 5: NP_UNPACK(5); break;
    default: return hipErrorInvalidValue;
    }
#undef NP_UNPACK
    return hipGetLastError();
}
hipError_t launch_unpermute_parts(const int *dist, const int *lut, const ConcatOut *parts, long long nslots, int *out,
                                  hipStream_t s) {
    if (nslots <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_unpermute_parts, dim3(grid_for(nslots, WG)), dim3(WG), 0, s, dist, lut, parts, nslots, out);
    return hipGetLastError();
}
hipError_t launch_decide(const DevState &st, const SchedDev &sp, int it_off, hipStream_t s) {
    hipLaunchKernelGGL(k_decide, dim3(1), dim3(WG), 0, s, st, sp, it_off);
    return hipGetLastError();
}
// The expansion of the reference's other schedules (single-source, scan frontier).
static hipError_t launch_scheme(const DevState &st, const SchedDev &sp, int it_off, bool unit, int wgs,
                                hipStream_t s) {
    const SolBufs sb{st.sbuf, st.sbcnt};
#define NP_SOL(M) do { if (unit) hipLaunchKernelGGL((k_sol_parent<M, true>), dim3(wgs), dim3(WG), 0, s, st, sb, it_off); \
                       else hipLaunchKernelGGL((k_sol_parent<M, false>), dim3(wgs), dim3(WG), 0, s, st, sb, it_off); } while (0)
    switch (sp.scheme) {
    case NP_SCHEME_THREAD: NP_SOL(SOL_THREAD); break;
    case NP_SCHEME_DUAL_QUEUE:
        NP_SOL(SOL_DUAL);
        if (unit) hipLaunchKernelGGL(k_sol_heavy<true>, dim3(wgs), dim3(WG), 0, s, st, it_off);
        else hipLaunchKernelGGL(k_sol_heavy<false>, dim3(wgs), dim3(WG), 0, s, st, it_off);
        break;
    case NP_SCHEME_LDS_BUFFER: NP_SOL(SOL_LDS); break;
    case NP_SCHEME_GLOBAL_BUFFER:
        NP_SOL(SOL_GLOBAL);
        if (unit) hipLaunchKernelGGL(k_sol_drain<true>, dim3(wgs), dim3(WG), 0, s, st, sb, it_off);
        else hipLaunchKernelGGL(k_sol_drain<false>, dim3(wgs), dim3(WG), 0, s, st, sb, it_off);
        break;
    case NP_SCHEME_WAVE_NESTED: NP_SOL(SOL_WAVE); break;
    case NP_SCHEME_WG_NESTED: NP_SOL(SOL_WGLIST); break;
    case NP_SCHEME_BFS_HIER: hipLaunchKernelGGL(k_bfs_hier, dim3(wgs), dim3(WG), 0, s, st, it_off); break;
    default: return hipErrorInvalidValue;
    }
#undef NP_SOL
    return hipGetLastError();
}

hipError_t launch_bfs_flat(const DevState &st, int level, int *changed, int wgs, hipStream_t s) {
    hipLaunchKernelGGL(k_bfs_flat, dim3(wgs), dim3(WG), 0, s, st.row, st.col, st.dist, (int)st.nslots, level,
                       changed);
    return hipGetLastError();
}

hipError_t launch_expand(const DevState &st, const SchedDev &sp, int it_off, bool batch, bool unit,
                         int wgs, hipStream_t s) {
    if (sp.scheme != NP_SCHEME_CONSOLIDATE) return launch_scheme(st, sp, it_off, unit, wgs, s);
    const bool push = sp.push != 0;
    if (st.kshift >= 0) {
#define NP_PK(U, B) hipLaunchKernelGGL((k_pk_expand<U, B>), dim3(wgs), dim3(WG), 0, s, st, it_off)
        if (unit) NP_PK(true, false);
        else if (st.bound) NP_PK(false, true);
        else NP_PK(false, false);
#undef NP_PK
        return hipGetLastError();
    }
#define NP_EXP(B, U, P) hipLaunchKernelGGL((k_expand<B, U, P>), dim3(wgs), dim3(WG), 0, s, st, it_off)
    if (batch) {
        if (unit) { if (push) NP_EXP(true, true, true); else NP_EXP(true, true, false); }
        else { if (push) NP_EXP(true, false, true); else NP_EXP(true, false, false); }
    } else {
        if (unit) { if (push) NP_EXP(false, true, true); else NP_EXP(false, true, false); }
        else { if (push) NP_EXP(false, false, true); else NP_EXP(false, false, false); }
    }
#undef NP_EXP
    return hipGetLastError();
}
hipError_t launch_advance(const DevState &st, int k, hipStream_t s) {
    hipLaunchKernelGGL(k_advance, dim3(1), dim3(64), 0, s, st, k);
    return hipGetLastError();
}
hipError_t launch_set_cfg(const DevState &st, int level, int klo, int khi, hipStream_t s) {
    hipLaunchKernelGGL(k_set_cfg, dim3(1), dim3(64), 0, s, st, level, klo, khi);
    return hipGetLastError();
}

hipError_t launch_mlp_forward(const float *p, const float *x, int batch, float *out, hipStream_t s) {
    if (batch <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_mlp_forward, dim3((batch + 127) / 128), dim3(128), 0, s, p, x, batch, out);
    return hipGetLastError();
}
size_t mlp_work_floats(int batch) { return (size_t)(batch > 0 ? batch : 1) * PER_SAMPLE; }
hipError_t launch_mlp_loss_grad(const float *p, const float *x, const int *label, const float *target,
                                int batch, float lam, float *work, float *grad, float *loss,
                                hipStream_t s) {
    if (batch <= 0) return hipErrorInvalidValue;
    hipLaunchKernelGGL(k_mlp_sample_grad, dim3((batch + 127) / 128), dim3(128), 0, s, p, x, label,
                       target, batch, lam, work);
    hipLaunchKernelGGL(k_mlp_reduce, dim3((NP_MLP_NPARAM + 1 + 127) / 128), dim3(128), 0, s, x, batch,
                       work, grad, loss);
    return hipGetLastError();
}
hipError_t launch_adam(float *p, const float *grad, float *m, float *v, int n, float lr, float b1,
                       float b2, float eps, int step, hipStream_t s) {
    float c1 = 1.f - powf(b1, (float)step), c2 = 1.f - powf(b2, (float)step);
    hipLaunchKernelGGL(k_adam, dim3((n + 255) / 256), dim3(256), 0, s, p, grad, m, v, n, lr, b1, b2, eps,
                       c1, c2);
    return hipGetLastError();
}

}  // namespace np
