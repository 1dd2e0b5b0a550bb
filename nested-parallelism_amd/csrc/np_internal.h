// np_internal.h -- internal interfaces between the C-ABI layer (np_api.cpp) and the
// HIP translation units (np_kernels.hip, np_gen.hip).  Not installed, not stable.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>
#include "np_common.h"
#include "../../include/np_sssp.h"

namespace np {

// Data passed between the lanes of one wavefront through LDS: the lanes run in step, so only the
// compiler has to keep the order of the accesses before and after (the barrier alone leaves it free
// to move memory accesses, the fence alone to let lanes run apart).
__device__ __forceinline__ void wave_lds_order() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}
// Device-scope stores and atomics of this wavefront are in memory before what follows it.  The
// fences keep the compiler from moving accesses across the wait (the wait alone would not); they
// name the workgroup because what they guard is itself device-scope: an agent-scope release would
// write the L2 back and invalidate it as well (PageRank's chunk counts, R-MAT s20: 2.8 -> 3.6 ms).
__device__ __forceinline__ void stores_done() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
    __builtin_amdgcn_s_waitcnt(0);
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
}

// Atomics on one cache line take turns (about 30 ns each, from whichever workgroup), so what every
// workgroup of a launch adds to is split over BAR_LEAVES lines, workgroup b on line b % BAR_LEAVES.
constexpr int BAR_LEAVES = 32;
struct alignas(128) BarLeaf {
    unsigned long long n;     // grid barrier: cumulative arrivals
    long long pairs;          // source-packed: queued (vertex, source) pairs, summed over iterations
    int dcnt[3];              // per compaction pass, a pack's per window (rotating): flagged vertices kept back
    int dmin[3];              // ... and the least distance among them
};

// Largest number of sources packed into one distance row.
constexpr int PACK_MAX = 32;

// Device-side control block of one solve.
struct Ctrl {
    BarLeaf leaf[BAR_LEAVES]; // per-line sums of the workgroups
    unsigned long long bar;   // grid barrier: cumulative leaf completions
    int error;                // NP_ERR_* raised by a kernel (0 = none)
    int done;                 // frontier emptied
    int iters;                // expansions performed
    int it_base;              // graph drive: iteration index of the captured chunk's first slot
    long long frontier_total; // sum of frontier sizes
    int cfg_level, cfg_klo, cfg_khi, cfg_pad;  // schedule decided for the next expansion
    int thresh;               // priority window: vertices with dist < thresh are expanded
    int pass;                 // compaction passes so far (host-loop / graph drives)
    int skip;                 // host-loop / graph drives: this slot only raised the window
    int full;                 // windowed pack: the next compaction looks at the deferred pairs too
    int win;                  // windowed pack: times the window has risen
    long long edges_total;    // source-packed: sum over iterations of the queued vertices' out-degrees
    long long items_total;    // source-packed: ... of out-degree x queued sources ((edge, source) items)
    int solo;                 // persistent drive: iterations of the last solo visit
    int filt;                 // source-packed bound filter: 0 off, 1 the next compaction computes every
                              // vertex's bound, 2 on (foff, fmask set)
    unsigned fmask;           // sources that take part in the bounds
    int foff[PACK_MAX];       // per source: its distance at the hub when the bounds were computed
};

// Everything an expansion / compaction touches.  Indices are "slots": the vertex ids of
// a single solve, or instance-tagged vertex ids of a batch (slot = base_i + v).
struct DevState {
    const int *row;           // row offsets, indexed VB_i + v (graphs concatenated)
    const int *col;           // local target ids
    const int *w;             // weights (unused for unit-weight solves)
    const unsigned char *cls; // out-degree class per slot
    int *dist;                // per slot
    unsigned *bm[2];          // update bitmaps per slot (scan uses bm[0]; push ping-pongs)
    int *queue[2];            // frontier, segmented by class (seg_off)
    const int *seg_off;       // [NCLS+1] class segment offsets inside a queue
    int *cnt;                 // [3][NCLS] frontier class counters, rotating by iteration
    const int *lut;           // batch: slot >> LUT_SHIFT -> instance
    const int2 *inst;         // batch: per instance {slot base, row base}
    long long nslots;
    long long nwords;         // bitmap words
    int inf;                  // unreached value written at init
    Ctrl *ctrl;
    // source-packed batch (kshift >= 0): 2^kshift sources of one graph per vertex row,
    // dist[(v << kshift) + i]; mflag[v] = sources pending at v; bm[0] = one byte per 8
    // vertices, nonzero where an mflag may be; qmask[] = source mask of each queue entry
    int kshift;               // -1: one distance per slot
    unsigned *mflag;
    unsigned *qmask[2];
    // NP_SCHEME_GLOBAL_BUFFER: heavy vertices of one expansion and the buffer's fill
    // counters [3], rotating by iteration
    int *sbuf;
    int *sbcnt;
    // source-packed, host-loop and graph drives: a counting kernel after each compaction
    // accumulates Ctrl::edges_total / items_total (set when the solve records a trace)
    int count_work;
    // source-packed, no priority window: a flagged vertex of out-degree class >= hold_cls that
    // fewer than hold_min of the pack's sources have reached is held back one compaction pass
    // (once per flagging; bm[1] marks the held vertices); hold_cls 0 = never
    int hold_cls;
    int hold_min;
    // source-packed with a priority window: sources of v whose distance was not below the window when
    // it was last looked at; null without a window
    unsigned *deferred;
    // source-packed bound filter (see pk_bound_code): one byte per vertex, null = off; a code step
    // is 2^fshift, and at least fmin sources have to have reached the hub (solver id 0)
    unsigned char *bound;
    int fshift;
    int fmin;
};

struct SchedDev {
    int learned;            // evaluate the MLP each iteration
    int level, klo, khi;    // fixed schedule (the fallback when the MLP is unusable)
    int push;               // NP_FRONTIER_PUSH
    int delta;              // priority window (0 = off)
    int max_iters;
    int trace_cap;
    int n_feat;             // vertex count used by the features
    const float *mlp;       // NP_MLP_NPARAM device floats
    np_trace_rec *trace;
    int scheme;             // NP_SCHEME_* (0: the consolidation bins)
    int solo;               // persistent drive: small frontiers run on one workgroup
};

// ---- kernels.hip: solve drivers ----------------------------------------------------
// Launch shapes are chosen by the callers in np_api.cpp.
hipError_t launch_fill_i32(int *p, long long n, int v, hipStream_t s);
hipError_t launch_fill_u32(unsigned *p, long long n, unsigned v, hipStream_t s);
hipError_t launch_degree_class(const int *row, int n, unsigned char *cls, int *hist, hipStream_t s);
// out3[0] = CSR violations, out3[1] = negative weights, out3[2] = largest weight (w may be
// null: no weight checks); out3 must hold zeros.
hipError_t launch_validate_csr(const int *row, const int *col, const int *w, int n, long long m, int *out3,
                               hipStream_t s);
// *out = largest finite distance of the state's buffer (0 when none).
hipError_t launch_max_finite(const DevState &st, int *out, hipStream_t s);
// *bad = reached edges u -> v with dist[v] = inf and dist[u] + w >= inf (a distance that the
// int32 range below inf cannot hold); batch: concatenated slots.
hipError_t launch_dist_escape(const DevState &st, bool batch, int *bad, hipStream_t s);
hipError_t launch_init_solve(const DevState &st, const int *d_src_slots, int nsrc, int push, int delta,
                             hipStream_t s);
hipError_t launch_reached_work(const int *row, const int *dist, int n, int inf,
                               unsigned long long *out2, hipStream_t s);
hipError_t launch_rebase_row(const int *row, int n, int add, int *out, hipStream_t s);
hipError_t launch_fill_lut(int *lut, long long first, long long count, int inst, hipStream_t s);
hipError_t launch_copy_cls(const unsigned char *src, unsigned char *dst, long long n,
                           hipStream_t s);

// Source-packed state: dist rows set to inf, source i of srcs[] at lane i (nsrc <= 2^kshift);
// delta > 0 starts a priority window at T = delta.
hipError_t launch_init_packed(const DevState &st, const int *d_srcs, int nsrc, int delta, hipStream_t s);
// out[to.off[j] + v] = dist[(map(v) << kshift) + j] for j < to.count with to.off[j] >= 0, map = old2new
// or identity (old2new null).
struct UnpackTo { long long off[PACK_MAX]; int count; };
hipError_t launch_unpack(const int *dist, int kshift, const UnpackTo &to, const int *old2new, int n, int *out,
                         hipStream_t s);
// out[p.off + v] = dist[p.base + p.old2new[v]] for every instance p of a concatenated part whose
// old2new is not null (lut: slot >> LUT_SHIFT -> index into parts).
struct ConcatOut { long long off; const int *old2new; int base, n; };
hipError_t launch_unpermute_parts(const int *dist, const int *lut, const ConcatOut *parts, long long nslots, int *out,
                                  hipStream_t s);

// Persistent drive: one cooperative launch.  `wgs` workgroups of 256 threads.  A state
// with kshift >= 0 runs the source-packed kernels (here and in compact/expand).
hipError_t launch_persistent(const DevState &st, const SchedDev &sp, bool batch, bool unit,
                             int wgs, hipStream_t s);
int persistent_max_wgs_per_cu(bool batch, bool unit, bool push, bool packed, bool solo, bool window);

// Host-loop / graph drive, one iteration = [compact] + decide + expand.
hipError_t launch_compact(const DevState &st, int it_off, bool batch, int wgs, hipStream_t s);
hipError_t launch_decide(const DevState &st, const SchedDev &sp, int it_off, hipStream_t s);
hipError_t launch_expand(const DevState &st, const SchedDev &sp, int it_off, bool batch, bool unit,
                         int wgs, hipStream_t s);
hipError_t launch_advance(const DevState &st, int k, hipStream_t s);
// NP_SCHEME_BFS_FLAT: one level-synchronous pass over every vertex (levels in st.dist);
// *changed (device) is set when a level was written.
hipError_t launch_bfs_flat(const DevState &st, int level, int *changed, int wgs, hipStream_t s);
// Stepping: force the next expansion's schedule (writes ctrl->cfg_*).
hipError_t launch_set_cfg(const DevState &st, int level, int klo, int khi, hipStream_t s);

// ---- kernels.hip: scheduler MLP ------------------------------------------------------
hipError_t launch_mlp_forward(const float *p, const float *x, int batch, float *out,
                              hipStream_t s);
// Per-sample forward+backward then per-parameter reduction: grad (NP_MLP_NPARAM) and the
// mean loss (loss[0]).  work: scratch of mlp_work_floats(batch) floats.
size_t mlp_work_floats(int batch);
hipError_t launch_mlp_loss_grad(const float *p, const float *x, const int *label,
                                const float *target, int batch, float lam, float *work,
                                float *grad, float *loss, hipStream_t s);
hipError_t launch_adam(float *p, const float *grad, float *m, float *v, int n, float lr,
                       float b1, float b2, float eps, int step, hipStream_t s);

// ---- bc.hip: betweenness centrality, up to 32 sources per batch -----------------------
struct BcDev {
    const int *row, *col;  // CSR (original ids)
    int n, ks;             // slots (v << ks) + j for batch source j < 2^ks
    uint2 *st;             // [n] bits per source: .x reached on a level up to the one in hand, .y reached
                           //     by the expansion in flight
    double *sig, *del;     // shortest-path counts and dependencies per slot
};
struct BcLevel {
    unsigned long long ctl;  // entries (low half) and chunks (high half); zero before the level
    long long first;         // first entry in ent_v/ent_m; zero for level 0
};
hipError_t launch_bc_reset(const BcDev &b, hipStream_t s);
hipError_t launch_bc_sources(const BcDev &b, const int *srcs, int nsrc, hipStream_t s);
// Vertices reached by the last expansion -> the entries of lv's level at ent_v/ent_m + lv->first and
// their chunks' records {v, mask, first edge, edges left in the row}; a chunk past cap sets *err
// (nothing is written past cap).
hipError_t launch_bc_compact(const BcDev &b, int *ent_v, unsigned *ent_m, BcLevel *lv, int4 *rec, long long cap,
                             int *err, hipStream_t s);
// Expansion of lv's chunks (their count is read on the device).  Forward, it sets lv[1].first.
hipError_t launch_bc_expand(const BcDev &b, bool fwd, BcLevel *lv, const int4 *rec, long long cap, double *bc,
                            int num_cus, hipStream_t s);
// Backward: the finished level's ne entries out of seen, and into bc and their slots' factors where
// the sweep has not done that (`all`: the deepest level, which no sweep has passed); the chunks of
// the next level's nn entries, counted in lv->ctl.
hipError_t launch_bc_finish(const BcDev &b, const int *ent_v, const unsigned *ent_m, int ne, bool all, double *bc,
                            const int *nxt_v, const unsigned *nxt_m, int nn, BcLevel *lv, int4 *rec, long long cap,
                            int *err, hipStream_t s);
hipError_t launch_bc_to_float(const double *bc, int n, float *out, hipStream_t s);

// ---- color.hip: graph coloring (longest decreasing-id path labels) -----------------------
// Dependency solve.  cnt, at: color_blocks(n) + 1 ints; tick, part: color_ticket_cap(n, m);
// color: n; ctl: 3.  part, color and ctl hold zeros before it; after it ctl[1] = the largest
// color, ctl[2] != 0 when a bounded wait expired.
struct ColorBufs {
    int *cnt, *at, *part, *color, *ctl;
    int2 *tick;
    void *temp;
    size_t temp_bytes;  // of color_scan (temp null queries it)
};
long long color_blocks(int n);
long long color_ticket_cap(int n, long long m);
hipError_t color_scan(void *temp, size_t *temp_bytes, const int *in, int *out, int n, hipStream_t s);
hipError_t launch_color_solve(const int *row, const int *col, int n, long long m, const ColorBufs &b, int num_cus,
                              hipStream_t s);
hipError_t launch_color_round(const int *row, const int *col, int n, int *color, int c, int *nonstop, hipStream_t s);

// ---- pagerank.hip: PageRank over the in-edge CSR ------------------------------------------
// Rows by length: < PR_HEAVY entries PR_GROUP lanes each; < PR_HUGE one wavefront each (med);
// longer rows (huge) in PR_CHUNK-entry chunks, one wavefront per chunk, partial sums in part[].
constexpr int PR_GROUP = 8;
constexpr int PR_HEAVY = 32;
constexpr int PR_CHUNK = 2048;
constexpr int PR_HUGE = 2 * PR_CHUNK;
struct RowBins {
    int *med, *nmed;              // medium rows [n]; count
    int *huge, *hc0, *nhuge;      // huge rows and their first chunk [m / PR_HUGE + 1]; count
    int *hleft;                   // chunks of each huge row still to finish (null: not kept)
    int *crow, *ck, *nchunk;      // chunk -> row, chunk index [pr_chunk_cap(m)]; count
    int *chuge;                   // chunk -> index into huge (null: not kept)
    double *part;                 // per-chunk partial sums [pr_chunk_cap(m)]
};
// Rotating sums of the iterations (see k_pr_pull), a cache line per slot: workgroup b adds to slot
// b % PR_SLOTS, because atomics on one line take turns (about 30 ns each: 2,048 workgroups on one
// pair of sums took longer than their rows).  Zero before launch_pr_init.
constexpr int PR_SLOTS = 64;
struct alignas(64) PrSlot { double dsum[3]; unsigned long long dmax[3]; };
struct PrSums {
    PrSlot slot[PR_SLOTS];
    int iters;
};
long long pr_chunk_cap(long long m);
// In-edge CSR: src[e] = source of edge e; sort (col, src) pairs; offsets from the sorted targets.
// src[e] = source of edge e for the m edges of the CSR row (heads: m ints of scratch; temp null
// queries *temp_bytes).
hipError_t pr_sources(void *temp, size_t *temp_bytes, const int *row, int n, long long m, int *heads, int *src,
                      hipStream_t s);
hipError_t pr_sort(void *temp, size_t *temp_bytes, const unsigned *key_in, unsigned *key_out, const int *val_in,
                   int *val_out, long long m, int end_bit, hipStream_t s);
hipError_t launch_pr_offsets(const unsigned *key, long long m, int n, int *irow, hipStream_t s);
// Bins over n rows with offsets off (counts *nmed, *nhuge, *nchunk zero on entry).
hipError_t launch_row_bins(const int *off, int n, long long m, const RowBins &rb, hipStream_t s);
// rank = r0, contributions and dangling sum of iteration 0.
hipError_t launch_pr_init(const int *row, int n, double r0, double *rank, double *contrib, PrSums *ps, hipStream_t s);
// Iteration i, rank in place, contrib -> ncontrib.  Nothing runs once an iteration changed no vertex
// by more than eps; ps->iters = iterations that ran, the greatest dmax[i % 3] of the slots = the largest change of
// the i-th.
hipError_t launch_pr_iteration(int i, PrSums *ps, const int *row, const int *irow, const int *pcol, const RowBins &rb,
                               double *rank, const double *contrib, double *ncontrib, int n, long long m, double damping,
                               double rw, double eps, int num_cus, hipStream_t s);
hipError_t launch_pr_to_float(const double *rank, const int *old2new, int n, float *out, hipStream_t s);
// SpMV y = A x over the graph's CSR, with row bins built by launch_row_bins.
hipError_t launch_spmv(const int *row, const int *col, const double *data, const double *x, double *y, int n,
                       const RowBins &rb, int num_cus, hipStream_t s);

// ---- gen.hip: generators and CSR construction ---------------------------------------
struct GenOut { int *row; int *col; int *w; };
// Builds CSR (reverse generation order per vertex) from an edge list in generation order.
hipError_t build_csr_device(const uint32_t *src, const uint32_t *dst, const int *w, int n,
                            long long m, GenOut *out, hipStream_t s);
hipError_t gen_rmat_edges(int scale, long long m, uint64_t seed, double a, double b, double c,
                          int permute, int wmin, int wmax, uint32_t *src, uint32_t *dst, int *w,
                          hipStream_t s);
hipError_t gen_er_edges(int n, long long m, uint64_t seed, int wmin, int wmax, uint32_t *src,
                        uint32_t *dst, int *w, hipStream_t s);
hipError_t gen_grid_edges(int rows, int cols, long long n_long, uint64_t seed, int wmin, int wmax,
                          const long long *grid_off, uint32_t *src, uint32_t *dst, int *w,
                          hipStream_t s);

hipError_t grid_offsets(int rows, int cols, long long *grid_off, hipStream_t s);

// Solver layout renumbered by decreasing in-degree.  `skew` = share of the edges that the
// top n/16 vertices receive; the layout is built (active) only when skew >= min_skew.
struct Relabel {
    bool active = false;
    double skew = 0.0;
    int *row = nullptr, *col = nullptr, *w = nullptr;  // renumbered CSR
    int *old2new = nullptr;                             // original id -> solver id
};
hipError_t relabel_by_indegree(const int *row, const int *col, const int *w, int n, long long m,
                               double min_skew, Relabel *out, hipStream_t s);
// out[v] = src[old2new[v]]
hipError_t launch_unpermute(const int *src, const int *old2new, int n, int *out, hipStream_t s);
// Thresholds of rmat_edge from probabilities.
void rmat_thresholds(double a, double b, double c, uint64_t *ta, uint64_t *tab, uint64_t *tabc);

}  // namespace np
