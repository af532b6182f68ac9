// ag_internal.h -- shared definitions of the HIP runtime and kernels (not installed).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>
#include <time.h>

#include "accelgraph.h"
#include "../host/ag_plan.h"

#define AG_MAX_EVENTS 2
#define AG_STAGE_SLOTS 4u
#define AG_STAGE_BYTES ((size_t)4 << 20)
#define AG_LANE_MAX 64u    // rows of a tile with at most this many elements: a lane each

struct ag_device {
    int ordinal;
    hipStream_t stream;
    uint64_t run_timeout_ms;
    uint32_t poll_us;
    uint32_t live_graphs;   // graphs and batches on this device, not yet freed
    struct ag_dgraph *graphs;   // list of the uploaded graphs (ag_dgraph::next)
    uint32_t num_cus;       // compute units (persistent-grid sizing)
    void *scratch;          // this device's copy of the ag_spmv_pull_noalloc scratch array
    // pinned ring of the staged transfers (ag_copy_in / ag_copy_out), allocated on first use
    char *stage;                        // [AG_STAGE_SLOTS][AG_STAGE_BYTES]
    hipEvent_t stage_ev[AG_STAGE_SLOTS];   // the last transfer through each slot
    uint32_t stage_used;                // slots whose event has been recorded (bit mask)
    uint32_t stage_next;                // slot of the next transfer
    hipEvent_t time_ev[2];              // a call's timed launches
};

// Buffers that ended sessions of a graph hand back for the next one to take (every PageRank call
// begins and ends a session): at most AG_PARK_BYTES of device memory, one pinned block and one
// set of events. Freed with the graph, or by ag_dev_malloc when memory runs out; counted in the
// graph's device bytes meanwhile.
#define AG_PARK_BLOCKS 8u
#define AG_PARK_BYTES ((size_t)1 << 30)
#define AG_PIN_BYTES ((size_t)64 << 10)
struct ag_parked {
    void *dev[AG_PARK_BLOCKS];
    size_t bytes[AG_PARK_BLOCKS];
    uint32_t n_dev;
    void *pin;               // [AG_PIN_BYTES]
    hipEvent_t ev[3];
    uint32_t has_ev;
};

// Device-resident graph: the plan arrays in HBM plus launch geometry.
struct ag_dgraph {
    ag_device *dev;
    ag_dgraph *next;     // of the device's list
    ag_plan_params params;
    uint32_t n, m;
    uint32_t bin_row[AG_NBINS + 1];
    uint64_t bin_edges[AG_NBINS];
    uint32_t bin_blocks[AG_NBINS];
    uint32_t slot_blk0[AG_NSLOTS + 1];
    uint32_t total_blocks;
    uint32_t n_tiles, n_hubs, n_segs;
    uint64_t device_bytes;
    // HBM arrays
    uint32_t *d2o;       // [n]
    uint32_t *h_d2o;     // [n] host copy of the device-row map
    uint32_t *off;       // [n+1]
    uint32_t *src;       // [m]
    float *w;            // [m] or null
    uint32_t *wq;        // [m] FloatToFixed32(w), built on first fixed SpMV, or user codes
    int wq_user;         // wq came from ag_graph_set_fixed_weights
    uint32_t *outdeg;    // [n]
    uint32_t *tile_row;  // [n_tiles+1]
    uint4 *rt;           // [n_rt] row tiles of the regular schedule (PullGeom::rt)
    uint32_t n_rt, n_heavy;
    uint32_t *seg_row, *seg_lo, *seg_hi;  // [n_segs]
    uint32_t *hub_seg0;  // [n_hubs+1]
    uint64_t *hub_part;    // [n_segs] 8-byte partial sums (float or u64 bits)
    // source blocking of the PageRank pull (blk.bits == 0: none); host copies of the
    // schedule scalars and HBM arrays of the block plan
    ag_block_plan blk;   // pointer members are device pointers here
    uint64_t *vpart;     // [blk.nv] partial sum of every virtual row (float or u64 bits)
    uint32_t *btick;     // [2 * AG_NXCD] pass-1 ticket counters (BlockGeom::tick), zeroed
    uint32_t bdyn;       // pass-1 tiles handed out by ticket (BlockGeom::dyn)
    uint32_t *vwq;       // [blk.mb] FloatToFixed32(vw), built on the first fixed SpMV
    // forward CSR in device row ids (out-edges), built on the first run with worklists
    uint32_t *fwd_off;   // [n+1]
    uint32_t *fwd_dst;   // [m] destination, ascending within a row
    // scratch for permuted vectors (x, y) of SpMV / gather, sized lazily
    void *vec_a;
    void *vec_b;
    size_t vec_bytes;
    // personalised PageRank: buffers and the captured solve, kept between calls
    struct ag_ppr_ws *ppr;
    struct ag_parked parked;   // buffers of ended PageRank sessions
};

// Frees g->ppr (ag_ppr.hip).
void ag_ppr_free_ws(ag_dgraph *g);

// Geometry passed by value to the pull kernels.
struct PullGeom {
    const uint32_t *off;
    const uint32_t *src;
    const uint32_t *tile_row;
    const uint32_t *seg_row;
    const uint32_t *seg_lo;
    const uint32_t *seg_hi;
    const uint32_t *hub_seg0;
    uint64_t *hub_part;
    const uint4 *rt;         // [n_rt] row tiles {first row, end row, first in-edge, end}
    uint32_t n_rt;
    uint32_t n_heavy;        // items of slot_blk0 before the row tiles (hub segments, block rows)
    uint32_t lane_max;       // rows of a tile up to this in-degree are summed by one lane
    uint32_t seq_max;        // and up to this one in stream order
    uint32_t n;
    uint32_t n_hubs;
    uint32_t seq_hubs;       // plan in reference order: a hub row is one segment, added by one
                             // lane in sequence (chunks staged through LDS)
    uint32_t bin_row[AG_NBINS + 1];
    uint32_t slot_blk0[AG_NSLOTS + 1];
};

// Source-blocked pull: virtual rows, the combine schedule and the work items of each slice.
struct BlockGeom {
    PullGeom V;              // off = voff, src = vsrc (virtual rows; null with sorted tiles)
    PullGeom C;              // off = coff, src = cidx (a row's partial slots)
    const uint32_t *item;    // [2 * n_items] pass-1 items
    const uint32_t *c_item;  // [2 * c_n_items] combine items
    const uint32_t *ct_row;  // [2 * c_n_tiles]
    const uint32_t *ct_start;
    const uint32_t *ct_pre;
    const uint16_t *lpos;
    uint64_t *part;          // [nv]
    uint32_t nblocks;
    uint32_t item_off[AG_NXCD + 1];
    uint32_t c_item_off[AG_NXCD + 1];
    // pass 1 over the L2 takes the items [item_lo[x], item_off[x + 1]) of slice x: from
    // item_off[x] (every tile), or from the end of the hot-segment tiles when the hot pass
    // (groups hgrp, hgrp_off) gathers those from LDS
    uint32_t item_lo[AG_NXCD];
    const uint32_t *hgrp;    // [3 * n_hgrp] {first item, item count, segment}
    uint32_t hgrp_off[AG_NXCD + 1];
    uint32_t hot_bits;
    uint32_t n_src;          // source (vertex) count: the last segment may be short
    // pass 1 hands out its tiles through per-slice tickets (no AG_ITEM_REG item in pass 1):
    // tick[x] = next ticket of slice x, tick[AG_NXCD + x] = its workgroups that have left;
    // both zero between launches
    uint32_t dyn;
    uint32_t *tick;
    uint32_t top0;           // first source of the first-pass LDS table (n_src: none)
    // pass-1 tiles sorted by source (sbits != 0): vsp[e] = position in the tile << sbits |
    // (source - tbase[item]); the per-edge weights are then in the same order
    const uint32_t *vsp;
    const uint32_t *tbase;
    uint32_t sbits;
    uint32_t has_reg;        // pass 1 has AG_ITEM_REG items: it finishes the unblocked rows
};

// Points pass 1 of B past the hot-segment tiles (when the hot pass runs before it).
void ag_block_geom_skip_hot(const ag_dgraph *g, BlockGeom &B);

// Persistent-grid size of a pull launch: resident workgroups per CU x CUs, capped by the
// number of work items. Per CU: the plan's wg_per_cu, else default_per_cu, never more than
// LDS allows.
uint32_t ag_pull_grid(const ag_dgraph *g, uint32_t lds_bytes, uint32_t default_per_cu = 4u);

// The same for the regular schedule in row tiles.
uint32_t ag_tile_grid(const ag_dgraph *g, uint32_t lds_bytes);

// Device-side iteration state of a PageRank session.
struct PrState {
    uint32_t iter;          // iterations executed so far
    uint32_t done;          // set when the stopping iteration is closed (the next launch's opening
                            // step, or the closing kernel at a step's end)
    uint32_t stop_iter;     // index of the stopping iteration
    int32_t refine_iter;    // first iteration that writes f32 contributions (-1: none yet)
    uint32_t last_active;
    double last_err;
    double best_err;        // smallest L1 delta of the 16-bit phase so far
    uint32_t stall;         // 16-bit iterations since best_err last improved by 1%
    uint32_t qmax_bits;     // quantised kinds: bits of the largest next contribution
    float qscale;           // quantised kinds: scale of the codes being gathered
    uint32_t dd_count[2];   // data-driven pull: worklist lengths by iteration parity
    uint32_t dd_hubs[2];    // data-driven pull: hub rows listed at the worklist's far end
};

// A PageRank session (ag_pr_begin .. ag_pr_end).
struct ag_pr_session {
    ag_dgraph *g;
    ag_pr_options o;
    uint32_t kind_code;         // 0 f32, 1 bf16, 2 f16, 64/32/16/8
    size_t celem;               // bytes per stored contribution
    PrState *st;                // device [2], by iteration parity
    PrState *st_host;           // pinned, the start of pin
    void *pin;                  // [AG_PIN_BYTES] state and history on their way to the caller
    void *blk[AG_PARK_BLOCKS];  // this session's device allocations
    size_t blk_bytes[AG_PARK_BLOCKS];
    uint32_t n_blk;
    double *part_err;
    uint32_t *part_act;
    uint32_t *part_cmax;        // quantised kinds: per-workgroup largest contribution bits
    double *hist_err;
    uint32_t *hist_act;
    float *rank;
    void *c[2];
    void *c16[2];
    uint32_t *dd_queue[2];      // data-driven pull: worklists by iteration parity
    uint8_t *dd_flag;           // data-driven pull: next-worklist marks [n rounded up to 4]
    double *fin_part;
    double *fin_sum;
    float *user;
    uint32_t enqueued;
    uint64_t *hist_t;           // device clock per iteration when record_history (start, end);
                                // hist_err, it and hist_act are one run of memory
    size_t hist_bytes;          // of hist_bytes bytes
    hipEvent_t loop_ev;         // before the first iteration
    uint32_t nparts;            // partials of one iteration's launches
    hipEvent_t step_ev[2];
    uint32_t step_launches;
    struct timespec t0;  // wall clock at ag_pr_begin
};

// Builds g->fwd_off / fwd_dst (the forward CSR in device row ids) from the uploaded inverse CSR,
// once; later calls return at once.
int ag_graph_forward(ag_dgraph *g);

int ag_set_error(int status, const char *fmt, ...);
int ag_hip_fail(hipError_t e, const char *what, const char *file, int line);
int ag_wait_stream(ag_device *dev);
int ag_wait_event(ag_device *dev, hipEvent_t ev);
// Host -> device copy on the device's stream, straight for small vectors and memory that the runtime
// knows (pinned memory may not be reused before a wait), else through the pinned ring. `largest`:
// bytes of the largest vector that the call moves, in or out (its vectors go the same way).
int ag_copy_in(ag_device *dev, void *dst, const void *host, size_t bytes, size_t largest);
// Device -> host copy after the work on the device's stream; done on return.
int ag_copy_out(ag_device *dev, void *host, const void *src, size_t bytes, size_t largest);
// Frees the parked buffers of a graph.
void ag_parked_free(ag_dgraph *g);
// hipMalloc for every allocation of the library: when device memory runs out, the parked buffers of
// all the device's graphs are freed and it tries once more. Returns a hipError_t.
hipError_t ag_dev_malloc_bytes(ag_device *dev, void **p, size_t bytes);
template <typename T>
static inline hipError_t ag_dev_malloc(ag_device *dev, T **p, size_t bytes)
{
    return ag_dev_malloc_bytes(dev, (void **)p, bytes);
}

#define AG_HIP(call)                                                   \
    do {                                                               \
        hipError_t ag_e_ = (call);                                     \
        if (ag_e_ != hipSuccess)                                       \
            return ag_hip_fail(ag_e_, #call, __FILE__, __LINE__);      \
    } while (0)

// graph_csr.c: parallel first touch of a new graph's host arrays (before bulk copies into them)
struct GraphCSR;
extern "C" void graphCSRPrefault(struct GraphCSR *g);

PullGeom ag_make_geom(const ag_dgraph *g);
// Regular schedule of the rows a source-blocked graph leaves unblocked (AG_ITEM_REG items).
PullGeom ag_make_unblocked_geom(const ag_dgraph *g);
BlockGeom ag_make_block_geom(const ag_dgraph *g);
// Grid of either pass of a source-blocked iteration: CUs x workgroups per CU (the plan's
// wg_per_cu, else default_per_cu, never more than resident_per_cu), a multiple of AG_NXCD. A
// persistent grid must fit on the device at once: a workgroup that waits for a free slot runs
// its whole share of the items after the others have finished. The gather pass defaults to 4
// per CU (it is bound by the rate of random L2 requests: more in flight only queue); the
// combine pass, whose reads are coalesced and whose time goes to dependent round trips,
// defaults to as many as fit, up to 8.
uint32_t ag_blocked_grid(const ag_dgraph *g, uint32_t resident_per_cu, uint32_t default_per_cu);

// Workgroups of `lanes` lanes of `kernel` that fit on one CU (registers and LDS).
template <typename K>
static inline uint32_t ag_resident_per_cu(K kernel, uint32_t lanes = AG_WG)
{
    int nb = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, kernel, (int)lanes, 0) != hipSuccess ||
        nb < 1)
        return 1u;
    return (uint32_t)nb;
}
int ag_ensure_vec(ag_dgraph *g, size_t bytes);
