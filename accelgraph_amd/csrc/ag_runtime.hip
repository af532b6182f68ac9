// ag_runtime.hip -- device contexts, error reporting, the bounded wait (watchdog) and graph
// upload of the accelgraph C-ABI.
//
// Replaces the reference's CAPI runtime boundary (02_capi_graph/src/capi_utils/capienv.c:
// setupAFUGraphCSR 329-372, startAFU 375-451, waitAFU 526-638, releaseAFU 765-782,
// mapGraphCSRToWED 832-874). The FPGA read host memory coherently through a work-element
// descriptor; here the arrays the pull path reads are uploaded into HBM once, in the
// degree-binned layout built by ag_plan_build, and every later run reuses them.
#include <stdarg.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>
#include <time.h>
#include <unistd.h>

#include <new>
#include <vector>

#include "ag_internal.h"
#include "ag_fixed_dev.h"

static thread_local char g_err[512] = "";

int ag_set_error(int status, const char *fmt, ...)
{
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(g_err, sizeof(g_err), fmt, ap);
    va_end(ap);
    return status;
}

int ag_hip_fail(hipError_t e, const char *what, const char *file, int line)
{
    int st = (e == hipErrorOutOfMemory) ? AG_ERR_OOM
             : (e == hipErrorNoDevice || e == hipErrorInvalidDevice) ? AG_ERR_NO_DEVICE
                                                                    : AG_ERR_HIP;
    return ag_set_error(st, "%s failed: %s (%s:%d)", what, hipGetErrorString(e), file, line);
}

extern "C" const char *ag_last_error(void) { return g_err; }

extern "C" int ag_abi_version(void) { return AG_ABI_VERSION; }

extern "C" const char *ag_status_string(int s)
{
    switch (s) {
    case AG_OK: return "ok";
    case AG_ERR_INVALID: return "invalid argument";
    case AG_ERR_NO_DEVICE: return "no usable device";
    case AG_ERR_HIP: return "HIP runtime error";
    case AG_ERR_OOM: return "out of memory";
    case AG_ERR_TIMEOUT: return "device wait timed out";
    case AG_ERR_UNSUPPORTED: return "unsupported option";
    default: return "unknown status";
    }
}

static uint64_t env_u64(const char *name, uint64_t dflt)
{
    const char *v = getenv(name);
    if (!v || !*v)
        return dflt;
    char *end = NULL;
    unsigned long long x = strtoull(v, &end, 10);
    return (end && *end == '\0') ? (uint64_t)x : dflt;
}

extern "C" int ag_device_count(int *count)
{
    if (!count)
        return ag_set_error(AG_ERR_INVALID, "count is null");
    int c = 0;
    hipError_t e = hipGetDeviceCount(&c);
    if (e != hipSuccess) {
        *count = 0;
        return ag_hip_fail(e, "hipGetDeviceCount", __FILE__, __LINE__);
    }
    *count = c;
    return AG_OK;
}

// Scratch of the allocation-free entry point ag_spmv_pull_noalloc (permuted x and y), a
// file-scope device array: every GPU the library runs on holds its own copy at its own
// address until the process ends. Host code never uses the array's name as an address: the
// address is taken once per device with hipGetSymbolAddress (that device current) when the
// device is first opened, and kept per ordinal.
static __device__ __align__(256) unsigned char scratch[AG_NOALLOC_SCRATCH_BYTES];
#define AG_MAX_ORDINALS 64
static void *g_scratch_ptr[AG_MAX_ORDINALS];

extern "C" int ag_device_open(int ordinal, ag_device **out)
{
    if (!out)
        return ag_set_error(AG_ERR_INVALID, "out is null");
    *out = NULL;
    int c = 0;
    hipError_t e = hipGetDeviceCount(&c);
    if (e != hipSuccess || c == 0)
        return ag_set_error(AG_ERR_NO_DEVICE, "no HIP device available (%s)",
                            e == hipSuccess ? "count is 0" : hipGetErrorString(e));
    if (ordinal < 0 || ordinal >= c)
        return ag_set_error(AG_ERR_INVALID, "device ordinal %d out of range [0,%d)", ordinal, c);
    AG_HIP(hipSetDevice(ordinal));
    ag_device *d = (ag_device *)calloc(1, sizeof(ag_device));
    if (!d)
        return ag_set_error(AG_ERR_OOM, "host allocation failed");
    d->ordinal = ordinal;
    d->run_timeout_ms = env_u64("ACCELERATOR_RUN_TIMEOUT_MS", 0);
    d->poll_us = (uint32_t)env_u64("ACCELERATOR_POLL_INTERVAL_US", 50);
    int cus = 0;
    e = hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, ordinal);
    if (e != hipSuccess || cus <= 0) {
        free(d);
        return ag_hip_fail(e, "hipDeviceGetAttribute(CU count)", __FILE__, __LINE__);
    }
    d->num_cus = (uint32_t)cus;
    if (ordinal < AG_MAX_ORDINALS && !g_scratch_ptr[ordinal]) {
        void *p = NULL;
        e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess || !p) {
            free(d);
            return ag_hip_fail(e, "hipGetSymbolAddress(scratch)", __FILE__, __LINE__);
        }
        g_scratch_ptr[ordinal] = p;
    }
    d->scratch = ordinal < AG_MAX_ORDINALS ? g_scratch_ptr[ordinal] : NULL;
    e = hipStreamCreateWithFlags(&d->stream, hipStreamNonBlocking);
    if (e != hipSuccess) {
        free(d);
        return ag_hip_fail(e, "hipStreamCreateWithFlags", __FILE__, __LINE__);
    }
    e = hipEventCreate(&d->time_ev[0]);
    if (e == hipSuccess) {
        e = hipEventCreate(&d->time_ev[1]);
        if (e != hipSuccess)
            (void)hipEventDestroy(d->time_ev[0]);
    }
    if (e != hipSuccess) {
        (void)hipStreamDestroy(d->stream);
        free(d);
        return ag_hip_fail(e, "hipEventCreate", __FILE__, __LINE__);
    }
    *out = d;
    return AG_OK;
}

extern "C" int ag_device_close(ag_device *d)
{
    if (!d)
        return AG_OK;
    if (d->live_graphs)
        return ag_set_error(AG_ERR_INVALID, "%u graph(s) still uploaded on this device; free "
                            "them before closing it", d->live_graphs);
    (void)hipSetDevice(d->ordinal);
    (void)hipStreamSynchronize(d->stream);
    if (d->stage) {
        for (uint32_t i = 0; i < AG_STAGE_SLOTS; i++)
            (void)hipEventDestroy(d->stage_ev[i]);
        (void)hipHostFree(d->stage);
    }
    (void)hipEventDestroy(d->time_ev[0]);
    (void)hipEventDestroy(d->time_ev[1]);
    (void)hipStreamDestroy(d->stream);
    free(d);
    return AG_OK;
}

extern "C" int ag_device_set_watchdog(ag_device *d, uint64_t run_timeout_ms, uint32_t poll_us)
{
    if (!d)
        return ag_set_error(AG_ERR_INVALID, "device is null");
    d->run_timeout_ms = run_timeout_ms;
    d->poll_us = poll_us ? poll_us : 1;
    return AG_OK;
}

static uint64_t now_ms(void)
{
    struct timespec ts;
    clock_gettime(CLOCK_MONOTONIC, &ts);
    return (uint64_t)ts.tv_sec * 1000ull + (uint64_t)ts.tv_nsec / 1000000ull;
}

// Wait for an event; bounded by the watchdog deadline when one is set.
int ag_wait_event(ag_device *d, hipEvent_t ev)
{
    if (d->run_timeout_ms == 0) {
        AG_HIP(hipEventSynchronize(ev));
        return AG_OK;
    }
    const uint64_t deadline = now_ms() + d->run_timeout_ms;
    for (;;) {
        const hipError_t e = hipEventQuery(ev);
        if (e == hipSuccess)
            return AG_OK;
        if (e != hipErrorNotReady)
            return ag_hip_fail(e, "hipEventQuery", __FILE__, __LINE__);
        if (now_ms() >= deadline)
            return ag_set_error(AG_ERR_TIMEOUT, "device work did not finish within %llu ms",
                                (unsigned long long)d->run_timeout_ms);
        usleep(d->poll_us);
    }
}

// Wait for all work on the device stream (the role of waitAFU's run deadline,
// capienv.c:526-638).
int ag_wait_stream(ag_device *d)
{
    if (d->run_timeout_ms == 0) {
        AG_HIP(hipStreamSynchronize(d->stream));
        return AG_OK;
    }
    hipEvent_t ev;
    AG_HIP(hipEventCreateWithFlags(&ev, hipEventDisableTiming));
    const hipError_t e = hipEventRecord(ev, d->stream);
    const int st = e == hipSuccess ? ag_wait_event(d, ev)
                                   : ag_hip_fail(e, "hipEventRecord", __FILE__, __LINE__);
    (void)hipEventDestroy(ev);
    return st;
}

// ------------------------------------------------------------------ device memory

hipError_t ag_dev_malloc_bytes(ag_device *dev, void **p, size_t bytes)
{
    hipError_t e = hipMalloc(p, bytes);
    if (e == hipErrorOutOfMemory) {
        (void)hipGetLastError();
        for (ag_dgraph *g = dev->graphs; g; g = g->next)
            ag_parked_free(g);
        e = hipMalloc(p, bytes);
    }
    return e;
}

// ------------------------------------------------------------------ staged transfers
//
// Callers' vectors are ordinary (pageable) memory, which the runtime moves through megabyte
// chunks copied by one core, page faults of a fresh output included: 9 GB/s, 15 of the 61 ms of a
// 20-iteration RMAT-25 call. Here chunks of 4 MB go through a pinned ring kept by the device,
// the link ahead of (or behind) the copies of eight cores: 16 MB each way 1.9 -> 1.1 ms, 134 MB
// out 14 -> 5 ms. Chunks of 1 MB were slower (1.4 ms; every chunk pays its launch and wait).
// Vectors of a call go straight while the larger of its vectors is below 1 MB: the ring's second
// copy, event and wait cost more than they save. A SpMV call (x in, y out; straight / ring, us) of
// 64 KB each way 50 / 60, 256 KB 66 / 83, 400 KB 78 / 93, 800 KB 114 / 118, 1 MB 149 / 133; 256 KB
// in and 512 KB out 81 / 95, 460 and 920 KB 107 / 117, 512 KB and 1 MB 132 / 125. One vector
// straight and the other through the ring was slower than either (600 KB: 127). Results of at most
// 16 KB leave through the ring, for which the link has a faster path out of pinned memory (16 KB
// each way 41, straight 43 to 56).
#define AG_STRAIGHT_BELOW ((size_t)1 << 20)
#define AG_PINNED_OUT ((size_t)16 << 10)

// Whether the device has its ring, allocated on first use. Without pinned memory for it transfers
// go straight.
static bool stage_open(ag_device *d)
{
    if (d->stage)
        return true;
    char *p = NULL;
    hipError_t e = hipHostMalloc((void **)&p, AG_STAGE_SLOTS * AG_STAGE_BYTES, hipHostMallocDefault);
    uint32_t i = 0;
    for (; e == hipSuccess && i < AG_STAGE_SLOTS; i++)
        e = hipEventCreateWithFlags(&d->stage_ev[i], hipEventDisableTiming);
    if (e != hipSuccess) {
        (void)hipGetLastError();   // no later launch reports it
        for (uint32_t k = 0; k + 1u < i; k++)   // the last one is the one that failed
            (void)hipEventDestroy(d->stage_ev[k]);
        if (p)
            (void)hipHostFree(p);
        return false;
    }
    d->stage = p;
    d->stage_used = d->stage_next = 0u;
    return true;
}

// Whether the runtime knows this memory (pinned, managed or a GPU's): it then copies it straight.
static bool is_known(const void *host)
{
    hipPointerAttribute_t at;
    if (hipPointerGetAttributes(&at, host) != hipSuccess) {
        (void)hipGetLastError();   // ordinary memory
        return false;
    }
    return at.type != hipMemoryTypeUnregistered;
}

// The ring's next slot, free of earlier transfers.
static int stage_slot(ag_device *d, uint32_t *slot)
{
    *slot = d->stage_next;
    d->stage_next = (d->stage_next + 1u) % AG_STAGE_SLOTS;
    return (d->stage_used >> *slot & 1u) ? ag_wait_event(d, d->stage_ev[*slot]) : AG_OK;
}

int ag_copy_in(ag_device *d, void *dst, const void *host, size_t bytes, size_t largest)
{
    if (bytes == 0)
        return AG_OK;
    if (largest < AG_STRAIGHT_BELOW || is_known(host) || !stage_open(d)) {
        AG_HIP(hipMemcpyAsync(dst, host, bytes, hipMemcpyHostToDevice, d->stream));
        return AG_OK;
    }
    int st = AG_OK;
    for (size_t o = 0; st == AG_OK && o < bytes; o += AG_STAGE_BYTES) {
        const size_t len = bytes - o < AG_STAGE_BYTES ? bytes - o : AG_STAGE_BYTES;
        uint32_t k = 0;
        st = stage_slot(d, &k);
        if (st != AG_OK)
            break;
        char *slot = d->stage + k * AG_STAGE_BYTES;
        ag_par_copy(slot, (const char *)host + o, len);
        AG_HIP(hipMemcpyAsync((char *)dst + o, slot, len, hipMemcpyHostToDevice, d->stream));
        AG_HIP(hipEventRecord(d->stage_ev[k], d->stream));
        d->stage_used |= 1u << k;
    }
    return st;
}

int ag_copy_out(ag_device *d, void *host, const void *src, size_t bytes, size_t largest)
{
    if (bytes == 0)
        return AG_OK;
    if ((largest < AG_STRAIGHT_BELOW && bytes > AG_PINNED_OUT) || is_known(host) ||
        !stage_open(d)) {
        AG_HIP(hipMemcpyAsync(host, src, bytes, hipMemcpyDeviceToHost, d->stream));
        return ag_wait_stream(d);
    }
    int st = AG_OK;
    const size_t chunks = (bytes + AG_STAGE_BYTES - 1) / AG_STAGE_BYTES;
    uint32_t slot[AG_STAGE_SLOTS];
    size_t sent = 0;
    for (size_t c = 0; st == AG_OK && c < chunks; c++) {
        // every slot in flight while a chunk is copied out of the oldest
        for (; st == AG_OK && sent < chunks && sent < c + AG_STAGE_SLOTS; sent++) {
            const size_t o = sent * AG_STAGE_BYTES;
            const size_t len = bytes - o < AG_STAGE_BYTES ? bytes - o : AG_STAGE_BYTES;
            uint32_t k = 0;
            st = stage_slot(d, &k);
            if (st != AG_OK)
                break;
            AG_HIP(hipMemcpyAsync(d->stage + k * AG_STAGE_BYTES, (const char *)src + o, len,
                                  hipMemcpyDeviceToHost, d->stream));
            AG_HIP(hipEventRecord(d->stage_ev[k], d->stream));
            d->stage_used |= 1u << k;
            slot[sent % AG_STAGE_SLOTS] = k;
        }
        if (st != AG_OK)
            break;
        const uint32_t k = slot[c % AG_STAGE_SLOTS];
        st = ag_wait_event(d, d->stage_ev[k]);
        if (st != AG_OK)
            break;
        const size_t o = c * AG_STAGE_BYTES;
        ag_par_copy((char *)host + o, d->stage + k * AG_STAGE_BYTES,
                    bytes - o < AG_STAGE_BYTES ? bytes - o : AG_STAGE_BYTES);
    }
    return st;
}

extern "C" int ag_device_sync(ag_device *d)
{
    if (!d)
        return ag_set_error(AG_ERR_INVALID, "device is null");
    AG_HIP(hipSetDevice(d->ordinal));
    return ag_wait_stream(d);
}

// ------------------------------------------------------------------ graph upload

template <typename T>
static int dev_upload(ag_dgraph *g, T **dst, const T *src, size_t count)
{
    size_t bytes = (count ? count : 1) * sizeof(T);
    AG_HIP(ag_dev_malloc(g->dev, dst, bytes));
    g->device_bytes += bytes;
    if (count)
        AG_HIP(hipMemcpyAsync(*dst, src, count * sizeof(T), hipMemcpyHostToDevice, g->dev->stream));
    return AG_OK;
}

extern "C" int ag_graph_free(ag_dgraph *g)
{
    if (!g)
        return AG_OK;
    (void)hipSetDevice(g->dev->ordinal);
    (void)hipStreamSynchronize(g->dev->stream);
    for (ag_dgraph **q = &g->dev->graphs; *q; q = &(*q)->next)
        if (*q == g) {
            *q = g->next;
            break;
        }
    ag_ppr_free_ws(g);
    ag_parked_free(g);
    void *ptrs[] = {g->d2o, g->off, g->src, g->w, g->wq, g->outdeg, g->tile_row, g->rt, g->seg_row,
                    g->seg_lo, g->seg_hi, g->hub_seg0, g->hub_part, g->vec_a, g->vec_b,
                    g->blk.voff, g->blk.vsrc, g->blk.vw, g->blk.item, g->blk.coff, g->blk.cidx,
                    g->blk.lpos, g->blk.ct_row, g->blk.ct_start, g->blk.ct_pre, g->blk.c_item,
                    g->blk.hgrp, g->blk.vsp, g->blk.tbase,
                    g->vpart, g->btick, g->vwq, g->fwd_off, g->fwd_dst};
    for (void *p : ptrs)
        if (p)
            (void)hipFree(p);
    free(g->h_d2o);
    if (g->dev->live_graphs)
        g->dev->live_graphs--;
    free(g);
    return AG_OK;
}

PullGeom ag_make_geom(const ag_dgraph *g)
{
    PullGeom G;
    G.off = g->off;
    G.src = g->src;
    G.tile_row = g->tile_row;
    G.seg_row = g->seg_row;
    G.seg_lo = g->seg_lo;
    G.seg_hi = g->seg_hi;
    G.hub_seg0 = g->hub_seg0;
    G.hub_part = g->hub_part;
    G.rt = g->rt;
    G.n_rt = g->n_rt;
    G.n_heavy = g->n_heavy;
    G.lane_max = g->params.thread_max_deg > AG_LANE_MAX ? g->params.thread_max_deg : AG_LANE_MAX;
    G.seq_max = g->params.thread_max_deg;
    G.n = g->n;
    G.n_hubs = g->n_hubs;
    G.seq_hubs = g->params.fp32_order == AG_ORDER_REFERENCE ? 1u : 0u;
    for (int b = 0; b <= AG_NBINS; b++)
        G.bin_row[b] = g->bin_row[b];
    for (int s = 0; s <= AG_NSLOTS; s++)
        G.slot_blk0[s] = g->slot_blk0[s];
    return G;
}

PullGeom ag_make_unblocked_geom(const ag_dgraph *g)
{
    PullGeom G = ag_make_geom(g);
    for (int s = 0; s <= AG_NSLOTS; s++)
        G.slot_blk0[s] = g->blk.r_slot_blk0[s];
    if (g->params.blocked_min_bin <= AG_BIN_HUB)
        G.n_hubs = 0;   // hub rows are blocked: their sums come from the combine pass
    return G;
}

BlockGeom ag_make_block_geom(const ag_dgraph *g)
{
    const ag_block_plan &B = g->blk;
    BlockGeom K;
    memset(&K, 0, sizeof(K));
    K.V.off = B.voff;
    K.V.src = B.vsrc;
    K.V.n = B.nv;
    K.C.off = B.coff;
    K.C.src = B.cidx;
    K.C.n = g->n;
    K.item = B.item;
    K.c_item = B.c_item;
    K.ct_row = B.ct_row;
    K.ct_start = B.ct_start;
    K.ct_pre = B.ct_pre;
    K.lpos = B.lpos;
    K.part = g->vpart;
    K.nblocks = B.nblocks;
    for (uint32_t x = 0; x <= AG_NXCD; x++) {
        K.item_off[x] = B.item_off[x];
        K.c_item_off[x] = B.c_item_off[x];
        K.hgrp_off[x] = B.hgrp_off[x];
    }
    for (uint32_t x = 0; x < AG_NXCD; x++)
        K.item_lo[x] = B.item_off[x];
    K.hgrp = B.hgrp;
    K.hot_bits = B.hot_bits;
    K.n_src = g->n;
    K.dyn = g->bdyn;
    K.tick = g->btick;
    K.top0 = B.bits ? B.top0 : g->n;
    K.vsp = B.vsp;
    K.tbase = B.tbase;
    K.sbits = B.bits && B.sorted ? B.bits : 0u;
    K.has_reg = B.r_slot_blk0[AG_NSLOTS] ? 1u : 0u;
    return K;
}

void ag_block_geom_skip_hot(const ag_dgraph *g, BlockGeom &K)
{
    for (uint32_t x = 0; x < AG_NXCD; x++)
        K.item_lo[x] = g->blk.hot_end[x];
}

// Resident four-wave workgroups per CU: the plan's wg_per_cu, by default 4 (16 waves per
// CU), never more than 160 KB of LDS allows. The gathers are bound by the rate of random L2
// requests, and more requests in flight only lengthen the queues (8 per CU measured 5-40%
// slower than 4 on RMAT-25 and ER-25).
static uint32_t wg_per_cu(const ag_dgraph *g, uint32_t lds_bytes, uint32_t dflt = 4u)
{
    uint32_t by_lds = lds_bytes ? (160u * 1024u) / lds_bytes : 32u;
    uint32_t per_cu = g->params.wg_per_cu ? g->params.wg_per_cu : dflt;
    if (per_cu > by_lds)
        per_cu = by_lds;
    return per_cu ? per_cu : 1u;
}

uint32_t ag_blocked_grid(const ag_dgraph *g, uint32_t resident_per_cu, uint32_t default_per_cu)
{
    // workgroup i runs on XCD i % AG_NXCD (round-robin dispatch), so slice x is served by the
    // workgroups with that residue; the grid is a multiple of AG_NXCD
    uint32_t per_cu = g->params.wg_per_cu ? g->params.wg_per_cu : default_per_cu;
    if (per_cu > resident_per_cu)
        per_cu = resident_per_cu;
    uint32_t grid = g->dev->num_cus * (per_cu ? per_cu : 1u) / AG_NXCD * AG_NXCD;
    return grid ? grid : AG_NXCD;
}

uint32_t ag_pull_grid(const ag_dgraph *g, uint32_t lds_bytes, uint32_t default_per_cu)
{
    uint32_t grid = g->dev->num_cus * wg_per_cu(g, lds_bytes, default_per_cu);
    return grid < g->total_blocks ? grid : g->total_blocks;
}

uint32_t ag_tile_grid(const ag_dgraph *g, uint32_t lds_bytes)
{
    const uint32_t grid = g->dev->num_cus * wg_per_cu(g, lds_bytes), items = g->n_heavy + g->n_rt;
    return grid < items ? grid : items;
}

// The largest e in (r, last] with off[e] <= lim, r + 1 if there is none: searched outwards from
// r + guess, the rows of the tile before (rows are ordered by degree class).
static uint32_t tile_end(const uint32_t *off, uint32_t r, uint32_t last, uint64_t lim,
                         uint32_t guess)
{
    if (off[last] <= lim)
        return last;
    uint32_t lo = r, hi = last, step = 4u;   // off[lo] <= lim < off[hi]
    const uint32_t p = guess < last - r ? r + guess : r;
    if (p > r && off[p] <= lim) {
        for (lo = p; hi - lo > step && off[lo + step] <= lim; step *= 2u)
            lo += step;
        hi = hi - lo > step ? lo + step : hi;
    } else if (p > r) {
        for (hi = p; hi - lo > step && off[hi - step] > lim; step *= 2u)
            hi -= step;
        lo = hi - lo > step ? hi - step : lo;
    }
    while (hi - lo > 1u) {
        const uint32_t mid = lo + (hi - lo) / 2u;
        if (off[mid] <= lim)
            lo = mid;
        else
            hi = mid;
    }
    return lo > r ? lo : r + 1u;
}

// Cuts the rows of the bins whose rows fit a tile into row tiles. A tile holds
// at most `nnz` in-edges (one row may hold more, up to AG_TILE_NNZ_MAX) and `rows` rows: as few
// as let the resident workgroups finish in as many rounds as full tiles would need, so that
// small graphs still give every CU work (RMAT-12: 256 in-edges a tile) and the last round is
// not nearly empty. Source-blocked plans, whose sums by the regular schedule are few, take full
// tiles at once. On the host: RMAT-22 2 ms (5 with a search of every tile's whole range).
static int cut_row_tiles(ag_dgraph *g, const uint32_t *off, bool blocked, std::vector<uint4> &rt)
{
    const ag_plan_params &q = g->params;
    // bins are ordered by degree: the first bin whose rows may exceed a tile ends the tiles
    const uint32_t max_deg[] = {q.thread_max_deg, q.group16_max_deg, q.wave_max_deg};
    int bins = 0;
    while (bins < 3 && max_deg[bins] <= AG_TILE_NNZ_MAX)
        bins++;
    const uint32_t row1 = g->bin_row[bins];
    const uint64_t m1 = g->n ? off[row1] : 0u;
    g->n_heavy = g->slot_blk0[AG_NSLOTS - bins];   // slots run from the heaviest bin down
    const uint64_t slots = (uint64_t)g->dev->num_cus * (q.wg_per_cu ? q.wg_per_cu : 4u);
    const uint64_t items = m1 / AG_TILE_NNZ_MAX + row1 / AG_TILE_ROWS_MAX + g->n_heavy + 1u;
    const uint64_t rounds = (items + slots - 1) / slots;
    try {
        const uint64_t budget = slots * rounds, room = budget - g->n_heavy;
        // items covers n_heavy: room > 0
        uint64_t nnz = blocked ? q.tile_nnz : (m1 + room - 1u) / room;
        for (nnz = nnz < AG_WG ? AG_WG : nnz;; nnz += nnz / 8u) {
            nnz = nnz < q.tile_nnz ? nnz : q.tile_nnz;
            const uint32_t rows = q.tile_rows < nnz ? q.tile_rows
                                                    : nnz < AG_WG ? AG_WG : (uint32_t)nnz;
            const bool last_try = nnz == q.tile_nnz;
            rt.clear();
            uint32_t r = 0, guess = 0;
            while (r < row1 && (last_try || rt.size() + g->n_heavy < budget)) {
                const uint32_t last = row1 - r < rows ? row1 : r + rows;
                const uint32_t e = tile_end(off, r, last, (uint64_t)off[r] + nnz, guess);
                rt.push_back(make_uint4(r, e, off[r], off[e]));
                guess = e - r;
                r = e;
            }
            if (r >= row1)
                break;
        }
    } catch (const std::bad_alloc &) {
        return ag_set_error(AG_ERR_OOM, "host allocation failed");
    }
    g->n_rt = (uint32_t)rt.size();
    return AG_OK;
}

// vec_a / vec_b: two scratch arrays of `bytes` each, used to permute SpMV/gather vectors
// between original and device order.
int ag_ensure_vec(ag_dgraph *g, size_t bytes)
{
    if (g->vec_bytes >= bytes)
        return AG_OK;
    if (g->vec_a)
        AG_HIP(hipFree(g->vec_a));
    if (g->vec_b)
        AG_HIP(hipFree(g->vec_b));
    g->vec_a = g->vec_b = NULL;
    g->vec_bytes = 0;
    AG_HIP(ag_dev_malloc(g->dev, &g->vec_a, bytes));
    AG_HIP(ag_dev_malloc(g->dev, &g->vec_b, bytes));
    g->vec_bytes = bytes;
    return AG_OK;
}

extern "C" int ag_graph_upload(ag_device *dev, uint32_t n, uint32_t m, const uint32_t *out_degree,
                               const uint32_t *inv_edges_idx, const uint32_t *inv_degree,
                               const uint32_t *inv_src, const float *inv_weight,
                               const ag_plan_params *params, ag_dgraph **out)
{
    if (!dev || !out)
        return ag_set_error(AG_ERR_INVALID, "device or out is null");
    *out = NULL;
    ag_plan plan;
    const char *msg = "";
    int st = ag_plan_build(n, m, out_degree, inv_edges_idx, inv_degree, inv_src, inv_weight,
                           params, &plan, &msg);
    if (st != AG_OK)
        return ag_set_error(st, "graph upload rejected: %s", msg);
    ag_dgraph *g = (ag_dgraph *)calloc(1, sizeof(ag_dgraph));
    if (!g) {
        ag_plan_free(&plan);
        return ag_set_error(AG_ERR_OOM, "host allocation failed");
    }
    g->dev = dev;
    g->next = dev->graphs;
    dev->graphs = g;
    dev->live_graphs++;
    g->params = plan.params;
    g->n = plan.n;
    g->m = plan.m;
    memcpy(g->bin_row, plan.bin_row, sizeof(g->bin_row));
    memcpy(g->bin_edges, plan.bin_edges, sizeof(g->bin_edges));
    memcpy(g->bin_blocks, plan.bin_blocks, sizeof(g->bin_blocks));
    memcpy(g->slot_blk0, plan.slot_blk0, sizeof(g->slot_blk0));
    g->total_blocks = plan.total_blocks;
    g->n_tiles = plan.n_tiles;
    g->n_hubs = plan.n_hubs;
    g->n_segs = plan.n_segs;

    hipError_t he = hipSetDevice(dev->ordinal);
    st = he == hipSuccess ? AG_OK : ag_hip_fail(he, "hipSetDevice", __FILE__, __LINE__);
    if (st == AG_OK) {
        g->h_d2o = (uint32_t *)malloc((size_t)(plan.n ? plan.n : 1) * sizeof(uint32_t));
        if (!g->h_d2o)
            st = ag_set_error(AG_ERR_OOM, "host allocation failed");
        else
            memcpy(g->h_d2o, plan.d2o, (size_t)plan.n * sizeof(uint32_t));
    }
    if (st == AG_OK) st = dev_upload(g, &g->d2o, plan.d2o, plan.n);
    if (st == AG_OK) st = dev_upload(g, &g->off, plan.off, (size_t)plan.n + 1);
    if (st == AG_OK) st = dev_upload(g, &g->src, plan.src, plan.m);
    if (st == AG_OK && plan.w) st = dev_upload(g, &g->w, plan.w, plan.m);
    if (st == AG_OK) st = dev_upload(g, &g->outdeg, plan.outdeg, plan.n);
    if (st == AG_OK) st = dev_upload(g, &g->tile_row, plan.tile_row, (size_t)plan.n_tiles + 1);
    std::vector<uint4> rt;   // outlives its copy: freed after the wait below
    if (st == AG_OK) st = cut_row_tiles(g, plan.off, plan.blk.bits != 0u, rt);
    if (st == AG_OK) st = dev_upload(g, &g->rt, rt.data(), rt.size());
    if (st == AG_OK) st = dev_upload(g, &g->seg_row, plan.seg_row, plan.n_segs);
    if (st == AG_OK) st = dev_upload(g, &g->seg_lo, plan.seg_lo, plan.n_segs);
    if (st == AG_OK) st = dev_upload(g, &g->seg_hi, plan.seg_hi, plan.n_segs);
    if (st == AG_OK) st = dev_upload(g, &g->hub_seg0, plan.hub_seg0, (size_t)plan.n_hubs + 1);
    if (st == AG_OK) {
        size_t pb = (size_t)(plan.n_segs ? plan.n_segs : 1) * sizeof(uint64_t);
        he = ag_dev_malloc(dev, &g->hub_part, pb);
        if (he != hipSuccess)
            st = ag_hip_fail(he, "hub scratch allocation", __FILE__, __LINE__);
        g->device_bytes += pb;
    }
    if (st == AG_OK && plan.blk.bits) {
        const ag_block_plan &B = plan.blk;
        g->blk = B;   // scalars; the pointers are replaced by device copies below
        g->blk.voff = g->blk.vsrc = g->blk.item = g->blk.coff = g->blk.cidx = NULL;
        g->blk.ct_row = g->blk.ct_start = g->blk.ct_pre = g->blk.c_item = NULL;
        g->blk.lpos = NULL;
        g->blk.vw = NULL;
        g->blk.hgrp = NULL;
        g->blk.vsp = g->blk.tbase = NULL;
        g->blk.hot_seg = NULL;   // host-only array of the plan, freed with it
        const size_t nt = B.c_n_tiles, nb = B.nblocks;
        st = dev_upload(g, &g->blk.voff, B.voff, (size_t)B.nv + 1);
        // with sorted tiles pass 1 reads only the packed ids (vsp): the ids in virtual-row
        // order stay on the host (4 bytes per blocked in-edge less in HBM)
        if (st == AG_OK && !B.sorted) st = dev_upload(g, &g->blk.vsrc, B.vsrc, B.mb);
        if (st == AG_OK && B.vw) st = dev_upload(g, &g->blk.vw, B.vw, B.mb);
        if (st == AG_OK) st = dev_upload(g, &g->blk.item, B.item, (size_t)B.n_items * 2);
        if (st == AG_OK) st = dev_upload(g, &g->blk.coff, B.coff, (size_t)plan.n + 1);
        if (st == AG_OK) st = dev_upload(g, &g->blk.cidx, B.cidx, B.nv);
        if (st == AG_OK) st = dev_upload(g, &g->blk.lpos, B.lpos, B.nv);
        if (st == AG_OK) st = dev_upload(g, &g->blk.ct_row, B.ct_row, nt * 2);
        if (st == AG_OK) st = dev_upload(g, &g->blk.ct_start, B.ct_start, nt * nb);
        if (st == AG_OK) st = dev_upload(g, &g->blk.ct_pre, B.ct_pre, nt * (nb + 1));
        if (st == AG_OK) st = dev_upload(g, &g->blk.c_item, B.c_item, (size_t)B.c_n_items * 2);
        if (st == AG_OK && B.n_hgrp) st = dev_upload(g, &g->blk.hgrp, B.hgrp, (size_t)B.n_hgrp * 3);
        if (st == AG_OK && B.sorted) st = dev_upload(g, &g->blk.vsp, B.vsp, B.mb);
        if (st == AG_OK && B.sorted) st = dev_upload(g, &g->blk.tbase, B.tbase, B.n_items);
        if (st == AG_OK) {
            size_t pb = (size_t)(B.nv ? B.nv : 1) * sizeof(uint64_t);
            he = ag_dev_malloc(dev, &g->vpart, pb);
            if (he != hipSuccess)
                st = ag_hip_fail(he, "partial-sum allocation", __FILE__, __LINE__);
            g->device_bytes += pb;
        }
        if (st == AG_OK) {
            // tickets only when pass 1 holds tiles alone (no AG_ITEM_REG item, whose FP64
            // error terms go to the running workgroup's partial); by default when the pieces
            // are at least half the in-edges (sources spread evenly over the blocks: there a
            // fixed round-robin lets the XCD's workgroups drift over more blocks than its L2
            // holds; on skewed graphs it measured faster)
            uint32_t reg = 0;
            for (uint32_t i = 0; i < B.n_items; i++)
                reg |= (B.item[2 * i + 1] & 15u) == AG_ITEM_REG;
            const uint32_t order = g->params.tile_order;
            g->bdyn = !reg && (order == AG_TILES_TICKET ||
                               (order == AG_TILES_AUTO && 2ull * B.nv >= B.mb));
            const size_t tb = 2 * AG_NXCD * sizeof(uint32_t);
            he = ag_dev_malloc(dev, &g->btick, tb);
            if (he == hipSuccess)
                he = hipMemsetAsync(g->btick, 0, tb, dev->stream);
            if (he != hipSuccess)
                st = ag_hip_fail(he, "ticket counter allocation", __FILE__, __LINE__);
            g->device_bytes += tb;
        }
    }
    // the host plan arrays must outlive the asynchronous copies, also those before a failure
    if (st == AG_OK)
        st = ag_wait_stream(dev);
    if (st != AG_OK)
        (void)hipStreamSynchronize(dev->stream);
    ag_plan_free(&plan);
    if (st != AG_OK) {
        ag_graph_free(g);
        return st;
    }
    *out = g;
    return AG_OK;
}

extern "C" int ag_graph_set_fixed_weights(ag_dgraph *g, const uint32_t *inv_edges_idx,
                                          const uint32_t *inv_degree, const uint32_t *wq)
{
    if (!g || (g->n && (!inv_edges_idx || !inv_degree)) || (g->m && !wq))
        return ag_set_error(AG_ERR_INVALID, "null argument");
    uint64_t total = 0;
    for (uint32_t r = 0; r < g->n; r++)
        total += inv_degree[g->h_d2o[r]];
    if (total != g->m)
        return ag_set_error(AG_ERR_INVALID, "degrees do not match the uploaded graph");
    uint32_t *buf = (uint32_t *)malloc((size_t)(g->m ? g->m : 1) * sizeof(uint32_t));
    if (!buf)
        return ag_set_error(AG_ERR_OOM, "host allocation failed");
    uint64_t o = 0;
    for (uint32_t r = 0; r < g->n; r++) {
        uint32_t v = g->h_d2o[r];
        memcpy(buf + o, wq + inv_edges_idx[v], (size_t)inv_degree[v] * sizeof(uint32_t));
        o += inv_degree[v];
    }
    hipError_t e = hipSetDevice(g->dev->ordinal);
    if (e == hipSuccess && !g->wq) {
        e = ag_dev_malloc(g->dev, &g->wq, (size_t)(g->m ? g->m : 1) * sizeof(uint32_t));
        if (e == hipSuccess)
            g->device_bytes += (size_t)g->m * sizeof(uint32_t);
    }
    if (e == hipSuccess && g->m)
        e = hipMemcpyAsync(g->wq, buf, (size_t)g->m * sizeof(uint32_t), hipMemcpyHostToDevice,
                           g->dev->stream);
    int st = (e == hipSuccess) ? ag_wait_stream(g->dev)
                               : ag_hip_fail(e, "fixed weight upload", __FILE__, __LINE__);
    if (st != AG_OK)
        (void)hipStreamSynchronize(g->dev->stream);   // buf must outlive its copy
    free(buf);
    if (st == AG_OK)
        g->wq_user = 1;
    return st;
}

extern "C" int ag_graph_get_info(const ag_dgraph *g, ag_graph_info *info)
{
    if (!g || !info)
        return ag_set_error(AG_ERR_INVALID, "graph or info is null");
    memset(info, 0, sizeof(*info));
    info->num_vertices = g->n;
    info->num_edges = g->m;
    for (int b = 0; b < AG_NBINS; b++) {
        info->bin_rows[b] = g->bin_row[b + 1] - g->bin_row[b];
        info->bin_edges[b] = g->bin_edges[b];
        info->bin_blocks[b] = g->bin_blocks[b];
    }
    info->num_tiles = g->n_tiles;
    info->num_segments = g->n_segs;
    info->has_weights = g->w != NULL;
    info->device_bytes = g->device_bytes;
    for (uint32_t i = 0; i < g->parked.n_dev; i++)
        info->device_bytes += g->parked.bytes[i];
    info->params = g->params;
    info->src_block_bits = g->blk.bits;
    info->src_blocks = g->blk.nblocks;
    info->virtual_rows = g->blk.nv;
    info->blocked_row0 = g->blk.bits ? g->blk.row0 : g->n;
    info->hot_segments = g->blk.n_hot;
    info->hot_segment_bits = g->blk.hot_bits;
    info->hot_edges = g->blk.hot_edges;
    info->top_sources = g->blk.bits && g->blk.top0 < g->n ? g->n - g->blk.top0 : 0u;
    info->top_edges = info->top_sources ? g->blk.top_edges : 0u;
    info->sorted_tiles = g->blk.bits && g->blk.sorted ? 1u : 0u;
    return AG_OK;
}

// ------------------------------------------------------------------ copy bandwidth

typedef uint32_t ag_u32x4 __attribute__((ext_vector_type(4)));

__global__ void ag_copy_kernel(const ag_u32x4 *__restrict__ in, ag_u32x4 *__restrict__ out,
                               uint64_t n16)
{
    const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n16; i += stride)
        __builtin_nontemporal_store(__builtin_nontemporal_load(&in[i]), &out[i]);
}

extern "C" int ag_device_copy_bandwidth(ag_device *dev, uint64_t bytes, uint32_t reps, double *gbps)
{
    if (!dev || !gbps || bytes < 16 || reps == 0)
        return ag_set_error(AG_ERR_INVALID, "bad argument");
    AG_HIP(hipSetDevice(dev->ordinal));
    const uint64_t n16 = bytes / 16;
    ag_u32x4 *a = NULL, *b = NULL;
    AG_HIP(ag_dev_malloc(dev, &a, n16 * 16));
    hipError_t e = ag_dev_malloc(dev, &b, n16 * 16);
    hipEvent_t e0 = NULL, e1 = NULL;
    if (e == hipSuccess)
        e = hipMemsetAsync(a, 1, n16 * 16, dev->stream);
    if (e == hipSuccess)
        e = hipEventCreate(&e0);
    if (e == hipSuccess)
        e = hipEventCreate(&e1);
    const uint32_t grid = dev->num_cus * 8;
    if (e == hipSuccess) {
        ag_copy_kernel<<<grid, 256, 0, dev->stream>>>(a, b, n16);  // warm-up
        e = hipEventRecord(e0, dev->stream);
    }
    for (uint32_t r = 0; r < reps && e == hipSuccess; r++) {
        ag_copy_kernel<<<grid, 256, 0, dev->stream>>>(a, b, n16);
        e = hipGetLastError();
    }
    if (e == hipSuccess)
        e = hipEventRecord(e1, dev->stream);
    int st = (e == hipSuccess) ? ag_wait_stream(dev) : ag_hip_fail(e, "copy bandwidth", __FILE__, __LINE__);
    if (st == AG_OK) {
        float ms = 0.0f;
        e = hipEventElapsedTime(&ms, e0, e1);
        if (e != hipSuccess)
            st = ag_hip_fail(e, "hipEventElapsedTime", __FILE__, __LINE__);
        else
            *gbps = (double)(2 * n16 * 16) * reps / ((double)ms * 1e-3) / 1e9;
    }
    if (e0)
        (void)hipEventDestroy(e0);
    if (e1)
        (void)hipEventDestroy(e1);
    (void)hipFree(a);
    if (b)
        (void)hipFree(b);
    return st;
}

// ------------------------------------------------------------------ fixed-point test hooks

__global__ void fixed_encode_kernel(uint32_t bits, const float *in, uint64_t *out, uint32_t n)
{
    uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n)
        return;
    float x = in[i];
    uint64_t q;
    if (bits == 64)
        q = ag_dev_double_to_fixed64((double)x);
    else if (bits == 32)
        q = ag_dev_float_to_fixed32(x);
    else if (bits == 16)
        q = ag_dev_float_to_fixed16(x);
    else
        q = ag_dev_float_to_fixed8(x);
    out[i] = q;
}

__global__ void fixed_decode_kernel(uint32_t bits, const uint64_t *in, double *out, uint32_t n)
{
    uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n)
        return;
    uint64_t q = in[i];
    double v;
    if (bits == 64)
        v = ag_dev_fixed64_to_double(q);
    else if (bits == 32)
        v = (double)ag_dev_fixed32_to_float(q);
    else if (bits == 16)
        v = (double)ag_dev_fixed16_to_float(q);
    else
        v = (double)ag_dev_fixed8_to_float(q);
    out[i] = v;
}

static int check_bits(uint32_t bits)
{
    if (bits != 64 && bits != 32 && bits != 16 && bits != 8)
        return ag_set_error(AG_ERR_INVALID, "fixed-point width must be 64, 32, 16 or 8 (got %u)", bits);
    return AG_OK;
}

extern "C" int ag_fixed_encode(ag_device *dev, uint32_t bits, const float *in, uint64_t *out, uint32_t n)
{
    if (!dev || (n && (!in || !out)))
        return ag_set_error(AG_ERR_INVALID, "null argument");
    int st = check_bits(bits);
    if (st != AG_OK || n == 0)
        return st;
    AG_HIP(hipSetDevice(dev->ordinal));
    float *din = NULL;
    uint64_t *dout = NULL;
    AG_HIP(ag_dev_malloc(dev, &din, (size_t)n * sizeof(float)));
    hipError_t e = ag_dev_malloc(dev, &dout, (size_t)n * sizeof(uint64_t));
    if (e == hipSuccess)
        e = hipMemcpyAsync(din, in, (size_t)n * sizeof(float), hipMemcpyHostToDevice, dev->stream);
    if (e == hipSuccess) {
        fixed_encode_kernel<<<(n + 255) / 256, 256, 0, dev->stream>>>(bits, din, dout, n);
        e = hipGetLastError();
    }
    if (e == hipSuccess)
        e = hipMemcpyAsync(out, dout, (size_t)n * sizeof(uint64_t), hipMemcpyDeviceToHost, dev->stream);
    int rc = (e == hipSuccess) ? ag_wait_stream(dev) : ag_hip_fail(e, "fixed encode", __FILE__, __LINE__);
    (void)hipFree(din);
    if (dout)
        (void)hipFree(dout);
    return rc;
}

extern "C" int ag_fixed_decode(ag_device *dev, uint32_t bits, const uint64_t *in, double *out, uint32_t n)
{
    if (!dev || (n && (!in || !out)))
        return ag_set_error(AG_ERR_INVALID, "null argument");
    int st = check_bits(bits);
    if (st != AG_OK || n == 0)
        return st;
    AG_HIP(hipSetDevice(dev->ordinal));
    uint64_t *din = NULL;
    double *dout = NULL;
    AG_HIP(ag_dev_malloc(dev, &din, (size_t)n * sizeof(uint64_t)));
    hipError_t e = ag_dev_malloc(dev, &dout, (size_t)n * sizeof(double));
    if (e == hipSuccess)
        e = hipMemcpyAsync(din, in, (size_t)n * sizeof(uint64_t), hipMemcpyHostToDevice, dev->stream);
    if (e == hipSuccess) {
        fixed_decode_kernel<<<(n + 255) / 256, 256, 0, dev->stream>>>(bits, din, dout, n);
        e = hipGetLastError();
    }
    if (e == hipSuccess)
        e = hipMemcpyAsync(out, dout, (size_t)n * sizeof(double), hipMemcpyDeviceToHost, dev->stream);
    int rc = (e == hipSuccess) ? ag_wait_stream(dev) : ag_hip_fail(e, "fixed decode", __FILE__, __LINE__);
    (void)hipFree(din);
    if (dout)
        (void)hipFree(dout);
    return rc;
}
