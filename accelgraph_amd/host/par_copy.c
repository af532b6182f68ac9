/*
 * par_copy.c -- host memory copies on all cores, for the staged transfers of ag_runtime.hip.
 *
 * One core copies about 10 GB/s and takes the page faults of a fresh destination one after the
 * other; the link to the GPU moves about 50 GB/s. Copies of 256 KB or more are cut into page runs,
 * one per thread, eight at most (4 and 16 measured the same or slower: 16 MB each way in 1.07,
 * 1.11 and 1.14 ms, 1.2 MB in 0.13 ms with any of them).
 */
#include <omp.h>
#include <string.h>

#include "ag_plan.h"

void ag_par_copy(void *dst, const void *src, size_t bytes)
{
    if (bytes < ((size_t)1 << 18)) {
        memcpy(dst, src, bytes);
        return;
    }
    /* the whole team enters, so that the regions around this one (the planner's) find their
     * threads again: a smaller team ends the others, and starting them took 3 ms of an upload */
    #pragma omp parallel
    {
        const size_t t = (size_t)omp_get_thread_num(), all = (size_t)omp_get_num_threads();
        const size_t n = all < 8 ? all : 8;
        const size_t part = ((bytes + n - 1) / n + 4095) & ~(size_t)4095;
        const size_t lo = t < n && t * part < bytes ? t * part : bytes;
        const size_t hi = lo + part < bytes ? lo + part : bytes;
        if (hi > lo)
            memcpy((char *)dst + lo, (const char *)src + lo, hi - lo);
    }
}
