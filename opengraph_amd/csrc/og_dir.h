/*
 * og_dir.h -- the direct pull (og_dir.hip, og_dir.c): the iterations of a
 * small graph in one persistent launch.
 *
 * Rows (new ids, the plan's CSR order kept) are packed into bins, one bin per
 * block, all blocks resident together.  An iteration of a block: gather its
 * in-edges' contributions from memory (they are few enough to stay in the
 * L2s) into LDS in CSR order, add its rows there (og_rowsum.h: the
 * reference's running sums to the bit), update them, store their next
 * contributions, meet the other blocks at a grid barrier.  Source ids, row
 * bounds, out-degrees and ranks stay in registers from one iteration to the
 * next; the last block folds the statistics and applies the stop rule while
 * the others go on.
 */
#ifndef OG_DIR_H
#define OG_DIR_H

#include <stddef.h>
#include <stdint.h>

#include <hip/hip_runtime_api.h>

#include "og_bin.h"
#include "og_internal.h"
#include "og_pr.h"

#ifdef __cplusplus
extern "C" {
#endif

#define OG_DIR_CAP OG_BIN_CAP      /* in-edge values in a block's LDS */
#define OG_DIR_THREADS 512u

/* One bin: rows [row0, row1), CSR positions [pos0, pos0 + cnt); kind
 * OG_BIN_THREAD_ROWS (a thread per row) or OG_BIN_WAVE_ROWS (a wavefront) of
 * at most OG_DIR_CAP in-edges, or OG_BIN_PIECE: one row of more, taken
 * OG_DIR_CAP in-edges at a time. */
typedef struct
{
    uint32_t row0, row1, pos0, cnt, kind, pad[3];
} og_dir_bin;

/* words of the grid barrier's state: per block, then per group of blocks,
 * the iterations it has done; 1 + the iteration that stopped the run; whether
 * a block gave up waiting */
#define OG_DIR_MAX_BLOCKS OG_DIR_THREADS
enum
{
    OG_DIR_GROUP = OG_DIR_MAX_BLOCKS,
    OG_DIR_STOP = OG_DIR_MAX_BLOCKS + 64,
    OG_DIR_FAIL = OG_DIR_MAX_BLOCKS + 128,
    OG_DIR_BAR_WORDS = OG_DIR_MAX_BLOCKS + 192
};

typedef struct og_dir_dev
{
    uint32_t n_bins;         /* blocks */
    uint32_t stats_cap;      /* statistics rows: iteration it writes row it % stats_cap */
    uint32_t spin;           /* polls of the grid barrier before a block gives up */
    uint32_t pad;
    const og_dir_bin *bins;
    uint32_t *bar;           /* OG_DIR_BAR_WORDS */
} og_dir_dev;

typedef struct og_dir_plan
{
    og_dir_dev d;
    void *mem_bins, *mem_bar;
} og_dir_plan;

/* The bins of a plan in CSR order for at most max_edges in-edges, max_row of
 * them in a row; *out stays NULL (and 0 is returned) where the graph does not
 * fit. */
int og_dir_plan_build(const og_plan *pl, int mode, uint32_t max_edges, uint32_t max_row, og_dir_plan **out);
void og_dir_plan_destroy(og_dir_plan *b);
/* Blocks of the kernel the device holds at once. */
uint32_t og_dir_resident(void);
/* Iterations [it0, it0 + n) from the contributions in c0 (it0 even) or c1;
 * ranks in a->r.  bar is zeroed before iteration 0.  With n > 1 the blocks
 * wait for each other, which takes all of them resident: where other work
 * keeps some of them out for `spin` polls, the waiting ones set bar's FAIL
 * word and leave, and the run is to be started again one iteration a launch
 * (n = 1: nothing waits; the statistics are partials for the final
 * reduction, as the other pulls'). */
int og_launch_dir(const og_dir_dev *b, const og_pr_dev *a, int mode, void *c0, void *c1, uint32_t it0, uint32_t n,
                  hipStream_t s);

#ifdef __cplusplus
}
#endif

#endif
