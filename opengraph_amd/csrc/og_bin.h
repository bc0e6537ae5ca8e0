/*
 * og_bin.h -- the binned pull (og_bin.hip, og_bin.c): pageRank.c:998-1011
 * as two streaming passes over an edge layout built once per graph.
 *
 * Rows (new ids, the plan's CSR order kept) are packed into bins whose
 * in-edges fit in one CU's LDS (OG_BIN_CAP values); sources fall in
 * segments of OG_BIN_SEG consecutive ids (their contributions fit in LDS).
 * The edges of bin b whose source lies in segment s form tile (b, s).
 * Entries (one per edge) are stored bin by bin, within a bin tile by tile
 * in segment order, within a tile in any order:
 *   pos[e]  u16  the edge's CSR position minus the bin's first position
 *               (OG_BIN_PAD: a padding entry; each tile is padded to
 *               OG_BIN_TILE_ALIGN entries, so every tile's values fill whole
 *               64-byte sectors, written by one block)
 *   val[e]  f32  the gathered contribution, written each iteration
 * The sources are stored in the gather's order instead -- segment by
 * segment, within a segment tile by tile (bins ascending), each tile padded
 * the same way -- so every aligned run of 16 of them (a quad) lies in one
 * tile, and its entries are one run of 16:
 *   src[f]       u16  source id minus the segment's first id
 *   qent[f / 16] u32  the entry of the quad's first source
 * One iteration:
 *   gather pass  one 1024-thread block per CU: per work item (a segment and
 *                a run of its sources), the segment's contributions are
 *                copied into LDS, then val[qent[f / 16] + f % 16] =
 *                lds[src[f]] for the item's sources, 4 consecutive ones
 *                per lane (one 8-byte source load, one quad entry, one
 *                16-byte value store), 256 per wavefront and step.
 *   sum pass     two 512-thread blocks per CU: per bin, val[e] is written
 *                to LDS slot pos[e] (the bin's in-edge values in CSR order),
 *                then every row is added from its slots in order -- the
 *                reference's running sum -- by a thread (rows of at most
 *                OG_BIN_WAVE_ROW in-edges) or a wavefront (longer rows,
 *                dozens of terms per lane and step), and the update runs.
 *                The next bin's entries and row metadata are loaded into
 *                registers while a bin's rows are added.  Rows with more
 *                than OG_BIN_CAP in-edges are cut into pieces of OG_BIN_CAP
 *                (bins of their own, first in the bin list), which one block
 *                takes one after the other.
 * Every row is therefore summed in the reference's order: the fp32 pull is
 * bit-exact, and every global access is a streaming one.
 */
#ifndef OG_BIN_H
#define OG_BIN_H

#include <stddef.h>
#include <stdint.h>

#include <hip/hip_runtime_api.h>

#include "og_internal.h"
#include "og_pr.h"

#ifdef __cplusplus
extern "C" {
#endif

#define OG_BIN_SEG 39936u      /* sources per segment: 156 KB of fp32 in LDS */
#define OG_BIN_CAP 19968u      /* in-edge values per bin: 78 KB of LDS, two bins per CU */
#define OG_BIN_PAD 0xFFFFu     /* pos of a padding entry */
/* rows with more in-edges are added by a wavefront (1024: 3 % slower at
 * R-MAT-24, the same at 20-22; fewer in small bins); the integer modes' bins take any number of
 * lanes per row instead */
#define OG_BIN_WAVE_ROW 2048u
#define OG_BIN_RPT 1u          /* rows per thread and bin: a bin holds at most RPT * THREADS rows */
#define OG_BIN_TILE_ALIGN 16u  /* tiles padded to 16 entries: 64-byte value runs */
#define OG_BIN_ITEM_SRC (2048u * 64u) /* sources per gather work item at most */
#define OG_BIN_SPARE 256u      /* spare entries past the last tile (the gather's idle stores) */
#define OG_BIN_THREADS 512u    /* sum blocks (two per CU) */
#define OG_BIN_GTHREADS 1024u  /* gather blocks (one per CU: a segment fills LDS) */

enum { OG_BIN_THREAD_ROWS = 0, OG_BIN_WAVE_ROWS = 1, OG_BIN_PIECE = 2 };

/* One bin: rows [row0, row1) (a piece: the long row row0, and in row1
 * whether it is the row's first and last piece), entries [ent0, ent1) (ent1 - ent0
 * a multiple of 16), first CSR position pos0, cnt in-edges. */
typedef struct
{
    uint32_t row0, row1, ent0, ent1;
    uint32_t pos0, kind, pad, cnt;
} og_bin_desc;

#define OG_BIN_FIRST 1u
#define OG_BIN_LAST 2u

/* Gather work item: segment seg, sources [f0, f1) (f0 and f1 multiples
 * of 16, within the segment's sources). */
typedef struct
{
    uint32_t seg, f0, f1, pad;
} og_bin_item;

/* Everything the binned kernels read, by value. */
typedef struct og_bin_dev
{
    uint32_t N, n_seg, n_items, n_bins, n_bins_live;
    uint32_t first_bin;          /* bins [0, first_bin) are the long rows' pieces */
    uint32_t n_edge_bins;        /* the bins past them hold the rows without in-edges */
    uint32_t n_ent;              /* entries in tiles; OG_BIN_SPARE spare ones follow */
    const og_bin_item *items;
    const uint32_t *qent;        /* n_ent / 16 */
    const uint16_t *src, *pos;
    float *val;
    const og_bin_desc *bins;
    const og_bin_desc *sched;    /* the bins with edges in the sum pass's order */
    const uint32_t *blk;         /* block i of the sum pass takes sched[blk[i], blk[i + 1]) */
} og_bin_dev;

typedef struct og_bin_plan
{
    og_bin_dev d;
    uint64_t n_ent;              /* entries (and sources) including padding and the spares */
    uint32_t n_zero_bins;
    uint32_t sum_grid;           /* blocks of the sum pass (its statistics partials) */
    /* device allocations */
    void *mem_items, *mem_qent, *mem_src, *mem_pos, *mem_val, *mem_bins;
    void *mem_sched, *mem_blk;
} og_bin_plan;

/* Runs of rows of one in-degree: the first row and the in-degree. */
typedef struct
{
    uint32_t row, deg;
} og_bin_run;
/* The runs of a plan's rows [0, Z), ascending (malloc'ed). */
int og_bin_runs(const og_plan *pl, og_bin_run **runs, size_t *n);
/* The longest row of the runs. */
static inline uint32_t og_bin_longest(const og_bin_run *run, size_t n)
{
    uint32_t most = 0;
    for (size_t i = 0; i < n; i++) most = run[i].deg > most ? run[i].deg : most;
    return most;
}

/* Builds the binned layout of a plan whose rows keep the reference's
 * in-neighbour order (relabel 2 or 0).  Not built (*out stays NULL, 0 is
 * returned) where a row has more than max_row in-edges or the tiles, padding
 * included, more than max_entries entries. */
int og_bin_plan_build(const og_plan *pl, int mode, uint32_t max_row, uint64_t max_entries, og_bin_plan **out);
void og_bin_plan_destroy(og_bin_plan *b);

/* Arithmetic the binned and direct pulls run in: 32-bit gathered elements,
 * fp32 sums in the reference's order or u64 sums (OG_MODE_FX64 gathers the fp32
 * quotients and converts them where they are added). */
static inline int og_bin_mode(int mode)
{
    return mode == OG_MODE_F32 || mode == OG_MODE_FX64 || mode == OG_MODE_FX32 || mode == OG_MODE_Q32;
}

/* One binned pull iteration in `mode`: gather, then the sum pass; ev0 / ev1 (may be
 * NULL) bracket them.  Statistics partials: the sum pass's blocks; then the
 * final reduction. */
int og_launch_bin_pull(const og_bin_dev *b, const og_pr_dev *a, int mode, uint32_t sum_grid, hipStream_t s,
                       hipEvent_t ev0, hipEvent_t ev1);

/* plan-build kernels (og_bin.hip): the rows' runs of equal in-degree
 * (pairs row, in-degree; *n zeroed by the caller), the tiles' sizes, their
 * places, the entries */
int og_launch_bin_runs(const uint32_t *row_ptr, uint32_t Z, uint32_t *runs, uint32_t cap, uint32_t *n, hipStream_t s);
int og_launch_bin_count(const og_bin_desc *bins, uint32_t n_bins, const uint32_t *cols, uint32_t n_seg,
                        uint32_t *quads, uint32_t *bin_quads, hipStream_t s);
int og_launch_bin_place(og_bin_desc *bins, uint32_t n_bins, uint32_t n_all, const uint32_t *bin_quads,
                        const uint32_t *quads, uint32_t n_seg, uint32_t *seg_src, hipStream_t s);
int og_launch_bin_sched(const og_bin_desc *bins, const uint32_t *order, uint32_t n, og_bin_desc *sched,
                        hipStream_t s);
int og_launch_bin_fill(const og_bin_desc *bins, uint32_t n_bins, const uint32_t *cols, uint32_t n_seg,
                       const uint32_t *quads, uint16_t *src, uint16_t *pos, uint32_t *qent, hipStream_t s);

#ifdef __cplusplus
}
#endif

#endif
