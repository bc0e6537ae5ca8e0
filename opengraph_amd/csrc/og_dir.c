/*
 * og_dir.c -- host side of the direct pull (og_dir.h): the rows of a small
 * graph packed into one bin per block.
 */
#include <stdlib.h>
#include <string.h>

#include "og_dir.h"
#include "og_internal.h"
#include "og_plan.h"

/* In-edges a block aims at: eight per thread.  More blocks make the grid
 * barrier longer, fewer leave CUs idle. */
#define OG_DIR_EDGES 4096u
/* Rows of more in-edges are added by a wavefront: a thread takes about 13
 * cycles a term, which the whole grid waits for.  In the integer modes all of a
 * block adds a row that is alone in it (every row of more than OG_DIR_EDGES is):
 * u64 pull, R-MAT-17 with 6 M edges 92 us an iteration by one wavefront, now
 * 39; one row of 210 k among 1 M edges 317 and 118. */
#define OG_DIR_WAVE_ROW OG_CH
#define OG_DIR_WAVE_ROW_INT 128u

void og_dir_plan_destroy(og_dir_plan *b)
{
    if (!b) return;
    og_dfree(b->mem_bins);
    og_dfree(b->mem_bar);
    free(b);
}

/* Bins of at most cap in-edges (or one row) into out (room for most);
 * returns their number, most + 1 when there are more. */
static uint32_t og_dir_pack(const og_bin_run *run, size_t n_runs, uint32_t Z, uint32_t cap, uint32_t wave_row,
                            og_dir_bin *out, uint32_t most)
{
    uint32_t n = 0, pos = 0;
    og_dir_bin *d = NULL;   /* the open bin */
    for (size_t i = 0; i < n_runs; i++)
    {
        const uint32_t r1 = i + 1 < n_runs ? run[i + 1].row : Z, deg = run[i].deg;
        const uint32_t kind = deg > OG_DIR_CAP ? OG_BIN_PIECE
                            : deg > wave_row ? OG_BIN_WAVE_ROWS : OG_BIN_THREAD_ROWS;
        uint32_t r = run[i].row;
        while (r < r1)
        {
            uint32_t room = 0;
            if (d && d->kind == kind)
            {
                room = !d->cnt ? (deg > cap || kind == OG_BIN_PIECE ? 1 : cap / deg)
                     : d->cnt < cap && kind != OG_BIN_PIECE ? (cap - d->cnt) / deg : 0;
                if (room > OG_DIR_THREADS - (d->row1 - d->row0)) room = OG_DIR_THREADS - (d->row1 - d->row0);
            }
            if (!room)
            {
                if (n == most) return most + 1;
                d = &out[n++];
                memset(d, 0, sizeof(*d));
                d->row0 = d->row1 = r;
                d->pos0 = pos;
                d->kind = kind;
                continue;
            }
            if (room > r1 - r) room = r1 - r;
            d->row1 += room;
            d->cnt += room * deg;
            pos += room * deg;
            r += room;
        }
    }
    return n;
}

int og_dir_plan_build(const og_plan *pl, int mode, uint32_t max_edges, uint32_t max_row, og_dir_plan **out)
{
    *out = NULL;
    const uint32_t E = pl->E, N = pl->N, Z = pl->Z;
    const uint32_t most = og_dir_resident();
    /* rows sorted within chunks are out of CSR order; past max_edges, or with
     * more rows than the resident threads, the streaming passes win */
    if (!E || !N || !most || E > max_edges || (pl->relabel == 1 && pl->H) || Z > most * OG_DIR_THREADS) return 0;
    og_dir_plan *b = (og_dir_plan *)calloc(1, sizeof(*b));
    og_dir_bin *bins = (og_dir_bin *)malloc((size_t)most * sizeof(og_dir_bin));
    og_bin_run *run = NULL;
    size_t n_runs = 0;
    int rc = -1;
    if (!b || !bins)
    {
        og_set_error("out of host memory");
        goto done;
    }
    if (og_bin_runs(pl, &run, &n_runs)) goto done;
    uint32_t n = most + 1;
    /* A plan in the caller's order groups its rows at OG_CH only, a bin holds one
     * kind, and another line cuts one at every other row: u32 pull, R-MAT-16, 28 us
     * an iteration with the integer line, 15 without; a thread takes long over a
     * u64 row, so small graphs keep it there (R-MAT-12 14 and 25, R-MAT-17 50
     * and 32). */
    const int by_degree_line = pl->relabel || (mode == OG_MODE_FX64 && E < (1u << 21));
    const uint32_t wave_row = mode != OG_MODE_F32 && by_degree_line ? OG_DIR_WAVE_ROW_INT : OG_DIR_WAVE_ROW;
    const int fits = og_bin_longest(run, n_runs) <= max_row;
    for (uint64_t cap = OG_DIR_EDGES; fits && n > most && cap <= OG_DIR_CAP; cap += cap / 4)
        if ((uint64_t)E <= cap * most) n = og_dir_pack(run, n_runs, Z, (uint32_t)cap, wave_row, bins, most);
    if (n > most)
    {
        rc = 0;
        og_dir_plan_destroy(b);
        b = NULL;
        goto done;
    }
    b->d.n_bins = n;
    /* polls of the barrier before a block gives up: a poll (64 cycles of sleep and
     * a round trip to memory) takes upwards of half a microsecond, an iteration
     * microseconds, or up to 0.55 ns per in-edge of its longest block, so some 10
     * ms and a few times the latter (OG_DIR_SPIN: another limit, small ones for
     * tests of the fallback) */
    uint32_t most_edges = 0;
    for (uint32_t i = 0; i < n; i++) most_edges = bins[i].cnt > most_edges ? bins[i].cnt : most_edges;
    const char *spin = getenv("OG_DIR_SPIN");
    b->d.spin = spin ? (uint32_t)strtoul(spin, NULL, 10) : (1u << 14) + most_edges / 256;
    b->mem_bins = og_dalloc((size_t)n * sizeof(og_dir_bin));
    b->mem_bar = og_dalloc(OG_DIR_BAR_WORDS * 4);
    if (!b->mem_bins || !b->mem_bar ||
        og_hip_check(og_copy(b->mem_bins, bins, (size_t)n * sizeof(og_dir_bin), hipMemcpyHostToDevice), "H2D bins"))
        goto done;
    b->d.bins = (const og_dir_bin *)b->mem_bins;
    b->d.bar = (uint32_t *)b->mem_bar;
    rc = 0;
done:
    free(bins);
    free(run);
    if (rc) og_dir_plan_destroy(b);
    else *out = b;
    return rc;
}
