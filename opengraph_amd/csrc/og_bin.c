/*
 * og_bin.c -- one-time build of the binned pull's edge layout (og_bin.h)
 * from a PageRank plan whose rows keep the reference's in-neighbour order.
 *
 * Device: the runs of equal in-degree of the (in-degree-ordered) rows; the
 * tiles' sizes by a histogram of each bin's segments and their places by
 * prefix sums; then each bin's entries, sources and quads.
 * Host: the rows are packed into bins run by run, the rows of more than
 * OG_BIN_CAP in-edges are cut into pieces, and each segment's sources into
 * work items.
 */
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

#include "og_bin.h"
#include "og_internal.h"
#include "og_plan.h"

#define OG_BIN_ZERO_ROWS (OG_BIN_RPT * OG_BIN_THREADS)   /* rows of a bin of rows without in-edges */

void og_bin_plan_destroy(og_bin_plan *b)
{
    if (!b) return;
    og_dfree(b->mem_items); og_dfree(b->mem_qent); og_dfree(b->mem_src);
    og_dfree(b->mem_pos); og_dfree(b->mem_val); og_dfree(b->mem_bins); og_dfree(b->mem_sched);
    og_dfree(b->mem_blk);
    free(b);
}

/* growable host arrays */
typedef struct
{
    void *p;
    size_t n, cap, elem;
} og_vec;

static void *og_vec_push(og_vec *v)
{
    if (v->n == v->cap)
    {
        size_t c = v->cap ? 2 * v->cap : 1024;
        void *q = realloc(v->p, c * v->elem);
        if (!q) return NULL;
        v->p = q;
        v->cap = c;
    }
    return (char *)v->p + (v->n++) * v->elem;
}

/* Device copy of a host array (NULL and error set on failure). */
static void *og_bin_upload(const void *h, size_t bytes)
{
    void *d = og_dalloc(bytes ? bytes : 16);
    if (!d) return NULL;
    if (bytes && og_hip_check(og_copy(d, h, bytes, hipMemcpyHostToDevice), "H2D bin layout"))
    {
        og_dfree(d);
        return NULL;
    }
    return d;
}

/* Host check of every index the binned kernels derive from the layout
 * (enabled by the environment variable OG_BIN_VERIFY): items within the
 * sources, every source's entry within the entries, each source within its
 * segment, each entry gathered once and its source the edge's (the CSR's
 * column at the entry's slot),
 * slots within their bins, bins and pieces within the entries, rows per bin,
 * CSR positions, the pieces first, and in the sum pass's lists every bin once
 * and each long row's pieces in order.  Runs before any binned kernel, so a bad layout
 * is an error, not a stray access. */
static int og_bin_verify(const og_bin_plan *b, const og_plan *pl, const uint32_t *rp)
{
    const og_bin_dev *d = &b->d;
    const size_t ne = (size_t)b->n_ent, nq = (ne - OG_BIN_SPARE) / OG_BIN_TILE_ALIGN;
    og_bin_item *items = (og_bin_item *)malloc((size_t)d->n_items * sizeof(og_bin_item) + 16);
    uint32_t *qent = (uint32_t *)malloc(nq * 4 + 4);
    uint16_t *src = (uint16_t *)malloc(ne * 2), *pos = (uint16_t *)malloc(ne * 2);
    og_bin_desc *bins = (og_bin_desc *)malloc((size_t)d->n_bins * sizeof(og_bin_desc) + 16);
    og_bin_desc *sched = (og_bin_desc *)malloc((size_t)d->n_edge_bins * sizeof(og_bin_desc) + 16);
    uint32_t *blk = (uint32_t *)malloc(((size_t)b->sum_grid + 1) * 4);
    uint8_t *taken = (uint8_t *)calloc((size_t)d->n_bins + 1, 1);
    uint32_t *gsrc = (uint32_t *)malloc(ne * 4);   /* source id gathered into each entry */
    uint32_t *cols = (uint32_t *)malloc((size_t)pl->E * 4 + 4);
    uint8_t *seen = (uint8_t *)calloc(ne, 1);
    int rc = -1;
#define OG_BIN_FAIL(...) do { og_set_error("binned layout check: " __VA_ARGS__); goto out; } while (0)
    if (!items || !qent || !src || !pos || !bins || !sched || !blk || !taken || !seen || !gsrc || !cols)
        OG_BIN_FAIL("out of host memory");
    if (og_hip_check(og_copy(items, d->items, (size_t)d->n_items * sizeof(og_bin_item), hipMemcpyDeviceToHost), "D2H") ||
        og_hip_check(og_copy(qent, d->qent, nq * 4, hipMemcpyDeviceToHost), "D2H") ||
        og_hip_check(og_copy(src, d->src, ne * 2, hipMemcpyDeviceToHost), "D2H") ||
        og_hip_check(og_copy(pos, d->pos, ne * 2, hipMemcpyDeviceToHost), "D2H") ||
        og_hip_check(og_copy(bins, d->bins, (size_t)d->n_bins * sizeof(og_bin_desc), hipMemcpyDeviceToHost), "D2H") ||
        og_hip_check(og_copy(sched, d->sched, (size_t)d->n_edge_bins * sizeof(og_bin_desc), hipMemcpyDeviceToHost), "D2H") ||
        og_hip_check(og_copy(blk, d->blk, ((size_t)b->sum_grid + 1) * 4, hipMemcpyDeviceToHost), "D2H") ||
        og_hip_check(og_copy(cols, pl->cols, (size_t)pl->E * 4, hipMemcpyDeviceToHost), "D2H"))
        goto out;
    for (uint32_t q = 0; q < d->n_items; q++)
    {
        const og_bin_item it = items[q];
        if (it.seg >= d->n_seg || it.f0 >= it.f1 || it.f1 > nq * OG_BIN_TILE_ALIGN || it.f0 % OG_BIN_TILE_ALIGN ||
            it.f1 % OG_BIN_TILE_ALIGN)
            OG_BIN_FAIL("item %u", q);
        const uint32_t nv = d->N - it.seg * OG_BIN_SEG < OG_BIN_SEG ? d->N - it.seg * OG_BIN_SEG : OG_BIN_SEG;
        for (uint32_t f = it.f0; f < it.f1; f++)
        {
            const uint64_t e = (uint64_t)qent[f / OG_BIN_TILE_ALIGN] + f % OG_BIN_TILE_ALIGN;
            if (e >= ne - OG_BIN_SPARE)
                OG_BIN_FAIL("source %u: entry %llu of %zu", f, (unsigned long long)e, ne - OG_BIN_SPARE);
            if (src[f] >= nv) OG_BIN_FAIL("source %u: %u past segment size %u", f, src[f], nv);
            if (seen[e]) OG_BIN_FAIL("entry %llu gathered twice", (unsigned long long)e);
            seen[e] = 1;
            gsrc[e] = it.seg * OG_BIN_SEG + src[f];
        }
    }
    uint64_t prev_end = 0;
    for (uint32_t q = 0; q < d->n_bins; q++)
    {
        const og_bin_desc bd = bins[q];
        if (bd.ent0 != prev_end || (bd.ent0 % OG_BIN_TILE_ALIGN) || bd.ent1 < bd.ent0 ||
            (bd.ent1 - bd.ent0) % OG_BIN_TILE_ALIGN || bd.ent1 - bd.ent0 < bd.cnt || bd.ent1 > ne - OG_BIN_SPARE ||
            bd.cnt > OG_BIN_CAP)
            OG_BIN_FAIL("bin %u entries [%u, %u) count %u", q, bd.ent0, bd.ent1, bd.cnt);
        prev_end = bd.ent1;
        if ((uint64_t)bd.pos0 + bd.cnt > pl->E) OG_BIN_FAIL("bin %u positions", q);
        if ((bd.kind == OG_BIN_PIECE) != (q < d->first_bin)) OG_BIN_FAIL("bin %u: pieces come first", q);
        if (bd.kind == OG_BIN_PIECE)
        {
            if (bd.row0 >= pl->Z || bd.pos0 < rp[bd.row0] || (uint64_t)bd.pos0 + bd.cnt > rp[bd.row0 + 1])
                OG_BIN_FAIL("piece %u", q);
        }
        else
        {
            if (bd.row0 > bd.row1 || bd.row1 > d->N || bd.row1 - bd.row0 > OG_BIN_RPT * OG_BIN_THREADS)
                OG_BIN_FAIL("bin %u rows", q);
            if (bd.cnt && (rp[bd.row0] != bd.pos0 || rp[bd.row1] - rp[bd.row0] != bd.cnt)) OG_BIN_FAIL("bin %u row offsets", q);
        }
        uint32_t real = 0;
        for (uint32_t e = bd.ent0; e < bd.ent1; e++)
        {
            if (pos[e] != OG_BIN_PAD)
            {
                if (pos[e] >= bd.cnt) OG_BIN_FAIL("entry %u: slot %u in bin %u of %u", e, pos[e], q, bd.cnt);
                if (seen[e] && gsrc[e] != cols[bd.pos0 + pos[e]])
                    OG_BIN_FAIL("entry %u: gathers source %u, the edge's is %u", e, gsrc[e], cols[bd.pos0 + pos[e]]);
                real++;
            }
            if (!seen[e]) OG_BIN_FAIL("entry %u never gathered", e);
        }
        if (real != bd.cnt) OG_BIN_FAIL("bin %u: %u entries for %u in-edges", q, real, bd.cnt);
    }
    /* the sum pass's order: every bin with edges in it once (the bins are
     * told apart by their first entry), a long row's pieces one after the
     * other in one block, the first and the last one marked */
    if (blk[0] != 0 || blk[b->sum_grid] != d->n_edge_bins) OG_BIN_FAIL("block lists");
    for (uint32_t i = 0; i < b->sum_grid; i++)
    {
        if (blk[i + 1] < blk[i] || blk[i + 1] > d->n_edge_bins) OG_BIN_FAIL("block list %u", i);
        uint32_t next = 0;   /* CSR position the long row under way goes on at, 0 for none */
        for (uint32_t q = blk[i]; q < blk[i + 1]; q++)
        {
            uint32_t lo = 0, hi = d->n_edge_bins;
            while (hi - lo > 1)
            {
                const uint32_t mid = (lo + hi) / 2;
                if (bins[mid].ent0 <= sched[q].ent0) lo = mid;
                else hi = mid;
            }
            if (memcmp(&bins[lo], &sched[q], sizeof(og_bin_desc)) || taken[lo]) OG_BIN_FAIL("block %u: bin %u", i, q);
            taken[lo] = 1;
            const og_bin_desc sd = sched[q];
            if (sd.kind != OG_BIN_PIECE)
            {
                if (next) OG_BIN_FAIL("block %u: a long row breaks off at %u", i, q);
                continue;
            }
            const int first = sd.pos0 == rp[sd.row0], last = sd.pos0 + sd.cnt == rp[sd.row0 + 1];
            if ((!first && next != sd.pos0) || (first && next) ||
                sd.row1 != ((first ? OG_BIN_FIRST : 0u) | (last ? OG_BIN_LAST : 0u)))
                OG_BIN_FAIL("block %u: piece %u", i, q);
            next = last ? 0 : sd.pos0 + sd.cnt;
        }
        if (next) OG_BIN_FAIL("block %u: a long row breaks off", i);
    }
    rc = 0;
#undef OG_BIN_FAIL
out:
    free(items); free(qent); free(src); free(pos); free(bins); free(sched); free(blk); free(taken); free(seen);
    free(gsrc); free(cols);
    return rc;
}

/* Runs of equal in-degree of the rows [0, Z): (first row, in-degree),
 * ascending by row; what the packing of rows into bins needs of the row
 * offsets.  A relabelled plan orders its rows by in-degree, so there are at
 * most about sqrt(2 E) runs and the device lists them; a plan in original
 * order (relabel 0) has its row offsets read back instead. */
static int og_bin_run_cmp(const void *a, const void *b)
{
    const uint32_t x = ((const og_bin_run *)a)->row, y = ((const og_bin_run *)b)->row;
    return x < y ? -1 : x > y;
}

static int og_bin_list_runs(const og_plan *pl, og_vec *runs)
{
    const uint32_t Z = pl->Z;
    hipStream_t s = og_stream();
    int rc = -1;
    if (pl->relabel)
    {
        uint64_t cap = 64;
        while (cap * cap < 2ull * pl->E) cap += cap / 8;
        cap += 64;
        uint32_t *d = og_dalloc(16 + cap * sizeof(og_bin_run));
        og_bin_run *h = (og_bin_run *)malloc(16 + cap * sizeof(og_bin_run));
        uint32_t n = 0;
        if (!h) og_set_error("out of host memory");
        if (d && h && !og_launch_fill_u32(d, 0, 4, s) &&
            !og_launch_bin_runs(pl->row_ptr, Z, d + 4, (uint32_t)cap, d, s) &&
            !og_hip_check(og_copy(h, d, 16 + cap * sizeof(og_bin_run), hipMemcpyDeviceToHost), "D2H row runs"))
        {
            n = *(const uint32_t *)h;
            if (n <= cap)
            {
                const og_bin_run *r = (const og_bin_run *)((const char *)h + 16);
                rc = 0;
                for (uint32_t i = 0; i < n && !rc; i++)
                {
                    og_bin_run *o = (og_bin_run *)og_vec_push(runs);
                    if (o) *o = r[i];
                    else { og_set_error("out of host memory"); rc = -1; }
                }
                if (!rc) qsort(runs->p, runs->n, sizeof(og_bin_run), og_bin_run_cmp);
            }
        }
        og_dfree(d);
        free(h);
        if (!rc || n <= cap) return rc;
    }
    uint32_t *rp = (uint32_t *)malloc(((size_t)Z + 1) * 4);
    if (!rp) { og_set_error("out of host memory"); return -1; }
    rc = og_hip_check(og_copy(rp, pl->row_ptr, ((size_t)Z + 1) * 4, hipMemcpyDeviceToHost), "D2H row_ptr");
    for (uint32_t r = 0; r < Z && !rc; r++)
    {
        const uint32_t d = rp[r + 1] - rp[r];
        if (r && d == ((og_bin_run *)runs->p)[runs->n - 1].deg) continue;
        og_bin_run *o = (og_bin_run *)og_vec_push(runs);
        if (!o) { og_set_error("out of host memory"); rc = -1; break; }
        o->row = r;
        o->deg = d;
    }
    free(rp);
    return rc;
}

int og_bin_runs(const og_plan *pl, og_bin_run **runs, size_t *n)
{
    og_vec v = {NULL, 0, 0, sizeof(og_bin_run)};
    const int rc = og_bin_list_runs(pl, &v);
    if (rc) free(v.p);
    *runs = rc ? NULL : (og_bin_run *)v.p;
    *n = rc ? 0 : v.n;
    return rc;
}

/* Bins: first the pieces of the long rows (more than OG_BIN_CAP in-edges;
 * OG_BIN_CAP in-edges each, in CSR order), then consecutive rows of one kind
 * (thread rows, wavefront rows of more than wave_row in-edges) with at
 * most cap <= OG_BIN_CAP in-edges together (or one row of more) and
 * OG_BIN_RPT * OG_BIN_THREADS rows. */
static int og_bin_pack(const og_plan *pl, const og_vec *runs, uint32_t cap, uint32_t wave_row, og_vec *bins)
{
    const og_bin_run *run = (const og_bin_run *)runs->p;
    const uint32_t Z = pl->Z;
    uint32_t pos = 0;
    for (size_t i = 0; i < runs->n; i++)
    {
        const uint32_t r1 = i + 1 < runs->n ? run[i + 1].row : Z, deg = run[i].deg;
        if (deg <= OG_BIN_CAP)
        {
            pos += (r1 - run[i].row) * deg;
            continue;
        }
        for (uint32_t r = run[i].row; r < r1; r++, pos += deg)
            for (uint32_t p0 = 0; p0 < deg; p0 += OG_BIN_CAP)
            {
                og_bin_desc *d = (og_bin_desc *)og_vec_push(bins);
                if (!d) return -1;
                memset(d, 0, sizeof(*d));
                d->row0 = r;
                d->row1 = (p0 == 0 ? OG_BIN_FIRST : 0u) | (deg - p0 <= OG_BIN_CAP ? OG_BIN_LAST : 0u);
                d->pos0 = pos + p0;
                d->kind = OG_BIN_PIECE;
                d->cnt = deg - p0 < OG_BIN_CAP ? deg - p0 : OG_BIN_CAP;
            }
    }
    og_bin_desc *d = NULL;   /* the open bin (the last one) */
    pos = 0;
    for (size_t i = 0; i < runs->n; i++)
    {
        const uint32_t r1 = i + 1 < runs->n ? run[i + 1].row : Z, deg = run[i].deg;
        const uint32_t kind = deg > wave_row ? OG_BIN_WAVE_ROWS : OG_BIN_THREAD_ROWS;
        uint32_t r = run[i].row;
        if (deg > OG_BIN_CAP)
        {
            pos += (r1 - r) * deg;
            d = NULL;
            continue;
        }
        while (r < r1)
        {
            uint32_t room = 0;
            if (d && d->kind == kind)
            {
                room = !d->cnt && deg > cap ? 1 : d->cnt < cap ? (cap - d->cnt) / deg : 0;
                const uint32_t rows = OG_BIN_RPT * OG_BIN_THREADS - (d->row1 - d->row0);
                if (room > rows) room = rows;
            }
            if (!room)
            {
                d = (og_bin_desc *)og_vec_push(bins);
                if (!d) return -1;
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
    return 0;
}

/* In-edges per bin: at least OG_BIN_PER_SLOT bins for each block of the sum
 * pass (its lists are static: with fewer, some blocks have one bin more than
 * others and the rest wait), as long as a tile keeps 64 entries (the tiles
 * are padded to 16) and a bin 4096. */
#define OG_BIN_PER_SLOT 4u
static uint32_t og_bin_cap(uint32_t E, uint32_t n_seg, uint32_t slots)
{
    uint64_t c = (uint64_t)E / ((uint64_t)OG_BIN_PER_SLOT * slots);
    if (c < 64ull * n_seg) c = 64ull * n_seg;
    if (c < 4096) c = 4096;
    return c > OG_BIN_CAP ? OG_BIN_CAP : (uint32_t)c;
}

/* fp32: rows of more in-edges are added by a wavefront: OG_BIN_WAVE_ROW, or a
 * sixth of a bin where a small graph's bins are so small that a few such rows
 * fill one, and the threads' long chains of adds would leave the rest of the
 * block idle (10 k vertices, 16 M edges, bins of 8192, 1680 terms a row: SpMV 97 us a
 * pass by threads, 62 by wavefronts; pull 103 and 78 us an iteration.  An eighth: 20 k
 * vertices with 840 terms a row the same, R-MAT-18 with 10 M edges 3 % slower.) */
static uint32_t og_bin_wave_row(uint32_t cap)
{
    return cap / 6 < OG_BIN_WAVE_ROW ? cap / 6 : OG_BIN_WAVE_ROW;
}

/* The sum pass's order: the bins dealt in their order (the long rows, the
 * longest ones, come first) to the block with the least so far, a long row's
 * pieces to one block.  order: the bins block by block; blk: where each
 * block's begin. */
typedef struct
{
    uint64_t load;
    uint32_t block;
} og_bin_slot;

static int og_slot_less(og_bin_slot a, og_bin_slot b)
{
    return a.load != b.load ? a.load < b.load : a.block < b.block;
}

static int og_bin_deal(const og_bin_desc *bins, uint32_t n, uint32_t slots, uint32_t *order, uint32_t *blk)
{
    og_bin_slot *heap = (og_bin_slot *)malloc((size_t)slots * sizeof(og_bin_slot));
    uint32_t *to = (uint32_t *)malloc((size_t)n * 4 + 4);
    if (!heap || !to)
    {
        free(heap); free(to);
        og_set_error("out of host memory");
        return -1;
    }
    for (uint32_t i = 0; i < slots; i++) { heap[i].load = 0; heap[i].block = i; }
    memset(blk, 0, ((size_t)slots + 1) * 4);
    for (uint32_t q = 0; q < n;)
    {
        uint32_t e = q;
        uint64_t cost = 0;
        do
            cost += bins[e].cnt + 2048u;   /* a bin's entries and its fixed part (barriers, latencies) */
        while (bins[e].kind == OG_BIN_PIECE && !(bins[e++].row1 & OG_BIN_LAST) && e < n);
        if (bins[q].kind != OG_BIN_PIECE) e = q + 1;
        for (; q < e; q++) to[q] = heap[0].block, blk[heap[0].block + 1]++;
        heap[0].load += cost;
        for (uint32_t i = 0;;)   /* sift the root down */
        {
            uint32_t c = 2 * i + 1;
            if (c >= slots) break;
            if (c + 1 < slots && og_slot_less(heap[c + 1], heap[c])) c++;
            if (!og_slot_less(heap[c], heap[i])) break;
            const og_bin_slot t = heap[i];
            heap[i] = heap[c];
            heap[c] = t;
            i = c;
        }
    }
    for (uint32_t i = 0; i < slots; i++) blk[i + 1] += blk[i];
    for (uint32_t q = n; q-- > 0;) order[--blk[to[q] + 1]] = q;   /* blk[i + 1] falls back to block i's first */
    for (uint32_t i = 0; i < slots; i++) blk[i] = blk[i + 1];
    blk[slots] = n;
    free(heap); free(to);
    return 0;
}

/* Sources per gather work item: one round of items over the blocks (one per
 * CU), or as many equal rounds as OG_BIN_ITEM_SRC allows; a segment's
 * sources are cut evenly.  (Runs of a fixed 131,072 sources left half of the
 * CUs idle at 2^24 edges.) */
static uint32_t og_bin_item_src(const uint32_t *seg_quads, uint32_t n_seg, uint32_t cus)
{
    const uint64_t total = (uint64_t)seg_quads[n_seg] * OG_BIN_TILE_ALIGN;
    const uint64_t rounds = (total + (uint64_t)cus * OG_BIN_ITEM_SRC - 1) / ((uint64_t)cus * OG_BIN_ITEM_SRC);
    const uint64_t most = rounds * cus;
    uint64_t size = (total + most - 1) / (most ? most : 1);
    if (size < 8192) size = 8192;
    for (int tries = 0; tries < 64; tries++)
    {
        uint64_t items = 0;
        for (uint32_t q = 0; q < n_seg; q++)
            items += ((uint64_t)(seg_quads[q + 1] - seg_quads[q]) * OG_BIN_TILE_ALIGN + size - 1) / size;
        if (items <= most) break;
        size += size / 32;
        if (size > OG_BIN_ITEM_SRC) return OG_BIN_ITEM_SRC;
    }
    return (uint32_t)size;
}

int og_bin_plan_build(const og_plan *pl, int mode, uint32_t max_row, uint64_t max_entries, og_bin_plan **out)
{
    *out = NULL;
    const uint32_t N = pl->N, E = pl->E, Z = pl->Z, H = pl->H;
    if (pl->relabel == 1 && H)
    {
        og_set_error("binned pull: the plan sorts long rows by source (relabel 1); it needs CSR order");
        return -1;
    }
    if (!E || !N)
    {
        og_set_error("binned pull: graph without edges");
        return -1;
    }
    og_bin_plan *b = (og_bin_plan *)calloc(1, sizeof(og_bin_plan));
    og_vec runs = {NULL, 0, 0, sizeof(og_bin_run)}, bins = {NULL, 0, 0, sizeof(og_bin_desc)};
    og_vec items = {NULL, 0, 0, sizeof(og_bin_item)};
    uint32_t *order = NULL, *blk = NULL, *d_order = NULL, *seg_src = NULL, *rp = NULL;
    uint32_t *d_quads = NULL, *d_bin_quads = NULL, *d_seg = NULL;
    void *scratch = NULL;
    hipStream_t s = og_stream();
    int rc = -1, unfit = 0;
    if (!b)
    {
        og_set_error("out of host memory");
        goto done;
    }
    if (og_bin_list_runs(pl, &runs)) goto done;
    if (og_bin_longest((const og_bin_run *)runs.p, runs.n) > max_row)
    {
        unfit = 1;
        rc = 0;
        goto done;
    }
    {
        const uint32_t n_seg = (N + OG_BIN_SEG - 1) / OG_BIN_SEG;
        const uint32_t cus = og_num_cus() > 0 ? (uint32_t)og_num_cus() : 1;
        const uint32_t cap = og_bin_cap(E, n_seg, 2 * cus);
        if (og_bin_pack(pl, &runs, cap, mode == OG_MODE_F32 ? og_bin_wave_row(cap) : OG_BIN_CAP, &bins))
        {
            og_set_error("out of host memory");
            goto done;
        }
        const uint32_t n_edge_bins = (uint32_t)bins.n;
        for (uint32_t q = 0; q < n_edge_bins && ((og_bin_desc *)bins.p)[q].kind == OG_BIN_PIECE; q++) b->d.first_bin++;
        /* two sum blocks per CU, no more than there are bins */
        b->sum_grid = n_edge_bins < 2 * cus ? n_edge_bins : 2 * cus;
        order = (uint32_t *)malloc((size_t)n_edge_bins * 4 + 4);
        blk = (uint32_t *)malloc(((size_t)b->sum_grid + 1) * 4);
        if (!order || !blk) { og_set_error("out of host memory"); goto done; }
        if (og_bin_deal((const og_bin_desc *)bins.p, n_edge_bins, b->sum_grid, order, blk)) goto done;
        /* rows without in-edges: epilogue-only bins, last */
        for (uint32_t r0 = Z; r0 < N; r0 += OG_BIN_ZERO_ROWS)
        {
            og_bin_desc *d = (og_bin_desc *)og_vec_push(&bins);
            if (!d) { og_set_error("out of host memory"); goto done; }
            memset(d, 0, sizeof(*d));
            d->row0 = r0;
            d->row1 = N - r0 < OG_BIN_ZERO_ROWS ? N : r0 + OG_BIN_ZERO_ROWS;
            d->pos0 = E;
            d->kind = OG_BIN_THREAD_ROWS;
        }
        b->n_zero_bins = (uint32_t)bins.n - n_edge_bins;
        if ((uint64_t)n_edge_bins * n_seg > 0xFFFF0000ull)
        {
            og_set_error("binned pull: graph too large for 32-bit tile keys");
            goto done;
        }
        b->d.N = N;
        b->d.n_seg = n_seg;
        b->d.n_bins = (uint32_t)bins.n;
        b->d.n_bins_live = (uint32_t)bins.n;
        b->d.n_edge_bins = n_edge_bins;

        /* ---- device: the tiles' sizes in quads (16 entries), segment by
         * segment; prefix sums give each tile's place among the sources and
         * each bin's among the entries ---- */
        const uint32_t n_cells = n_edge_bins * n_seg;
        b->mem_bins = og_bin_upload(bins.p, bins.n * sizeof(og_bin_desc));
        d_quads = og_dalloc(((size_t)n_cells + 1) * 4);
        d_bin_quads = og_dalloc(((size_t)n_edge_bins + 1) * 4);
        d_seg = og_dalloc(((size_t)n_seg + 1) * 4);
        const size_t sc = og_scan_scratch_bytes(n_cells), sb = og_scan_scratch_bytes(n_edge_bins);
        scratch = og_dalloc(sc > sb ? sc : sb);
        seg_src = (uint32_t *)malloc(((size_t)n_seg + 1) * 4);
        if (!seg_src) { og_set_error("out of host memory"); goto done; }
        if (!b->mem_bins || !d_quads || !d_bin_quads || !d_seg || !scratch) goto done;
        og_bin_desc *d_bins = (og_bin_desc *)b->mem_bins;
        if (og_launch_bin_count(d_bins, n_edge_bins, pl->cols, n_seg, d_quads, d_bin_quads, s) ||
            og_scan_exclusive(d_quads, d_quads, n_cells, scratch, s) ||
            og_scan_exclusive(d_bin_quads, d_bin_quads, n_edge_bins, scratch, s) ||
            og_launch_bin_place(d_bins, n_edge_bins, b->d.n_bins, d_bin_quads, d_quads, n_seg, d_seg, s) ||
            og_hip_check(og_copy(seg_src, d_seg, ((size_t)n_seg + 1) * 4, hipMemcpyDeviceToHost), "D2H segments"))
            goto done;
        const uint64_t ent = (uint64_t)seg_src[n_seg] * OG_BIN_TILE_ALIGN;
        if (ent + OG_BIN_SPARE > 0xFFFFFFFFull)
        {
            og_set_error("binned pull: graph too large for 32-bit entries");
            goto done;
        }
        if (ent > max_entries)
        {
            unfit = 1;
            rc = 0;
            goto done;
        }
        b->n_ent = ent + OG_BIN_SPARE;   /* spare entries past the last tile */
        b->d.n_ent = (uint32_t)ent;
        b->mem_src = og_dalloc(b->n_ent * 2);
        b->mem_pos = og_dalloc(b->n_ent * 2);
        b->mem_val = og_dalloc(b->n_ent * 4);
        b->mem_qent = og_dalloc(ent / OG_BIN_TILE_ALIGN * 4);
        b->mem_sched = og_dalloc((size_t)n_edge_bins * sizeof(og_bin_desc));
        b->mem_blk = og_bin_upload(blk, ((size_t)b->sum_grid + 1) * 4);
        d_order = (uint32_t *)og_bin_upload(order, (size_t)n_edge_bins * 4);
        if (!b->mem_src || !b->mem_pos || !b->mem_val || !b->mem_qent || !b->mem_sched || !b->mem_blk || !d_order)
            goto done;
        if (og_launch_bin_sched(d_bins, d_order, n_edge_bins, (og_bin_desc *)b->mem_sched, s) ||
            og_launch_bin_fill(d_bins, n_edge_bins, pl->cols, n_seg, d_quads, (uint16_t *)b->mem_src,
                               (uint16_t *)b->mem_pos, (uint32_t *)b->mem_qent, s) ||
            og_launch_fill_u32((uint32_t *)((uint16_t *)b->mem_src + ent), 0, OG_BIN_SPARE / 2, s))
            goto done;

        /* ---- host: the work items ---- */
        const uint32_t item_src = og_bin_item_src(seg_src, n_seg, cus);
        for (uint32_t q = 0; q < n_seg; q++)
        {
            const uint64_t quads = seg_src[q + 1] - seg_src[q];
            const uint64_t parts = (quads * OG_BIN_TILE_ALIGN + item_src - 1) / item_src;
            for (uint64_t k = 0; k < parts; k++)
            {
                og_bin_item *it = (og_bin_item *)og_vec_push(&items);
                if (!it) { og_set_error("out of host memory"); goto done; }
                it->seg = q;
                it->f0 = (uint32_t)((seg_src[q] + quads * k / parts) * OG_BIN_TILE_ALIGN);
                it->f1 = (uint32_t)((seg_src[q] + quads * (k + 1) / parts) * OG_BIN_TILE_ALIGN);
                it->pad = 0;
            }
        }
        b->mem_items = og_bin_upload(items.p, items.n * sizeof(og_bin_item));
        if (!b->mem_items) goto done;
        b->d.n_items = (uint32_t)items.n;
        b->d.items = (const og_bin_item *)b->mem_items;
        b->d.qent = (const uint32_t *)b->mem_qent;
        b->d.src = (const uint16_t *)b->mem_src;
        b->d.pos = (const uint16_t *)b->mem_pos;
        b->d.val = (float *)b->mem_val;
        b->d.bins = d_bins;
        b->d.sched = (const og_bin_desc *)b->mem_sched;
        b->d.blk = (const uint32_t *)b->mem_blk;
        if (getenv("OG_BIN_VERIFY"))
        {
            rp = (uint32_t *)malloc(((size_t)N + 1) * 4);
            if (!rp) { og_set_error("out of host memory"); goto done; }
            if (og_hip_check(og_copy(rp, pl->row_ptr, ((size_t)N + 1) * 4, hipMemcpyDeviceToHost), "D2H row_ptr") ||
                og_bin_verify(b, pl, rp))
                goto done;
        }
    }
    rc = 0;
done:
    if (hipStreamSynchronize(s) != hipSuccess && !rc)
    {
        og_set_error("binned pull: the layout's kernels failed");
        rc = -1;
    }
    og_dfree(d_quads); og_dfree(d_bin_quads); og_dfree(d_seg); og_dfree(scratch);
    og_dfree(d_order);
    free(runs.p); free(bins.p); free(items.p); free(order); free(blk); free(seg_src); free(rp);
    if (rc || unfit) og_bin_plan_destroy(b);
    else *out = b;
    return rc;
}
