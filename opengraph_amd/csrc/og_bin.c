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
    og_dfree(b->mem_pos); og_dfree(b->mem_val); og_dfree(b->mem_bins); og_dfree(b->mem_long_row);
    og_dfree(b->mem_long_bin); og_dfree(b->mem_ticket);
    free(b);
}

/* Sum and long-row blocks take half a CU's LDS each: two block slots per
 * CU (a long-row block has twice the threads at half the registers).  The
 * long rows get up to one slot in eight, the sum pass the rest, side by
 * side.  Workgroups are dealt to the XCDs in turn, so the sum pass leaves a
 * whole number of slots per XCD free (the long-row blocks rounded up to a
 * multiple of OG_BIN_XCDS); otherwise a long-row block can find its XCD
 * full and wait for a sum block to end. */
#define OG_BIN_XCDS 8u

uint32_t og_bin_long_grid(const og_bin_plan *b)
{
    /* the long rows' share of the slots: their in-edges' share of E, times
     * 1.6 (an in-edge costs a long-row block about 1.6 times what it costs
     * the sum pass: R-MAT-24 measurements), in whole XCD rounds, between
     * OG_BIN_XCDS and a quarter of the CUs */
    const uint32_t cus = (uint32_t)og_num_cus();
    const uint32_t cap = cus / 4 ? cus / 4 : 1;
    uint64_t l = b->n_edges ? (uint64_t)(2.0 * cus * 1.6 * (double)b->long_terms / (double)b->n_edges) : 0;
    l = (l + OG_BIN_XCDS - 1) / OG_BIN_XCDS * OG_BIN_XCDS;
    if (l < OG_BIN_XCDS) l = OG_BIN_XCDS;
    if (l > cap) l = cap;
    return b->d.n_long < l ? b->d.n_long : (uint32_t)l;
}

uint32_t og_bin_sum_grid(const og_bin_plan *b)
{
    const uint32_t slots = 2u * (uint32_t)og_num_cus();   /* two blocks per CU */
    const uint32_t l = (og_bin_long_grid(b) + OG_BIN_XCDS - 1) / OG_BIN_XCDS * OG_BIN_XCDS;
    return slots > l ? slots - l : 1;
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
 * CSR positions, the pieces first and each long row's pieces covering its
 * in-edges in order.  Runs before any binned kernel, so a bad layout
 * is an error, not a stray access. */
static int og_bin_verify(const og_bin_plan *b, const og_plan *pl, const uint32_t *rp)
{
    const og_bin_dev *d = &b->d;
    const size_t ne = (size_t)b->n_ent, nq = (ne - OG_BIN_SPARE) / OG_BIN_TILE_ALIGN;
    og_bin_item *items = (og_bin_item *)malloc((size_t)d->n_items * sizeof(og_bin_item) + 16);
    uint32_t *qent = (uint32_t *)malloc(nq * 4 + 4);
    uint16_t *src = (uint16_t *)malloc(ne * 2), *pos = (uint16_t *)malloc(ne * 2);
    og_bin_desc *bins = (og_bin_desc *)malloc((size_t)d->n_bins * sizeof(og_bin_desc) + 16);
    uint32_t *lrow = (uint32_t *)malloc((size_t)d->n_long * 4 + 4), *lbin = (uint32_t *)malloc((size_t)d->n_long * 4 + 4);
    uint32_t *gsrc = (uint32_t *)malloc(ne * 4);   /* source id gathered into each entry */
    uint32_t *cols = (uint32_t *)malloc((size_t)pl->E * 4 + 4);
    uint8_t *seen = (uint8_t *)calloc(ne, 1);
    int rc = -1;
#define OG_BIN_FAIL(...) do { og_set_error("binned layout check: " __VA_ARGS__); goto out; } while (0)
    if (!items || !qent || !src || !pos || !bins || !lrow || !lbin || !seen || !gsrc || !cols)
        OG_BIN_FAIL("out of host memory");
    if (og_hip_check(og_copy(items, d->items, (size_t)d->n_items * sizeof(og_bin_item), hipMemcpyDeviceToHost), "D2H") ||
        og_hip_check(og_copy(qent, d->qent, nq * 4, hipMemcpyDeviceToHost), "D2H") ||
        og_hip_check(og_copy(src, d->src, ne * 2, hipMemcpyDeviceToHost), "D2H") ||
        og_hip_check(og_copy(pos, d->pos, ne * 2, hipMemcpyDeviceToHost), "D2H") ||
        og_hip_check(og_copy(bins, d->bins, (size_t)d->n_bins * sizeof(og_bin_desc), hipMemcpyDeviceToHost), "D2H") ||
        og_hip_check(og_copy(lrow, d->long_row, (size_t)d->n_long * 4, hipMemcpyDeviceToHost), "D2H") ||
        og_hip_check(og_copy(lbin, d->long_bin, (size_t)d->n_long * 4, hipMemcpyDeviceToHost), "D2H") ||
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
    uint64_t pieces = 0;
    for (uint32_t q = 0; q < d->n_long; q++)
    {
        const uint32_t r = lrow[q];
        if (r >= pl->Z) OG_BIN_FAIL("long row %u", q);
        const uint32_t n = rp[r + 1] - rp[r];
        for (uint32_t c0 = 0, k = lbin[q]; c0 < n; c0 += OG_BIN_CAP, k++, pieces++)
            if (k >= d->first_bin || bins[k].kind != OG_BIN_PIECE || bins[k].row0 != r || bins[k].pos0 != rp[r] + c0 ||
                bins[k].cnt != (n - c0 < OG_BIN_CAP ? n - c0 : OG_BIN_CAP))
                OG_BIN_FAIL("long row %u: piece %u", q, k);
    }
    if (pieces != d->first_bin) OG_BIN_FAIL("%llu pieces for %u piece bins", (unsigned long long)pieces, d->first_bin);
    rc = 0;
#undef OG_BIN_FAIL
out:
    free(items); free(qent); free(src); free(pos); free(bins); free(lrow); free(lbin); free(seen);
    free(gsrc); free(cols);
    return rc;
}

/* Runs of equal in-degree of the rows [0, Z): (first row, in-degree),
 * ascending by row; what the packing of rows into bins needs of the row
 * offsets.  A relabelled plan orders its rows by in-degree, so there are at
 * most about sqrt(2 E) runs and the device lists them; a plan in original
 * order (relabel 0) has its row offsets read back instead. */
typedef struct
{
    uint32_t row, deg;
} og_bin_run;

static int og_bin_run_cmp(const void *a, const void *b)
{
    const uint32_t x = ((const og_bin_run *)a)->row, y = ((const og_bin_run *)b)->row;
    return x < y ? -1 : x > y;
}

static int og_bin_runs(const og_plan *pl, og_vec *runs)
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

/* Long rows (more than OG_BIN_CAP in-edges) and bins: first the pieces of
 * the long rows (OG_BIN_CAP in-edges each, in CSR order), then consecutive
 * rows of one kind (thread rows, wavefront rows of more than OG_BIN_WAVE_ROW
 * in-edges) with at most OG_BIN_CAP in-edges and OG_BIN_RPT * OG_BIN_THREADS
 * rows together. */
typedef struct
{
    uint32_t row, deg, bin;
} og_bin_long;

static int og_bin_long_cmp(const void *a, const void *b)
{
    const og_bin_long *x = (const og_bin_long *)a, *y = (const og_bin_long *)b;
    if (x->deg != y->deg) return x->deg > y->deg ? -1 : 1;
    return x->row < y->row ? -1 : x->row > y->row;
}

static int og_bin_pack(const og_plan *pl, const og_vec *runs, og_vec *bins, og_vec *longs)
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
        {
            og_bin_long *l = (og_bin_long *)og_vec_push(longs);
            if (!l) return -1;
            l->row = r;
            l->deg = deg;
            l->bin = (uint32_t)bins->n;
            for (uint32_t p0 = 0; p0 < deg; p0 += OG_BIN_CAP)
            {
                og_bin_desc *d = (og_bin_desc *)og_vec_push(bins);
                if (!d) return -1;
                memset(d, 0, sizeof(*d));
                d->row0 = r;
                d->row1 = (uint32_t)longs->n - 1;
                d->pos0 = pos + p0;
                d->kind = OG_BIN_PIECE;
                d->cnt = deg - p0 < OG_BIN_CAP ? deg - p0 : OG_BIN_CAP;
            }
        }
    }
    og_bin_desc *d = NULL;   /* the open bin (the last one) */
    pos = 0;
    for (size_t i = 0; i < runs->n; i++)
    {
        const uint32_t r1 = i + 1 < runs->n ? run[i + 1].row : Z, deg = run[i].deg;
        const uint32_t kind = deg > OG_BIN_WAVE_ROW ? OG_BIN_WAVE_ROWS : OG_BIN_THREAD_ROWS;
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
                room = (OG_BIN_CAP - d->cnt) / deg;
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

int og_bin_plan_build(const og_plan *pl, og_bin_plan **out)
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
    og_vec longs = {NULL, 0, 0, sizeof(og_bin_long)}, items = {NULL, 0, 0, sizeof(og_bin_item)};
    uint32_t *ids = NULL, *seg_src = NULL, *rp = NULL;
    uint32_t *d_quads = NULL, *d_bin_quads = NULL, *d_seg = NULL;
    void *scratch = NULL;
    hipStream_t s = og_stream();
    int rc = -1;
    if (!b)
    {
        og_set_error("out of host memory");
        goto done;
    }
    if (og_bin_runs(pl, &runs)) goto done;
    if (og_bin_pack(pl, &runs, &bins, &longs))
    {
        og_set_error("out of host memory");
        goto done;
    }
    {
        const uint32_t n_long = (uint32_t)longs.n, n_edge_bins = (uint32_t)bins.n;
        b->n_edges = E;
        b->d.first_bin = 0;
        for (uint32_t q = 0; q < n_edge_bins && ((og_bin_desc *)bins.p)[q].kind == OG_BIN_PIECE; q++) b->d.first_bin++;
        /* the long rows, longest first, and each one's first piece */
        if (n_long) qsort(longs.p, n_long, sizeof(og_bin_long), og_bin_long_cmp);
        ids = (uint32_t *)malloc((size_t)(n_long + 1) * 8);
        if (!ids) { og_set_error("out of host memory"); goto done; }
        for (uint32_t i = 0; i < n_long; i++)
        {
            const og_bin_long *l = (const og_bin_long *)longs.p + i;
            ids[i] = l->row;
            ids[n_long + i] = l->bin;
            b->long_terms += l->deg;
        }
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
        const uint32_t n_seg = (N + OG_BIN_SEG - 1) / OG_BIN_SEG;
        if ((uint64_t)n_edge_bins * n_seg > 0xFFFF0000ull)
        {
            og_set_error("binned pull: graph too large for 32-bit tile keys");
            goto done;
        }
        b->d.N = N;
        b->d.n_seg = n_seg;
        b->d.n_bins = (uint32_t)bins.n;
        b->d.n_bins_live = (uint32_t)bins.n;
        b->d.n_long = n_long;

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
        b->n_ent = ent + OG_BIN_SPARE;   /* spare entries past the last tile */
        b->d.n_ent = (uint32_t)ent;
        b->mem_src = og_dalloc(b->n_ent * 2);
        b->mem_pos = og_dalloc(b->n_ent * 2);
        b->mem_val = og_dalloc(b->n_ent * 4);
        b->mem_qent = og_dalloc(ent / OG_BIN_TILE_ALIGN * 4);
        b->mem_long_row = og_bin_upload(ids, (size_t)n_long * 4);
        b->mem_long_bin = og_bin_upload(ids + n_long, (size_t)n_long * 4);
        b->mem_ticket = og_dalloc(256);
        if (!b->mem_src || !b->mem_pos || !b->mem_val || !b->mem_qent || !b->mem_long_row || !b->mem_long_bin ||
            !b->mem_ticket)
            goto done;
        if (og_launch_bin_fill(d_bins, n_edge_bins, pl->cols, n_seg, d_quads, (uint16_t *)b->mem_src,
                               (uint16_t *)b->mem_pos, (uint32_t *)b->mem_qent, s) ||
            og_launch_fill_u32((uint32_t *)((uint16_t *)b->mem_src + ent), 0, OG_BIN_SPARE / 2, s))
            goto done;

        /* ---- host: the work items: each segment's sources in runs of at
         * most OG_BIN_ITEM_SRC ---- */
        for (uint32_t q = 0; q < n_seg; q++)
        {
            const uint64_t end = (uint64_t)seg_src[q + 1] * OG_BIN_TILE_ALIGN;
            for (uint64_t f0 = (uint64_t)seg_src[q] * OG_BIN_TILE_ALIGN; f0 < end; f0 += OG_BIN_ITEM_SRC)
            {
                og_bin_item *it = (og_bin_item *)og_vec_push(&items);
                if (!it) { og_set_error("out of host memory"); goto done; }
                it->seg = q;
                it->f0 = (uint32_t)f0;
                it->f1 = (uint32_t)(end - f0 < OG_BIN_ITEM_SRC ? end : f0 + OG_BIN_ITEM_SRC);
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
        b->d.long_row = (const uint32_t *)b->mem_long_row;
        b->d.long_bin = (const uint32_t *)b->mem_long_bin;
        b->d.ticket = (uint32_t *)b->mem_ticket;
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
    free(runs.p); free(bins.p); free(longs.p); free(items.p); free(ids); free(seg_src); free(rp);
    if (rc) og_bin_plan_destroy(b);
    else *out = b;
    return rc;
}
