/*
 * og_pr_run.h -- the state of one PageRank run on the GPU (ogpu_pr), shared
 * by its host orchestration (og_pagerank.c) and the SpMV entry points
 * (og_spmv.c), which drive the same pull and push kernels.
 */
#ifndef OG_PR_RUN_H
#define OG_PR_RUN_H

#include "og_internal.h"
#include "og_pr.h"
#include "opengraph_amd_ext.h"

#ifdef __cplusplus
extern "C" {
#endif

struct ogpu_pr
{
    og_graph *g;
    og_plan *plan;
    int own_plan;
    ogpu_pr_options opt;
    int mode, push, quant, dd;
    og_pr_dev dev;
    uint32_t gv;              /* grid of the per-vertex kernels */
    uint32_t parts_cap;       /* entries of the first-level partial arrays */
    uint32_t n_final_pull, n_final_vert;
    float *r;
    void *c[2];
    void *cq;
    void *next;
    void *chunk_sum;
    float *init_d;
    float *out_old;
    double *d_sum;
    double *part_err, *fin_err;
    uint32_t *part_act, *fin_act;
    float *part_min, *part_max, *fin_min, *fin_max;
    uint32_t *ticket, *done;
    og_iter_stat *stats;
    uint32_t stats_cap;
    og_qparams *qp;
    uint32_t *done_host;
    uint32_t it;
    /* per-iteration end events of a run, kernel timing pairs of enqueue */
    hipEvent_t *iter_ev;
    uint32_t n_iter_ev;
    hipEvent_t *kev;
    uint32_t n_kev, kev_used;
    double seconds_plan;
    uint32_t rows;
    og_iter_stat *rows_host;
    /* data-driven state: two byte worklists, changed flags, residuals */
    uint8_t *wl[2];
    uint8_t *changed;
    float *resid;
    /* learned start: features (N x 4) and reduction scratch */
    float *feat;
    double *lscratch;
    /* every-row-exact fp32 pull: rows [0, C) longest first (device) */
    uint32_t *chain_rows;
    /* binned pull (og_bin.h): layout, blocks of its final reduction */
    struct og_bin_plan *bins;
    uint32_t n_final_bin;
    /* direct pull (og_dir.h): the iterations of a small graph in one
     * launch */
    struct og_dir_plan *dir;
    uint32_t dir_single;      /* runs left to go one iteration a launch */
    og_pr_report *report;     /* host memory a whole run's results land in */
    /* partitioned push (og_push_part_kernel): destination ranges (device
     * n_pp + 1 row bounds), each inverse-CSR edge's offset in its range,
     * the first range pushed, blocks of its final reduction */
    uint32_t *pp_v0;
    uint16_t *pp_dloc;
    uint32_t n_pp, pp_first, n_final_pp;
    /* the last start vector offered (ogpu_pr_set_init, the learned start)
     * was rejected and the runs start from the uniform vector */
    uint32_t init_fallback;
    /* drop-in runs print the reference's per-iteration table rows as the
     * iterations complete: rows [0, printed) are out, print_done after the
     * stopping row */
    int print_rows, print_done;
    uint32_t printed;
};

/* Create a run of opt->variant on graph g; plan may be supplied (borrowed)
 * or is built here.  Buffers are allocated, the state is not initialized. */
int og_pr_create_with(og_graph *g, og_plan *plan, const ogpu_pr_options *opt, ogpu_pr **out);
/* The same; spmv: for SpMV passes on the direct or binned passes.  Where a
 * variant other than 0 would not be on them *out stays NULL (and 0 is returned). */
int og_pr_create_as(og_graph *g, og_plan *plan, const ogpu_pr_options *opt, int spmv, ogpu_pr **out);
/* Grow an event array to `need` created events. */
int og_pr_events(hipEvent_t **arr, uint32_t *have, uint32_t need);
/* The drop-ins' device copy of a caller's GraphCSR, cached by pointer and array
 * identity, and its cached plans: og_plan_build's relabel 1 (with forward edges
 * when need_forward), and relabel 2 with the rows of more than OG_CH in-edges
 * first (longest first), as the direct and binned passes build theirs. */
struct GraphCSR;
int og_cache_graph(struct GraphCSR *graph, og_graph **g);
int og_cache_plan(int need_forward, og_plan **plan);
int og_cache_csr_plan(og_plan **plan);
/* An SpMV run on graph g over a borrowed plan (NULL: built here).  streamed 0: by
 * the code's own kernels; otherwise, unless its options or the plan ask for
 * those, on the direct or binned passes, and where -p 1 to 3 are not faster there
 * *out stays NULL and 0 is returned. */
int og_spmv_create_as(og_graph *g, og_plan *plan, const ogpu_spmv_options *opt, int streamed, ogpu_spmv **out);

#ifdef __cplusplus
}
#endif

#endif
