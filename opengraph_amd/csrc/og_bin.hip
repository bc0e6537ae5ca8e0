/*
 * og_bin.hip -- gfx950 kernels of the binned pull (layout and passes
 * described in og_bin.h) and of its one-time layout build.
 *
 * Row sums and their exactness: og_rowsum.h.
 */
#include <hip/hip_runtime.h>

#include "og_bin.h"
#include "og_internal.h"
#include "og_pr.h"
#include "og_rowsum.h"

#define BT OG_BIN_THREADS
#define BW (OG_BIN_THREADS / 64)
#define GT OG_BIN_GTHREADS       /* the gather pass's blocks */
#define GW (OG_BIN_GTHREADS / 64)
#define GATHER_Q 8u   /* runs of 4 consecutive sources per lane in flight in the gather */

/* ------------------------------------------------------------------ */
/* gather pass                                                         */
/* ------------------------------------------------------------------ */

typedef uint32_t og_u32x2 __attribute__((ext_vector_type(2)));
typedef float og_f32x4g __attribute__((ext_vector_type(4)));

/* The sources (4 u16 in one 8-byte load) and quad entry of this lane's
 * GATHER_Q runs of 4 sources from f (256 apart; f a multiple of 4, so a run
 * lies in one quad), branch-free (indices clamped to the item's last run)
 * so that all the loads issue before any is waited for. */
__device__ __forceinline__ void og_bin_gather_batch(const og_bin_dev &b, uint32_t f, uint32_t f1,
                                                    og_u32x2 (&sv)[GATHER_Q], uint32_t (&qv)[GATHER_Q])
{
#pragma unroll
    for (uint32_t u = 0; u < GATHER_Q; u++)
    {
        const uint32_t fu = min(f + 256u * u, f1 - 4);
        sv[u] = __builtin_nontemporal_load((const og_u32x2 *)(b.src + fu));
        qv[u] = __builtin_nontemporal_load(&b.qent[fu / OG_BIN_TILE_ALIGN]);
    }
}

__global__ __launch_bounds__(GT) void og_bin_gather_kernel(og_bin_dev b, const float *__restrict__ c,
                                                           const uint32_t *done)
{
    __shared__ __align__(16) float seg[OG_BIN_SEG];
    if (*done) return;
    const uint32_t lane = threadIdx.x & 63;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    for (uint32_t q = blockIdx.x; q < b.n_items; q += gridDim.x)
    {
        const og_bin_item it = b.items[q];
        const uint32_t v0 = it.seg * OG_BIN_SEG;
        const uint32_t nv = min(OG_BIN_SEG, b.N - v0);
        __syncthreads();   /* the previous item's reads of seg are done */
        {
            const float4 *c4 = (const float4 *)(c + v0);
            float4 *s4 = (float4 *)seg;
            for (uint32_t i = threadIdx.x; i < nv / 4; i += GT) s4[i] = c4[i];
            for (uint32_t i = (nv & ~3u) + threadIdx.x; i < nv; i += GT) seg[i] = c[v0 + i];
        }
        __syncthreads();
        /* wavefront w takes the runs of 4 sources f = f0 + 256 * (w * Q +
         * k * GW * Q + u) + 4 * lane (f0 and f1 are multiples of 16, so a
         * run lies in one quad and is wholly inside or past the item); each
         * run's 4 values go to 4 consecutive entries, one 16-byte store
         * (a quad's entry is a multiple of 16).  Software pipelined: the
         * next batch's loads are issued before this batch's stores (loads
         * complete in order, and a wait for this batch's loads must not
         * also wait for stores issued after them) */
        uint32_t f = it.f0 + 256u * GATHER_Q * wave + 4u * lane;
        og_u32x2 sv[GATHER_Q];
        uint32_t qv[GATHER_Q];
        og_bin_gather_batch(b, f, it.f1, sv, qv);
        for (; f < it.f1; f += 256u * GATHER_Q * GW)
        {
            og_u32x2 sv2[GATHER_Q];
            uint32_t qv2[GATHER_Q];
            og_bin_gather_batch(b, f + 256u * GATHER_Q * GW, it.f1, sv2, qv2);
            og_f32x4g x[GATHER_Q];   /* every lane's sources are valid ones (clamped) */
#pragma unroll
            for (uint32_t u = 0; u < GATHER_Q; u++)
            {
                x[u].x = seg[sv[u].x & 0xFFFFu];
                x[u].y = seg[sv[u].x >> 16];
                x[u].z = seg[sv[u].y & 0xFFFFu];
                x[u].w = seg[sv[u].y >> 16];
            }
            /* lanes past the item's end write the OG_BIN_SPARE spare
             * entries past the last tile instead: unconditional stores keep
             * the count of memory operations in flight static */
#pragma unroll
            for (uint32_t u = 0; u < GATHER_Q; u++)
            {
                const uint32_t fu = f + 256u * u;
                const uint32_t e = fu < it.f1 ? qv[u] + fu % OG_BIN_TILE_ALIGN : b.n_ent + 4u * lane;
                __builtin_nontemporal_store(x[u], (og_f32x4g *)(b.val + e));
            }
#pragma unroll
            for (uint32_t u = 0; u < GATHER_Q; u++)
            {
                sv[u] = sv2[u];
                qv[u] = qv2[u];
            }
        }
    }
}

/* ------------------------------------------------------------------ */
/* sum pass                                                            */
/* ------------------------------------------------------------------ */

/* What a bin's rows need besides their values -- slot range (row
 * offsets), old rank, out-degree -- of the row a thread holds.  fp32 thread
 * rows: thread t row t; wavefront rows: lane l of wavefront w the wavefront's
 * l-th (row w + BW * l); integer modes: thread t row t / G, G lanes per row.
 * Loaded with the bin's entries, one bin ahead, so adding a bin's rows issues
 * no global load (a load there would wait for the next bin's entries too:
 * loads complete in order). */
struct og_bin_meta
{
    uint32_t p0, p1, deg;
    float prev;
};

/* integer modes: log2 of the lanes per row, all the block's threads on the
 * bin's rows, at most a wavefront each */
__device__ __forceinline__ uint32_t og_bin_group(const og_bin_desc &d)
{
    const uint32_t n = d.row1 - d.row0;   /* <= BT */
    return min(6u, n <= 1 ? 6u : (uint32_t)__builtin_clz(n - 1) - (uint32_t)__builtin_clz(BT - 1));
}

template <int MODE>
__device__ __forceinline__ void og_bin_meta_load(const og_pr_dev &a, const og_bin_desc &d, og_bin_meta &m)
{
    if (d.kind == OG_BIN_PIECE)
    {
        m.prev = __builtin_nontemporal_load(&a.r[d.row0]);
        m.deg = __builtin_nontemporal_load(&a.outdeg[d.row0]);
        return;
    }
    const uint32_t t = MODE != OG_MODE_F32             ? threadIdx.x >> og_bin_group(d)
                       : d.kind == OG_BIN_WAVE_ROWS ? (threadIdx.x >> 6) + BW * (threadIdx.x & 63)
                                                     : threadIdx.x;
    const uint32_t v = d.row0 + t;
    if (v < d.row1)
    {
        m.p0 = a.row_ptr[v];
        m.p1 = a.row_ptr[v + 1];
        m.prev = __builtin_nontemporal_load(&a.r[v]);
        m.deg = __builtin_nontemporal_load(&a.outdeg[v]);
    }
}

/* A bin's entries, 8 per thread and sweep: OG_BIN_SWEEPS sweeps cover a
 * full bin; loaded into registers ahead of time (the next bin's while this
 * one's rows are added). */
#define OG_BIN_SWEEPS ((OG_BIN_CAP + 8 * BT - 1) / (8 * BT))

typedef uint32_t og_u32x4 __attribute__((ext_vector_type(4)));
typedef float og_f32x4 __attribute__((ext_vector_type(4)));

struct og_bin_regs
{
    og_u32x4 p[OG_BIN_SWEEPS];
    og_f32x4 x0[OG_BIN_SWEEPS], x1[OG_BIN_SWEEPS];
};

__device__ __forceinline__ void og_bin_load(const og_bin_dev &b, const og_bin_desc &d, og_bin_regs &r)
{
#pragma unroll
    for (uint32_t k = 0; k < OG_BIN_SWEEPS; k++)
    {
        const uint32_t e = d.ent0 + 8 * (threadIdx.x + k * BT);
        if (e < d.ent1)
        {
            r.p[k] = __builtin_nontemporal_load((const og_u32x4 *)(b.pos + e));
            r.x0[k] = __builtin_nontemporal_load((const og_f32x4 *)(b.val + e));
            r.x1[k] = __builtin_nontemporal_load((const og_f32x4 *)(b.val + e + 4));
        }
    }
}

/* 8 entries' values to their slots (padding entries skipped) */
__device__ __forceinline__ void og_bin_scatter8(float *slot, og_u32x4 p, og_f32x4 x0, og_f32x4 x1)
{
    const uint32_t pp[8] = {p.x & 0xFFFFu, p.x >> 16, p.y & 0xFFFFu, p.y >> 16,
                            p.z & 0xFFFFu, p.z >> 16, p.w & 0xFFFFu, p.w >> 16};
    const float xx[8] = {x0.x, x0.y, x0.z, x0.w, x1.x, x1.y, x1.z, x1.w};
#pragma unroll
    for (uint32_t t = 0; t < 8; t++)
        if (pp[t] != OG_BIN_PAD) slot[pp[t]] = xx[t];
}

/* The bin's entries: the registers' sweeps, then (a bin whose tiles'
 * padding takes it past OG_BIN_SWEEPS sweeps: up to 15 entries per tile)
 * the rest straight from memory. */
__device__ __forceinline__ void og_bin_put(const og_bin_dev &b, float *slot, const og_bin_desc &d,
                                           const og_bin_regs &r)
{
#pragma unroll
    for (uint32_t k = 0; k < OG_BIN_SWEEPS; k++)
    {
        const uint32_t e = d.ent0 + 8 * (threadIdx.x + k * BT);
        if (e < d.ent1) og_bin_scatter8(slot, r.p[k], r.x0[k], r.x1[k]);
    }
    for (uint32_t e = d.ent0 + 8 * (threadIdx.x + OG_BIN_SWEEPS * BT); e < d.ent1; e += 8 * BT)
        og_bin_scatter8(slot, __builtin_nontemporal_load((const og_u32x4 *)(b.pos + e)),
                        __builtin_nontemporal_load((const og_f32x4 *)(b.val + e)),
                        __builtin_nontemporal_load((const og_f32x4 *)(b.val + e + 4)));
}

/* Block i takes the bins sched[blk[i], blk[i + 1]) in that order (a long
 * row's pieces one after the other); integer modes put all the block's
 * threads on a bin's rows, a power of two each (a thread per row, the fp32
 * split, left most of them idle: 400 us at R-MAT-22, now 128); then, while rows
 * without in-edges still change, every gridDim.x-th of their bins.  Bound by the
 * streamed entries (6 bytes each), at smaller sizes by the wavefront rows; two
 * blocks a CU, so that one's rows overlap the other's entries.  R-MAT-24: 449 us
 * = 4.7 TB/s by the HBM counters, as the gather pass (567 us beside a long-row
 * kernel on CUs of its own before); R-MAT-22: 117 us, where that kernel's longest row
 * took 158; R-MAT-16, whose wavefront rows bound it: 17 us against 33. */
template <int MODE>
__global__ __launch_bounds__(BT, 4) void og_bin_sum_kernel(og_bin_dev b, og_pr_dev a)
{
    typedef typename og_mode<MODE>::acc A;
    __shared__ __align__(16) float slot[OG_BIN_CAP];
    if (*a.done) return;
    og_bin_stat st;
    og_bin_stat_init(st);
    const uint32_t lane = threadIdx.x & 63;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    uint32_t q = b.blk[blockIdx.x];
    const uint32_t qe = b.blk[blockIdx.x + 1];
    og_bin_desc d;
    og_bin_regs regs;
    og_bin_meta meta;
    A carry = 0;          /* a long row's sum between its pieces: wavefront 0's running one, or a thread's share */
    static_assert(OG_BIN_RPT == 1 && OG_BIN_THREADS == 512, "a thread holds one row; og_bin_group");
    if (q < qe)
    {
        d = b.sched[q];
        og_bin_load(b, d, regs);
        og_bin_meta_load<MODE>(a, d, meta);
    }
    for (; q < qe; q++)
    {
        __syncthreads();   /* the previous bin's reads of slot are done */
        /* this bin's values to their CSR slots */
        og_bin_put(b, slot, d, regs);
        const og_bin_desc cd = d;
        const og_bin_meta cm = meta;
        /* the next bin's entries and row metadata load while this one's
         * rows are added */
        if (q + 1 < qe)
        {
            d = b.sched[q + 1];
            og_bin_load(b, d, regs);
            og_bin_meta_load<MODE>(a, d, meta);
        }
        __syncthreads();
        if constexpr (MODE != OG_MODE_F32)
        {
            if (cd.kind != OG_BIN_PIECE)
            {
                const uint32_t lg = og_bin_group(cd), G = 1u << lg;
                const uint32_t v = cd.row0 + (threadIdx.x >> lg);
                if (v < cd.row1)
                {
                    const uint32_t j0 = cm.p0 - cd.pos0, j1 = cm.p1 - cd.pos0, g = threadIdx.x & (G - 1);
                    A s = G == 1 ? og_bin_int_row_sum<MODE>(slot, j0, j1)
                                 : og_bin_int_strided<MODE>(slot, j0 + g, j1, G);
                    for (uint32_t o = 1; o < G; o <<= 1) s += __shfl_xor(s, o, 64);
                    if (g == 0) og_bin_epilogue_pf<MODE>(a, v, s, cm.prev, cm.deg, st);
                }
            }
            else
            {
                /* every thread its share of the row's pieces, added up at the last */
                if (cd.row1 & OG_BIN_FIRST) carry = 0;
                carry += og_bin_int_strided<MODE>(slot, threadIdx.x, cd.cnt, BT);
                if (cd.row1 & OG_BIN_LAST)
                {
                    A s = carry;
                    for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o, 64);
                    __syncthreads();   /* slot is read */
                    if (lane == 0) ((uint64_t *)slot)[wave] = s;
                    __syncthreads();
                    if (threadIdx.x == 0)
                    {
                        s = 0;
                        for (uint32_t w = 0; w < BW; w++) s += ((const uint64_t *)slot)[w];
                        og_bin_epilogue_pf<MODE>(a, cd.row0, s, cm.prev, cm.deg, st);
                    }
                }
            }
        }
        else if (cd.kind == OG_BIN_THREAD_ROWS)
        {
            const uint32_t v = cd.row0 + threadIdx.x;
            if (v < cd.row1)
            {
                /* (a SpMV pass continues the row's running y) */
                const float s = og_bin_row_sum(slot, cm.p0 - cd.pos0, cm.p1 - cd.pos0, a.spmv ? cm.prev : 0.0f);
                og_bin_epilogue_pf<MODE>(a, v, s, cm.prev, cm.deg, st);
            }
        }
        else
        {
            /* wavefront w's rows row0 + w, + BW, ... (a piece: wavefront 0,
             * the whole bin, going on from the row's earlier pieces) */
            const bool piece = cd.kind == OG_BIN_PIECE;
            const bool first = !piece || (cd.row1 & OG_BIN_FIRST), last = !piece || (cd.row1 & OG_BIN_LAST);
            const uint32_t row1 = piece ? cd.row0 + 1 : cd.row1;
            uint32_t l = 0;
            for (uint32_t v = cd.row0 + wave; v < row1; v += BW, l++)
            {
                const uint32_t j0 = piece ? 0 : (uint32_t)__builtin_amdgcn_readlane(cm.p0, l) - cd.pos0;
                const uint32_t j1 = piece ? cd.cnt : (uint32_t)__builtin_amdgcn_readlane(cm.p1, l) - cd.pos0;
                const float prev = og_bin_lane(cm.prev, l);
                const uint32_t deg = (uint32_t)__builtin_amdgcn_readlane(cm.deg, l);
                carry = og_bin_wave_sum(slot, j0, j1, !first ? carry : a.spmv ? prev : 0.0f,
                                        first ? OG_BIN_HEAD : 0);
                if (last && lane == 0) og_bin_epilogue_pf<MODE>(a, v, carry, prev, deg, st);
            }
        }
    }
    for (q = b.n_edge_bins + blockIdx.x; q < b.n_bins_live; q += gridDim.x)
    {
        const og_bin_desc z = b.bins[q];
#pragma unroll
        for (uint32_t k = 0; k < OG_BIN_RPT; k++)
        {
            const uint32_t v = z.row0 + threadIdx.x + BT * k;
            if (v < z.row1) og_bin_epilogue<MODE>(a, v, 0, st);
        }
    }
    og_bin_write_part(a, blockIdx.x, og_bin_block_stat<BT, MODE == OG_MODE_Q32>(st));
}

/* ------------------------------------------------------------------ */
/* launch                                                              */
/* ------------------------------------------------------------------ */

extern "C" int og_launch_bin_pull(const og_bin_dev *b, const og_pr_dev *a, int mode, uint32_t sum_grid, hipStream_t s,
                                  hipEvent_t ev0, hipEvent_t ev1)
{
    if (ev0 && og_hip_check(hipEventRecord(ev0, s), "hipEventRecord")) return -1;
    if (b->n_items)
        OG_LAUNCH(og_bin_gather_kernel, dim3(og_num_cus() > 0 ? og_num_cus() : 1), dim3(GT), 0, s, *b,
                  (const float *)a->g_in,
                  (const uint32_t *)a->done);
    switch (mode)
    {
    case OG_MODE_F32: OG_LAUNCH(og_bin_sum_kernel<OG_MODE_F32>, dim3(sum_grid), dim3(BT), 0, s, *b, *a); break;
    case OG_MODE_FX64: OG_LAUNCH(og_bin_sum_kernel<OG_MODE_FX64>, dim3(sum_grid), dim3(BT), 0, s, *b, *a); break;
    case OG_MODE_FX32: OG_LAUNCH(og_bin_sum_kernel<OG_MODE_FX32>, dim3(sum_grid), dim3(BT), 0, s, *b, *a); break;
    case OG_MODE_Q32: OG_LAUNCH(og_bin_sum_kernel<OG_MODE_Q32>, dim3(sum_grid), dim3(BT), 0, s, *b, *a); break;
    default: og_set_error("og_launch_bin_pull: bad mode %d", mode); return -1;
    }
    if (ev1 && og_hip_check(hipEventRecord(ev1, s), "hipEventRecord")) return -1;
    return og_hip_check(og_launch_status(), "og_bin_pull");
}

/* ------------------------------------------------------------------ */
/* layout build                                                        */
/* ------------------------------------------------------------------ */

/* (row, in-degree) of every row [0, Z) whose in-degree differs from the
 * row before, in any order; *n counts them (those past cap are only
 * counted). */
__global__ void og_bin_runs_kernel(const uint32_t *__restrict__ row_ptr, uint32_t Z, uint2 *__restrict__ out,
                                   uint32_t cap, uint32_t *n)
{
    for (uint32_t r = blockIdx.x * blockDim.x + threadIdx.x; r < Z; r += gridDim.x * blockDim.x)
    {
        const uint32_t p = row_ptr[r], d = row_ptr[r + 1] - p;
        if (r && p - row_ptr[r - 1] == d) continue;
        const uint32_t i = atomicAdd(n, 1u);
        if (i < cap) out[i] = make_uint2(r, d);
    }
}

/* The layout build: one block per bin.  The CSR positions of a bin are
 * consecutive, so its tiles need no sort over the edges: a histogram of the
 * bin's segments in LDS gives the tiles' sizes, and once prefix sums have
 * placed the tiles, a second sweep over the bin's columns hands every edge
 * the next free entry of its tile (an LDS counter; any order within a tile
 * will do, since an entry's slot says where its value belongs).  Bound by the
 * LDS counters of the segment with the most sources' edges; it replaced a
 * stable radix sort of E (tile, position) pairs and a host pass over the
 * tiles: R-MAT-22, 67 M edges, 0.64 ms for both kernels against 3.3 ms of
 * kernels plus 11 ms of host work and copies.  Graphs of more than BUILD_SEGS segments take their segments in
 * windows of that many. */
#define BUILD_SEGS 4096u
#define BUILD_T 256u

/* counts of the bin's columns in segments [s0, s0 + ns) */
__device__ __forceinline__ void og_bin_seg_counts(const uint32_t *__restrict__ cols, const og_bin_desc &d, uint32_t s0,
                                                  uint32_t ns, uint32_t *cnt)
{
    for (uint32_t i = threadIdx.x; i < ns; i += BUILD_T) cnt[i] = 0;
    __syncthreads();
    for (uint32_t k = threadIdx.x; k < d.cnt; k += BUILD_T)
    {
        const uint32_t sg = cols[d.pos0 + k] / OG_BIN_SEG - s0;
        if (sg < ns) atomicAdd(&cnt[sg], 1u);
    }
    __syncthreads();
}

/* quads[s * n_bins + b] = quads of tile (b, s); bin_quads[b] = their sum */
__global__ __launch_bounds__(BUILD_T) void og_bin_count_kernel(const og_bin_desc *__restrict__ bins, uint32_t n_bins,
                                                               const uint32_t *__restrict__ cols, uint32_t n_seg,
                                                               uint32_t *__restrict__ quads,
                                                               uint32_t *__restrict__ bin_quads)
{
    __shared__ uint32_t cnt[BUILD_SEGS];
    __shared__ uint32_t s_tot;
    const uint32_t b = blockIdx.x;
    const og_bin_desc d = bins[b];
    if (threadIdx.x == 0) s_tot = 0;
    uint32_t tot = 0;
    for (uint32_t s0 = 0; s0 < n_seg; s0 += BUILD_SEGS)
    {
        const uint32_t ns = min(BUILD_SEGS, n_seg - s0);
        __syncthreads();
        og_bin_seg_counts(cols, d, s0, ns, cnt);
        for (uint32_t i = threadIdx.x; i < ns; i += BUILD_T)
        {
            const uint32_t q = (cnt[i] + OG_BIN_TILE_ALIGN - 1) / OG_BIN_TILE_ALIGN;
            quads[(size_t)(s0 + i) * n_bins + b] = q;
            tot += q;
        }
    }
    for (int o = 32; o > 0; o >>= 1) tot += __shfl_xor(tot, o, 64);
    if ((threadIdx.x & 63) == 0) atomicAdd(&s_tot, tot);
    __syncthreads();
    if (threadIdx.x == 0) bin_quads[b] = s_tot;
}

/* The bins' entry ranges from the scanned bin_quads (the bins past the
 * n_bins with edges are empty, at the end), and seg_src[s] = the first quad
 * of segment s among the sources (seg_src[n_seg] = all of them). */
__global__ void og_bin_place_kernel(og_bin_desc *__restrict__ bins, uint32_t n_bins, uint32_t n_all,
                                    const uint32_t *__restrict__ bin_quads, const uint32_t *__restrict__ quads,
                                    uint32_t n_seg, uint32_t *__restrict__ seg_src)
{
    const uint32_t n = max(n_all, n_seg + 1);
    for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x)
    {
        if (i < n_all)
        {
            bins[i].ent0 = OG_BIN_TILE_ALIGN * bin_quads[min(i, n_bins)];
            bins[i].ent1 = OG_BIN_TILE_ALIGN * bin_quads[min(i + 1, n_bins)];
        }
        if (i <= n_seg) seg_src[i] = quads[(size_t)i * n_bins];
    }
}

__global__ void og_bin_sched_kernel(const og_bin_desc *__restrict__ bins, const uint32_t *__restrict__ order, uint32_t n,
                                    og_bin_desc *__restrict__ sched)
{
    for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x)
        sched[i] = bins[order[i]];
}

__global__ __launch_bounds__(BUILD_T) void og_bin_fill_kernel(const og_bin_desc *__restrict__ bins, uint32_t n_bins,
                                                              const uint32_t *__restrict__ cols, uint32_t n_seg,
                                                              const uint32_t *__restrict__ quads,
                                                              uint16_t *__restrict__ src, uint16_t *__restrict__ pos,
                                                              uint32_t *__restrict__ qent)
{
    __shared__ uint32_t cnt[BUILD_SEGS];   /* the tile's entries, then its next free one */
    __shared__ uint32_t eb[BUILD_SEGS];    /* its first entry's quad */
    __shared__ uint32_t sb[BUILD_SEGS];    /* its first source's quad */
    __shared__ uint32_t s_wave[BUILD_T / 64];
    const uint32_t b = blockIdx.x;
    const uint32_t lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const og_bin_desc d = bins[b];
    uint32_t base = d.ent0 / OG_BIN_TILE_ALIGN;   /* first quad of the window's tiles */
    for (uint32_t s0 = 0; s0 < n_seg; s0 += BUILD_SEGS)
    {
        const uint32_t ns = min(BUILD_SEGS, n_seg - s0);
        __syncthreads();
        og_bin_seg_counts(cols, d, s0, ns, cnt);
        /* the tiles' first entries: exclusive scan of their quads */
        for (uint32_t i0 = 0; i0 < ns; i0 += BUILD_T)
        {
            const uint32_t i = i0 + threadIdx.x;
            const uint32_t c = i < ns ? cnt[i] : 0;
            const uint32_t q = (c + OG_BIN_TILE_ALIGN - 1) / OG_BIN_TILE_ALIGN;
            const uint32_t incl = og_bin_wave_scan(q);
            if (lane == 63) s_wave[w] = incl;
            __syncthreads();
            uint32_t pre = base, tot = 0;
            for (uint32_t k = 0; k < BUILD_T / 64; k++)
            {
                pre += k < w ? s_wave[k] : 0;
                tot += s_wave[k];
            }
            base += tot;
            if (i < ns)
            {
                const uint32_t e = pre + incl - q;
                eb[i] = e;
                if (c)
                {
                    const uint32_t f = quads[(size_t)(s0 + i) * n_bins + b];
                    sb[i] = f;
                    for (uint32_t k = 0; k < q; k++) qent[f + k] = OG_BIN_TILE_ALIGN * (e + k);
                    /* padding: slot OG_BIN_PAD, source 0 */
                    for (uint32_t k = c; k < OG_BIN_TILE_ALIGN * q; k++)
                    {
                        src[(size_t)OG_BIN_TILE_ALIGN * f + k] = 0;
                        pos[(size_t)OG_BIN_TILE_ALIGN * e + k] = (uint16_t)OG_BIN_PAD;
                    }
                }
                cnt[i] = 0;
            }
            __syncthreads();
        }
        for (uint32_t k = threadIdx.x; k < d.cnt; k += BUILD_T)
        {
            const uint32_t v = cols[d.pos0 + k], sv = v / OG_BIN_SEG, sg = sv - s0;
            if (sg >= ns) continue;
            const uint32_t r = atomicAdd(&cnt[sg], 1u);
            src[(size_t)OG_BIN_TILE_ALIGN * sb[sg] + r] = (uint16_t)(v - sv * OG_BIN_SEG);
            pos[(size_t)OG_BIN_TILE_ALIGN * eb[sg] + r] = (uint16_t)k;
        }
    }
}

static unsigned og_bin_grid(uint64_t n)
{
    uint64_t g = (n + 255) / 256;
    if (g > 8192) g = 8192;
    return g ? (unsigned)g : 1u;
}

extern "C" int og_launch_bin_runs(const uint32_t *row_ptr, uint32_t Z, uint32_t *runs, uint32_t cap, uint32_t *n,
                                  hipStream_t s)
{
    if (!Z) return 0;
    OG_LAUNCH(og_bin_runs_kernel, dim3(og_bin_grid(Z)), dim3(256), 0, s, row_ptr, Z, (uint2 *)runs, cap, n);
    return og_hip_check(og_launch_status(), "og_bin_runs_kernel");
}

extern "C" int og_launch_bin_count(const og_bin_desc *bins, uint32_t n_bins, const uint32_t *cols, uint32_t n_seg,
                                   uint32_t *quads, uint32_t *bin_quads, hipStream_t s)
{
    if (!n_bins) return 0;
    OG_LAUNCH(og_bin_count_kernel, dim3(n_bins), dim3(BUILD_T), 0, s, bins, n_bins, cols, n_seg, quads, bin_quads);
    return og_hip_check(og_launch_status(), "og_bin_count_kernel");
}

extern "C" int og_launch_bin_place(og_bin_desc *bins, uint32_t n_bins, uint32_t n_all, const uint32_t *bin_quads,
                                   const uint32_t *quads, uint32_t n_seg, uint32_t *seg_src, hipStream_t s)
{
    OG_LAUNCH(og_bin_place_kernel, dim3(og_bin_grid(n_all > n_seg ? n_all : n_seg + 1)), dim3(256), 0, s, bins, n_bins,
              n_all, bin_quads, quads, n_seg, seg_src);
    return og_hip_check(og_launch_status(), "og_bin_place_kernel");
}

extern "C" int og_launch_bin_sched(const og_bin_desc *bins, const uint32_t *order, uint32_t n, og_bin_desc *sched,
                                   hipStream_t s)
{
    if (!n) return 0;
    OG_LAUNCH(og_bin_sched_kernel, dim3(og_bin_grid(n)), dim3(256), 0, s, bins, order, n, sched);
    return og_hip_check(og_launch_status(), "og_bin_sched_kernel");
}

extern "C" int og_launch_bin_fill(const og_bin_desc *bins, uint32_t n_bins, const uint32_t *cols, uint32_t n_seg,
                                  const uint32_t *quads, uint16_t *src, uint16_t *pos, uint32_t *qent, hipStream_t s)
{
    if (!n_bins) return 0;
    OG_LAUNCH(og_bin_fill_kernel, dim3(n_bins), dim3(BUILD_T), 0, s, bins, n_bins, cols, n_seg, quads, src, pos, qent);
    return og_hip_check(og_launch_status(), "og_bin_fill_kernel");
}
