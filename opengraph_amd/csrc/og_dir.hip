/*
 * og_dir.hip -- gfx950 kernel of the direct pull (og_dir.h).
 *
 * What bounds a small graph is not its bytes but the chain of one iteration:
 * launches, the gathers' latency, the longest row's sum, the reduction, and
 * the gaps between them.  us an iteration, whole runs of 100, binned pull
 * (three launches, with the same row sums) against this one: R-MAT, 2^10
 * vertices and 12 k edges 18.2 and 6.3; 2^14 and 200 k 22.5 and 9.2; 2^16 and
 * 1 M 27.8 and 18.5; uniform, 20,000 vertices and 300 k edges 17.6 and 7.1.
 * Of the 6.3 about 0.8 wait at the barrier for the slowest block, 1 gather, 3
 * add the longest row, 1.2 reduce the block's statistics and get its stores
 * out; at 2^16 vertices the block of the longest row (13 k terms) gathers for
 * 6 us after the caches' invalidation and adds for 8, the others wait.  (A
 * predicted binade per lane, and a block's eight wavefronts on one row, were no
 * faster: the crossings' serial steps and the barriers between the wavefronts
 * took what the parallel adds gave.)
 */
#include <hip/hip_runtime.h>

#include "og_dir.h"
#include "og_internal.h"
#include "og_pr.h"
#include "og_rowsum.h"

#define DT OG_DIR_THREADS
#define DW (OG_DIR_THREADS / 64)
#define DQ 4u               /* values of a thread read together */
#define DG 12u              /* values of a thread gathered together */
#define DBATCH (DG * DT)    /* in-edges whose source ids a block keeps in registers */

template <typename T> __device__ __forceinline__ T og_dir_peek(const T *p)
{
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

template <typename T> __device__ __forceinline__ void og_dir_post(T *p, T x)
{
    __hip_atomic_store(p, x, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

/* The grid barrier.  A block that has finished iteration `it` posts its
 * statistics and then it + 1 as its flag; the first block of each DGRP waits
 * for its group's flags and posts the group's, and everyone waits for the
 * groups' (few blocks: for each other's).  Everything blocks pass to each
 * other goes through agent-scope accesses, so a wavefront only waits for its
 * own stores, and one cache invalidation per block follows.  (A write-back and
 * an invalidation per wavefront around one shared counter made the barrier of
 * 512 blocks 60 us long; all blocks polling all flags took 8 us more than this
 * at 512.) */
#define DGRP 32u
#define DFAIL_EVERY 64u   /* polls between looks at FAIL (a look at each would lengthen every wait) */
__device__ __forceinline__ bool og_dir_poll(const og_dir_dev &b, uint32_t word, uint32_t n, uint32_t it)
{
    bool ok = true;
    if (threadIdx.x < n)
    {
        uint32_t k = 0;
        while (og_dir_peek(&b.bar[word + threadIdx.x]) <= it && k < b.spin)
        {
            __builtin_amdgcn_s_sleep(1);
            k++;
            if (k % DFAIL_EVERY == DFAIL_EVERY / 2 && og_dir_peek(&b.bar[OG_DIR_FAIL])) k = b.spin;
        }
        ok = k < b.spin;
    }
    /* those still waiting, and those that get a CU only now, leave too within
     * DFAIL_EVERY polls; the host starts again */
    if (!ok) og_dir_post(&b.bar[OG_DIR_FAIL], 1u);
    return __syncthreads_and(ok);
}

__device__ __forceinline__ void og_dir_done(const og_dir_dev &b, const og_pr_dev &a, uint32_t it, const og_bin_stat &st)
{
    const og_bin_stat mine = og_bin_block_stat<DT>(st);
    if (threadIdx.x == 0)
    {
        const uint32_t k = (it & 1u) * gridDim.x + blockIdx.x;
        og_dir_post(&a.part_err[k], mine.err);
        og_dir_post(&a.part_act[k], mine.active);
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   /* this wavefront's stores are out */
    __syncthreads();
    if (threadIdx.x == 0) og_dir_post(&b.bar[blockIdx.x], it + 1);
}

/* False: some block did not get here within another's b.spin polls; every block
 * leaves. */
__device__ __forceinline__ bool og_dir_wait(const og_dir_dev &b, uint32_t it)
{
    const uint32_t nb = gridDim.x;
    bool ok = true;
    if (nb <= 2 * DGRP) ok = og_dir_poll(b, 0, nb, it);
    else
    {
        if (blockIdx.x % DGRP == 0)
        {
            ok = og_dir_poll(b, blockIdx.x, min(DGRP, nb - blockIdx.x), it);
            if (ok && threadIdx.x == 0) og_dir_post(&b.bar[OG_DIR_GROUP + blockIdx.x / DGRP], it + 1);
        }
        ok = ok && og_dir_poll(b, OG_DIR_GROUP, (nb + DGRP - 1) / DGRP, it);
    }
    if (threadIdx.x < 64) __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
    __syncthreads();
    return ok;
}

/* Iteration `it`'s statistics row from the blocks' partials, in block order,
 * and the stop rule; by the last block, whose rows are the shortest.  The
 * others learn of a stop one iteration later (STOP = it + 1, out before this
 * block's next flag) and fall back to the ranks of iteration `it`, which
 * keeps the reduction off the iteration's critical path. */
__device__ __forceinline__ void og_dir_fold(const og_dir_dev &b, const og_pr_dev &a, uint32_t it)
{
    og_bin_stat f;
    og_bin_stat_init(f);
    if (threadIdx.x < gridDim.x)
    {
        const uint32_t k = (it & 1u) * gridDim.x + threadIdx.x;
        f.err = og_dir_peek(&a.part_err[k]);
        f.active = og_dir_peek(&a.part_act[k]);
    }
    f = og_bin_block_stat<DT>(f);
    if (threadIdx.x == 0 && !og_dir_peek(&b.bar[OG_DIR_STOP]))
    {
        f.err /= (double)a.N;
        if (it >= 2 && 0.0 >= a.epsilon) f.active += a.N - a.Z;   /* the rows without in-edges, left out by now */
        a.stats[it % b.stats_cap].error_total = f.err;
        a.stats[it % b.stats_cap].active = f.active;
        if ((a.stop_l1 ? f.err < a.epsilon : f.active == 0) && a.allow_stop)
        {
            *a.done = 1;
            og_dir_post(&b.bar[OG_DIR_STOP], it + 1);
        }
    }
}

/* The thread's number, new to the compiler at every use: kept out of the loop
 * over iterations, the bounded indices of all its values would be held in
 * registers that there are none for. */
__device__ __forceinline__ uint32_t og_dir_thread()
{
    uint32_t t = threadIdx.x;
    asm volatile("" : "+v"(t));
    return t;
}

/* The source ids of values [i0, i0 + DBATCH) of the n at CSR position pos,
 * thread t those of i0 + t, i0 + t + DT, ... (past the end, the last one's). */
__device__ __forceinline__ void og_dir_ids(const uint32_t *__restrict__ cols, uint32_t pos, uint32_t i0, uint32_t n,
                                           uint32_t (&id)[DG])
{
    const uint32_t t = og_dir_thread();
#pragma unroll
    for (uint32_t g = 0; g < DG; g += DQ)
        if (i0 + g * DT < n)
        {
#pragma unroll
            for (uint32_t u = g; u < g + DQ; u++) id[u] = cols[pos + min(i0 + u * DT + t, n - 1)];
        }
}

__device__ __forceinline__ void og_dir_load(const float *c, uint32_t i0, uint32_t n, const uint32_t (&id)[DG],
                                            float (&x)[DG])
{
#pragma unroll
    for (uint32_t g = 0; g < DG; g += DQ)
        if (i0 + g * DT < n)
        {
#pragma unroll
            for (uint32_t u = g; u < g + DQ; u++)
            {
                uint32_t o = id[u];
                asm volatile("" : "+v"(o));   /* or all the ids are held as 64-bit offsets */
                x[u] = c[o];
            }
        }
}

__device__ __forceinline__ void og_dir_put(uint32_t i0, uint32_t n, const float (&x)[DG], float *slot)
{
    const uint32_t t = og_dir_thread();
#pragma unroll
    for (uint32_t g = 0; g < DG; g += DQ)
        if (i0 + g * DT < n)
        {
#pragma unroll
            for (uint32_t u = g; u < g + DQ; u++)
            {
                const uint32_t i = i0 + u * DT + t;
                if (i < n) slot[i] = x[u];
            }
        }
}

template <int MODE, bool WAIT>
__global__ __launch_bounds__(DT, 4) void og_dir_kernel(og_dir_dev b, og_pr_dev a, float *c0, float *c1, uint32_t it0,
                                                       uint32_t n_it)
{
    typedef typename og_mode<MODE>::acc A;
    __shared__ __align__(16) float slot[OG_DIR_CAP];
    if (*a.done) return;
    const uint32_t lane = threadIdx.x & 63;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const og_dir_bin d = b.bins[blockIdx.x];
    const bool piece = d.kind == OG_BIN_PIECE;
    /* integer modes: a long row alone in its block is added by the whole block */
    const bool alone = MODE != OG_MODE_F32 && d.kind != OG_BIN_THREAD_ROWS && d.row1 - d.row0 == 1;
    uint32_t id[DG];   /* the first DBATCH in-edges' */
    og_dir_ids(a.cols, d.pos0, 0, d.cnt, id);
    /* this thread's row (lane l of wavefront w: the wavefront's l-th) */
    const uint32_t v = d.row0 + (d.kind == OG_BIN_THREAD_ROWS ? threadIdx.x : wave + DW * lane);
    const bool mine = v < d.row1;
    uint32_t p0 = 0, p1 = 0, deg = 0;
    float r = 0.0f;
    if (mine)
    {
        p0 = a.row_ptr[v] - d.pos0;
        p1 = a.row_ptr[v + 1] - d.pos0;
        deg = a.outdeg[v];
        r = a.r[v];
    }
    const bool last = blockIdx.x == gridDim.x - 1;
    float rp = r;   /* the rank one iteration back */
    uint32_t stop = 0;
    for (uint32_t it = it0; it < it0 + n_it; it++)
    {
        const float *c = it & 1 ? c1 : c0;
        float *cn = it & 1 ? c0 : c1;
        const bool others = WAIT && it > it0 && !a.spmv;   /* (an SpMV pass reads the same terms every time) */
        if (others && !og_dir_wait(b, it - 1)) return;
        og_bin_stat st;
        og_bin_stat_init(st);
        /* the rank of a row from its sum, its statistics and next
         * contribution (pageRank.c:1016-1028, :989-996) */
        auto update = [&](uint32_t row, A sum, float prev, uint32_t dg) {
            if (a.spmv)   /* fp32: the running y, started from the old one; u64: added onto y */
            {
                if constexpr (MODE == OG_MODE_F32) return sum;
                ((uint64_t *)a.next)[row] += (uint64_t)sum;
                return prev;
            }
            const float nr = og_next_rank<MODE>(sum, a.qp);
            const double err = fabs((double)(nr - prev));
            st.err += err;
            st.active += err >= a.epsilon;
            og_dir_post(&cn[row], og_bin_contrib<MODE>(nr, dg));
            return nr;
        };
        A y = 0;
        for (uint32_t q0 = 0; q0 < d.cnt; q0 += OG_DIR_CAP)
        {
            const uint32_t n = min(d.cnt - q0, OG_DIR_CAP);
            const uint32_t sw = others && q0 == 0 ? og_dir_peek(&b.bar[OG_DIR_STOP]) : 0;
            const uint32_t pos = d.pos0 + q0;
            {
                /* batch by batch, the next one's ids on their way */
                uint32_t nid[DG];
                float x[DG];
                const uint32_t i1 = q0 == 0 ? DBATCH : 0;
                og_dir_ids(a.cols, pos, i1, n, nid);
                if (q0 == 0)
                {
                    og_dir_load(c, 0, n, id, x);
                    og_dir_put(0, n, x, slot);
                }
                for (uint32_t i0 = i1; i0 < n; i0 += DBATCH)
                {
                    uint32_t cid[DG];
#pragma unroll
                    for (uint32_t u = 0; u < DG; u++) cid[u] = nid[u];
                    og_dir_ids(a.cols, pos, i0 + DBATCH, n, nid);
                    og_dir_load(c, i0, n, cid, x);
                    og_dir_put(i0, n, x, slot);
                }
            }
            if (others && q0 == 0)
            {
                /* (a stop at it - 1, which only some blocks may see yet,
                 * counts at the next iteration) */
                if (sw && sw < it) stop = sw;
                if (stop) break;
                if (last) og_dir_fold(b, a, it - 1);
            }
            __syncthreads();
            if (d.kind == OG_BIN_THREAD_ROWS)
            {
                rp = r;
                if (mine)
                    r = update(v, og_row_by_thread<MODE>(slot, p0, p1, (A)(MODE == OG_MODE_F32 && a.spmv ? r : 0.0f)), r,
                               deg);
            }
            else if (alone)
            {
                /* every thread its share, added up at the row's end */
                if constexpr (MODE != OG_MODE_F32)
                {
                    y += og_bin_int_strided<MODE>(slot, threadIdx.x, n, DT);
                    if (q0 + n >= d.cnt)
                    {
                        for (int o = 32; o > 0; o >>= 1) y += __shfl_xor(y, o, 64);
                        __syncthreads();   /* slot is read */
                        if (lane == 0) ((A *)slot)[wave] = y;
                        __syncthreads();
                        if (threadIdx.x == 0)
                        {
                            y = 0;
                            for (uint32_t w = 0; w < DW; w++) y += ((const A *)slot)[w];
                            rp = r;
                            r = update(v, y, r, deg);
                        }
                    }
                }
            }
            else
            {
                /* wavefront w's rows row0 + w, + DW, ... (a row in pieces: wavefront 0) */
                uint32_t l = 0;
                for (uint32_t row = d.row0 + wave; row < d.row1; row += DW, l++)
                {
                    const uint32_t j0 = piece ? 0 : (uint32_t)__builtin_amdgcn_readlane(p0, l);
                    const uint32_t j1 = piece ? n : (uint32_t)__builtin_amdgcn_readlane(p1, l);
                    const float prev = og_bin_lane(r, l);
                    const uint32_t dg = (uint32_t)__builtin_amdgcn_readlane(deg, l);
                    const A y0 = q0 ? y : (A)(MODE == OG_MODE_F32 && a.spmv ? prev : 0.0f);
                    y = og_row_by_wave<MODE, 28>(slot, j0, j1, y0, q0 ? 0 : OG_BIN_HEAD);
                    if (lane == l && q0 + n >= d.cnt)
                    {
                        rp = r;
                        r = update(row, y, prev, dg);
                    }
                }
            }
            __syncthreads();   /* the values are added */
        }
        if (stop) break;
        if (a.spmv) continue;
        if (it < 2)
        {
            /* rows without in-edges reach their fixed rank in iteration 0 and
             * have both contribution buffers filled after iteration 1 */
            for (uint32_t z = a.Z + blockIdx.x * DT + threadIdx.x; z < a.N; z += gridDim.x * DT)
                a.r[z] = update(z, 0, a.r[z], a.outdeg[z]);
        }
        if (WAIT) og_dir_done(b, a, it, st);
        else
        {
            og_bin_stat f = og_bin_block_stat<DT>(st);
            f.err /= (double)a.N;
            og_bin_write_part(a, blockIdx.x, f);   /* folded by the final reduction */
        }
    }
    if (WAIT && !a.spmv && !stop)
    {
        /* a stop at the iteration before the last, then the last one's row */
        if (!og_dir_wait(b, it0 + n_it - 1)) return;
        stop = og_dir_peek(&b.bar[OG_DIR_STOP]) == it0 + n_it - 1;
        __syncthreads();
        if (last) og_dir_fold(b, a, it0 + n_it - 1);
    }
    if (mine) a.r[v] = stop ? rp : r;
}

/* (the fp32 kernel needs the most registers) */
extern "C" uint32_t og_dir_resident(void)
{
    int nb = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, (const void *)og_dir_kernel<OG_MODE_F32, true>, DT, 0) !=
        hipSuccess)
        return 0;
    const uint32_t n = nb > 0 ? (uint32_t)nb * (uint32_t)og_num_cus() : 0;
    return n < OG_DIR_MAX_BLOCKS ? n : OG_DIR_MAX_BLOCKS;
}

template <int MODE>
static void og_launch_dir_t(const og_dir_dev *b, const og_pr_dev *a, float *c0, float *c1, uint32_t it0, uint32_t n,
                            hipStream_t s)
{
    if (n > 1 || a->spmv)
        OG_LAUNCH((og_dir_kernel<MODE, true>), dim3(b->n_bins), dim3(DT), 0, s, *b, *a, c0, c1, it0, n);
    else if (n)
        OG_LAUNCH((og_dir_kernel<MODE, false>), dim3(b->n_bins), dim3(DT), 0, s, *b, *a, c0, c1, it0, n);
}

extern "C" int og_launch_dir(const og_dir_dev *b, const og_pr_dev *a, int mode, void *c0, void *c1, uint32_t it0,
                             uint32_t n, hipStream_t s)
{
    switch (mode)
    {
    case OG_MODE_F32: og_launch_dir_t<OG_MODE_F32>(b, a, (float *)c0, (float *)c1, it0, n, s); break;
    case OG_MODE_FX64: og_launch_dir_t<OG_MODE_FX64>(b, a, (float *)c0, (float *)c1, it0, n, s); break;
    case OG_MODE_FX32: og_launch_dir_t<OG_MODE_FX32>(b, a, (float *)c0, (float *)c1, it0, n, s); break;
    default: og_set_error("og_launch_dir: bad mode %d", mode); return -1;
    }
    return og_hip_check(og_launch_status(), "og_dir_kernel");
}
