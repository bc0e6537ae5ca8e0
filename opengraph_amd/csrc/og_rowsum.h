/*
 * og_rowsum.h -- the exact row sums of the pulls that put a bin's in-edge
 * values in LDS (og_bin.hip, og_dir.hip), and the update of a row.
 *
 * Exactness.  The reference adds a row's in-edges one after the other into
 * an fp32 running sum (pageRank.c:998-1011).  Here every row is added in
 * that order from LDS: one thread per short row, one wavefront per longer
 * row, a row longer than a bin piece by piece by one wavefront.  A wavefront
 * adds a few dozen terms per lane at a time (og_bin_wave_sum).  While the
 * running sum y stays in one binade [2^(e-1), 2^e), every representable
 * value is a multiple of u = 2^(e-24) and a term a >= 0 moves y by a whole
 * number of u that depends only on a and, where a / u ends in exactly one
 * half, on whether y / u is even.  So what a run of terms does to any y of
 * the binade is two numbers, the move of an even and of an odd y, and the
 * hardware's own adds give them: the run added to the binade's first two
 * values.  The pairs compose (an associative scan over the lanes); the first
 * lane whose terms leave the binade, or are negative or not finite, adds its
 * terms one by one from its exact y, and the scan goes on after it in the
 * new binade.  The result equals the sequential fp32 sum bit for bit.
 */
#ifndef OG_ROWSUM_H
#define OG_ROWSUM_H

#include <hip/hip_runtime.h>

#include "og_bin.h"
#include "og_modes.h"
#include "og_pr.h"

#define OG_BIN_HEAD 64u  /* leading terms of a wavefront row added one by one */

__device__ __forceinline__ float og_bin_uniform(float x)
{
    return __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(x)));
}

__device__ __forceinline__ float og_bin_lane(float x, uint32_t k)
{
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(x), k));
}

/* Inclusive prefix sum over the wavefront with DPP lane moves: shifts by
 * 1, 2, 4 and 8 within each row of 16 lanes (lanes shifted in from outside
 * the row read 0), then row 1 and row 3 add the last lane of the row below
 * (row_bcast:15), then rows 2 and 3 add lane 31 (row_bcast:31).  Every
 * disabled lane adds 0. */
__device__ __forceinline__ uint32_t og_bin_wave_scan(uint32_t v)
{
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x111, 0xF, 0xF, true);   /* row_shr:1 */
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x112, 0xF, 0xF, true);   /* row_shr:2 */
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x114, 0xF, 0xF, true);   /* row_shr:4 */
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x118, 0xF, 0xF, true);   /* row_shr:8 */
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x142, 0xA, 0xF, false);  /* row_bcast:15 */
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x143, 0xC, 0xF, false);  /* row_bcast:31 */
    return v;
}

/* (d0, d1): the moves of an even and of an odd running sum over a run of
 * terms; the run A, then the run B. */
struct og_bin_move
{
    uint32_t d0, d1;
};

__device__ __forceinline__ og_bin_move og_bin_then(og_bin_move a, og_bin_move b)
{
    og_bin_move c;
    c.d0 = a.d0 + ((a.d0 & 1u) ? b.d1 : b.d0);
    c.d1 = a.d1 + ((a.d1 & 1u) ? b.d0 : b.d1);
    return c;
}

/* the run of the lanes that the DPP control reads, then this lane's (lanes
 * with none there read the empty run) */
template <int CTRL, int ROWS, bool BOUND>
__device__ __forceinline__ void og_bin_scan_step(og_bin_move &m)
{
    og_bin_move p;
    p.d0 = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)m.d0, CTRL, ROWS, 0xF, BOUND);
    p.d1 = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)m.d1, CTRL, ROWS, 0xF, BOUND);
    m = og_bin_then(p, m);
}

/* Inclusive scan of the lanes' runs, by the steps of og_bin_wave_scan. */
__device__ __forceinline__ void og_bin_move_scan(og_bin_move &m)
{
    og_bin_scan_step<0x111, 0xF, true>(m);
    og_bin_scan_step<0x112, 0xF, true>(m);
    og_bin_scan_step<0x114, 0xF, true>(m);
    og_bin_scan_step<0x118, 0xF, true>(m);
    og_bin_scan_step<0x142, 0xA, false>(m);
    og_bin_scan_step<0x143, 0xC, false>(m);
}

/* One thread's sequential fp32 sum of slot[j, j1): the 16-byte groups
 * wholly inside the range are read 16 values at a time into two register
 * sets used in turn, each refilled right after it is added, so the loads
 * of one are in flight while the other is added. */
__device__ __forceinline__ void og_bin_add16(float &s, const float4 (&x)[4], uint32_t groups)
{
#pragma unroll
    for (uint32_t u = 0; u < 4; u++)
        if (u < groups)
        {
            s = s + x[u].x;
            s = s + x[u].y;
            s = s + x[u].z;
            s = s + x[u].w;
        }
}

__device__ __forceinline__ void og_bin_load16(const float4 *s4, uint32_t q, float4 (&x)[4])
{
    constexpr uint32_t QMAX = OG_BIN_CAP / 4 - 1;   /* last float4 of slot */
#pragma unroll
    for (uint32_t u = 0; u < 4; u++) x[u] = s4[min(q + u, QMAX)];
}

__device__ __forceinline__ float og_bin_row_sum(const float *slot, uint32_t j, uint32_t j1, float s0)
{
    float s = s0;
    const uint32_t qe = j1 >> 2;                     /* groups [q, qe) lie inside */
    uint32_t q = (j + 3) >> 2;
    if (q >= qe)
    {
        for (; j < j1; j++) s = s + slot[j];
        return s;
    }
    for (; j < 4 * q; j++) s = s + slot[j];          /* head up to a group boundary */
    const float4 *s4 = reinterpret_cast<const float4 *>(slot);
    float4 A[4], B[4];
    og_bin_load16(s4, q, A);
    og_bin_load16(s4, q + 4, B);
    for (; q + 8 <= qe; q += 8)
    {
        /* scheduling barriers keep each refill after the adds of its set
         * and before the adds of the other */
        og_bin_add16(s, A, 4);
        __builtin_amdgcn_sched_barrier(0);
        og_bin_load16(s4, q + 8, A);
        __builtin_amdgcn_sched_barrier(0);
        og_bin_add16(s, B, 4);
        __builtin_amdgcn_sched_barrier(0);
        og_bin_load16(s4, q + 12, B);
        __builtin_amdgcn_sched_barrier(0);
    }
    const uint32_t g = qe - q;                       /* 0..7 groups left, in A then B */
    og_bin_add16(s, A, g < 4 ? g : 4);
    og_bin_add16(s, B, g > 4 ? g - 4 : 0);
    for (j = 4 * qe; j < j1; j++) s = s + slot[j];   /* tail */
    return s;
}

/* One step of og_bin_wave_sum: T consecutive terms per lane (in x) added in
 * lane order onto the running sum with bits yb (uniform). */
template <uint32_t T>
__device__ __forceinline__ uint32_t og_bin_wave_step(const float4 (&x)[T / 4], uint32_t yb)
{
    const uint32_t lane = threadIdx.x & 63;
    uint32_t sign = 0;
#pragma unroll
    for (uint32_t k = 0; k < T / 4; k++)
        sign |= __float_as_uint(x[k].x) | __float_as_uint(x[k].y) | __float_as_uint(x[k].z) | __float_as_uint(x[k].w);
    uint32_t p = 0;   /* lanes below p are added */
    for (;;)
    {
        uint32_t f = p;
        if (yb - 0x0D800000u < 0x64000000u)   /* 2^-100 <= y < 2^100 */
        {
            const uint32_t bb = yb & 0xFF800000u;
            float s0 = __uint_as_float(bb), s1 = __uint_as_float(bb | 1u);
#pragma unroll
            for (uint32_t k = 0; k < T / 4; k++)
            {
                s0 = s0 + x[k].x;
                s1 = s1 + x[k].x;
                s0 = s0 + x[k].y;
                s1 = s1 + x[k].y;
                s0 = s0 + x[k].z;
                s1 = s1 + x[k].z;
                s0 = s0 + x[k].w;
                s1 = s1 + x[k].w;
            }
            og_bin_move m;
            m.d0 = __float_as_uint(s0) - bb;
            m.d1 = __float_as_uint(s1) - (bb | 1u);
            const bool bad = ((sign >> 31) != 0) | (m.d0 >= (1u << 23)) | (m.d1 >= (1u << 23));
            m.d0 = bad ? 1u << 24 : m.d0;   /* 64 of them stay below 2^31 */
            m.d1 = bad ? 1u << 24 : m.d1;
            m.d0 = lane < p ? 0u : m.d0;
            m.d1 = lane < p ? 0u : m.d1;
            og_bin_move_scan(m);
            const uint32_t d = (yb & 1u) ? m.d1 : m.d0;
            const uint64_t fail = __ballot((yb & 0x7FFFFFu) + d >= (1u << 23));
            if (!fail) return yb + (uint32_t)__builtin_amdgcn_readlane(d, 63);
            f = (uint32_t)__builtin_ctzll(fail);
            if (f) yb += (uint32_t)__builtin_amdgcn_readlane(d, f - 1);
        }
        /* lane f's terms one by one */
        float s = __uint_as_float(yb);
#pragma unroll
        for (uint32_t k = 0; k < T / 4; k++)
        {
            s = s + x[k].x;
            s = s + x[k].y;
            s = s + x[k].z;
            s = s + x[k].w;
        }
        yb = (uint32_t)__builtin_amdgcn_readlane(__float_as_uint(s), f);
        p = f + 1;
        if (p == 64) return yb;
    }
}

/* Lane's T terms slot[j + T * lane ..] (j a multiple of 4), those at or past
 * j1 as +0 when TAIL.  T is a multiple of 4 and not of 8: the lanes' 16-byte
 * reads then fall on all the banks. */
template <uint32_t T, bool TAIL>
__device__ __forceinline__ void og_bin_wave_read(const float *slot, uint32_t j, uint32_t j1, float4 (&x)[T / 4])
{
    constexpr uint32_t QMAX = OG_BIN_CAP / 4 - 1;
    const float4 *s4 = reinterpret_cast<const float4 *>(slot);
    const uint32_t i = j + T * (threadIdx.x & 63);
#pragma unroll
    for (uint32_t k = 0; k < T / 4; k++)
    {
        x[k] = s4[TAIL ? min(i / 4 + k, QMAX) : i / 4 + k];
        if (TAIL)
        {
            x[k].x = i + 4 * k < j1 ? x[k].x : 0.0f;
            x[k].y = i + 4 * k + 1 < j1 ? x[k].y : 0.0f;
            x[k].z = i + 4 * k + 2 < j1 ? x[k].z : 0.0f;
            x[k].w = i + 4 * k + 3 < j1 ? x[k].w : 0.0f;
        }
    }
}

/* The sequential fp32 sum of slot[j, j1) (LDS) onto y0, one wavefront, result
 * uniform: `head` leading terms (and those up to a multiple of 4) one after
 * the other -- near 0 the running sum crosses a binade every few terms --
 * then 64 * WT terms a step.  head = 0: y0 is the sum so far of a row taken
 * in pieces. */
#define OG_BIN_WT 36u   /* terms per lane and step (28: 2 % slower at R-MAT 20-22) */
#define OG_BIN_WS 12u   /* of a last step of at most 64 * 12 terms */
template <uint32_t WT = OG_BIN_WT>
__device__ __forceinline__ float og_bin_wave_sum(const float *slot, uint32_t j, uint32_t j1, float y0, uint32_t head)
{
    const uint32_t jh = min((j + head + 3u) & ~3u, j1);
    uint32_t yb = (uint32_t)__builtin_amdgcn_readfirstlane(
        __float_as_int(jh > j ? og_bin_row_sum(slot, j, jh, y0) : y0));
    j = jh;
    for (; j1 - j >= 64u * WT; j += 64u * WT)
    {
        float4 x[WT / 4];
        og_bin_wave_read<WT, false>(slot, j, j1, x);
        yb = og_bin_wave_step<WT>(x, yb);
    }
    if (j1 - j > 64u * OG_BIN_WS)
    {
        float4 x[WT / 4];
        og_bin_wave_read<WT, true>(slot, j, j1, x);
        yb = og_bin_wave_step<WT>(x, yb);
    }
    else if (j < j1)
    {
        float4 x[OG_BIN_WS / 4];
        og_bin_wave_read<OG_BIN_WS, true>(slot, j, j1, x);
        yb = og_bin_wave_step<OG_BIN_WS>(x, yb);
    }
    return __uint_as_float(yb);
}

/* ---- integer modes: u64 sums, exact in any order ----
 * A value in LDS is the gathered 32-bit element: the fixed-point or quantized
 * number itself, or (OG_MODE_FX64) the fp32 quotient its Q32.32 number is the
 * conversion of. */
template <int MODE> __device__ __forceinline__ uint64_t og_bin_int(float x)
{
    if constexpr (MODE == OG_MODE_FX64) return og_fixed64_split(x);
    else return __float_as_uint(x);
}

template <int MODE> __device__ __forceinline__ uint64_t og_bin_int4(float4 x)
{
    return (og_bin_int<MODE>(x.x) + og_bin_int<MODE>(x.y)) + (og_bin_int<MODE>(x.z) + og_bin_int<MODE>(x.w));
}

/* one thread's sum of slot[j, j1) */
template <int MODE> __device__ __forceinline__ uint64_t og_bin_int_row_sum(const float *slot, uint32_t j, uint32_t j1)
{
    uint64_t s = 0;
    for (; (j & 3u) && j < j1; j++) s += og_bin_int<MODE>(slot[j]);
    const float4 *s4 = reinterpret_cast<const float4 *>(slot);
    for (; j + 8 <= j1; j += 8)
    {
        const float4 x = s4[j / 4], y = s4[j / 4 + 1];
        s += og_bin_int4<MODE>(x) + og_bin_int4<MODE>(y);
    }
    for (; j < j1; j++) s += og_bin_int<MODE>(slot[j]);
    return s;
}

/* every G-th value from slot[j] on (j: this lane's first), below j1 */
template <int MODE>
__device__ __forceinline__ uint64_t og_bin_int_strided(const float *slot, uint32_t j, uint32_t j1, uint32_t G)
{
    uint64_t s = 0;
    for (; j + 3 * G < j1; j += 4 * G)
    {
        const float4 x = make_float4(slot[j], slot[j + G], slot[j + 2 * G], slot[j + 3 * G]);
        s += og_bin_int4<MODE>(x);
    }
    for (; j < j1; j += G) s += og_bin_int<MODE>(slot[j]);
    return s;
}

/* one wavefront's, the same in every lane */
template <int MODE> __device__ __forceinline__ uint64_t og_bin_int_wave_sum(const float *slot, uint32_t j, uint32_t j1)
{
    uint64_t s = og_bin_int_strided<MODE>(slot, j + (threadIdx.x & 63), j1, 64);
    for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o, 64);
    return s;
}

/* Row sums in the mode's own way: fp32 in order onto y0, integers onto 0. */
template <int MODE>
__device__ __forceinline__ typename og_mode<MODE>::acc og_row_by_thread(const float *slot, uint32_t j, uint32_t j1,
                                                                        typename og_mode<MODE>::acc y0)
{
    if constexpr (MODE == OG_MODE_F32) return og_bin_row_sum(slot, j, j1, y0);
    else return y0 + og_bin_int_row_sum<MODE>(slot, j, j1);
}

template <int MODE, uint32_t WT>
__device__ __forceinline__ typename og_mode<MODE>::acc og_row_by_wave(const float *slot, uint32_t j, uint32_t j1,
                                                                      typename og_mode<MODE>::acc y0, uint32_t head)
{
    if constexpr (MODE == OG_MODE_F32) return og_bin_wave_sum<WT>(slot, j, j1, y0, head);
    else return y0 + og_bin_int_wave_sum<MODE>(slot, j, j1);
}

/* running statistics of the updates a thread made */
struct og_bin_stat
{
    double err;
    uint32_t active;
    float cmin, cmax;   /* quantized modes: of the contributions */
};

__device__ __forceinline__ void og_bin_stat_init(og_bin_stat &s)
{
    s.err = 0.0;
    s.active = 0;
    s.cmin = 3.402823466e38f;
    s.cmax = -3.402823466e38f;
}

/* the contribution of a rank as the gather wants it: fp32 quotients but for
 * FX32's numbers (pageRank.c:989-996, fixedPoint.h:31) */
template <int MODE> __device__ __forceinline__ float og_bin_contrib(float r, uint32_t deg)
{
    const float q = deg ? r / (float)deg : 0.0f;
    if constexpr (MODE == OG_MODE_FX32)
        return __uint_as_float(deg ? (uint32_t)og_x86_f2i64(q * 65536.0f + (q >= 0 ? 0.5f : -0.5f)) : 0u);
    else return q;
}

/* pageRank.c:1016-1028 and the next contribution (pageRank.c:989-996),
 * with the old rank and out-degree already loaded. */
template <int MODE>
__device__ __forceinline__ void og_bin_epilogue_pf(const og_pr_dev &a, uint32_t v, typename og_mode<MODE>::acc sum,
                                                   float prev, uint32_t deg, og_bin_stat &st)
{
    if (a.spmv)
    {
        /* SpMV pass: fp32, the running y, started from the old one, is the sum */
        if constexpr (MODE == OG_MODE_F32) __builtin_nontemporal_store(sum, &a.r[v]);
        else ((uint64_t *)a.next)[v] += sum;
        return;
    }
    const float nr = og_next_rank<MODE>(sum, a.qp);
    __builtin_nontemporal_store(nr, &a.r[v]);
    const double err = fabs((double)(nr - prev));
    st.err += err / (double)a.N;
    st.active += err >= a.epsilon;
    const float c = og_bin_contrib<MODE>(nr, deg);
    __builtin_nontemporal_store(c, &((float *)a.c_out)[v]);
    if constexpr (MODE == OG_MODE_Q32)
    {
        st.cmin = fminf(st.cmin, c);
        st.cmax = fmaxf(st.cmax, c);
    }
}

template <int MODE>
__device__ __forceinline__ void og_bin_epilogue(const og_pr_dev &a, uint32_t v, typename og_mode<MODE>::acc sum,
                                                og_bin_stat &st)
{
    const float prev = __builtin_nontemporal_load(&a.r[v]);
    const uint32_t deg = __builtin_nontemporal_load(&a.outdeg[v]);
    og_bin_epilogue_pf<MODE>(a, v, sum, prev, deg, st);
}

/* the statistics over the block of NT threads (fixed order; MM: with the
 * contributions' range); result in thread 0 */
template <uint32_t NT, bool MM = false>
__device__ og_bin_stat og_bin_block_stat(og_bin_stat s)
{
    constexpr uint32_t W = NT / 64;
    __shared__ double sh_err[W];
    __shared__ uint32_t sh_act[W];
    __shared__ float sh_min[MM ? W : 1], sh_max[MM ? W : 1];
    const uint32_t lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    for (int o = 32; o > 0; o >>= 1)
    {
        s.err += __shfl_down(s.err, o, 64);
        s.active += __shfl_down(s.active, o, 64);
        if constexpr (MM)
        {
            s.cmin = fminf(s.cmin, __shfl_down(s.cmin, o, 64));
            s.cmax = fmaxf(s.cmax, __shfl_down(s.cmax, o, 64));
        }
    }
    if (lane == 0)
    {
        sh_err[w] = s.err;
        sh_act[w] = s.active;
        if constexpr (MM)
        {
            sh_min[w] = s.cmin;
            sh_max[w] = s.cmax;
        }
    }
    __syncthreads();
    og_bin_stat r;
    og_bin_stat_init(r);
    if (threadIdx.x == 0)
        for (uint32_t i = 0; i < W; i++)
        {
            r.err += sh_err[i];
            r.active += sh_act[i];
            if constexpr (MM)
            {
                r.cmin = fminf(r.cmin, sh_min[i]);
                r.cmax = fmaxf(r.cmax, sh_max[i]);
            }
        }
    __syncthreads();
    return r;
}

/* first-level partial idx of the final reduction */
__device__ __forceinline__ void og_bin_write_part(const og_pr_dev &a, uint32_t idx, const og_bin_stat &r)
{
    if (threadIdx.x == 0)
    {
        a.part_err[idx] = r.err;
        a.part_act[idx] = r.active;
        a.part_min[idx] = r.cmin;
        a.part_max[idx] = r.cmax;
    }
}

#endif
