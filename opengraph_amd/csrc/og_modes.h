/*
 * og_modes.h -- the arithmetic of the PageRank variants on the GPU: element
 * and accumulator types, the next rank from a row's sum, the contribution
 * the next iteration gathers.
 */
#ifndef OG_MODES_H
#define OG_MODES_H

#include <hip/hip_runtime.h>

#include "og_common.h"
#include "og_pr.h"

/* ------------------------------------------------------------------ */
/* per-mode arithmetic                                                 */
/* ------------------------------------------------------------------ */

template <int MODE> struct og_mode;
template <> struct og_mode<OG_MODE_F32>  { typedef float    elem; typedef float    acc; };
template <> struct og_mode<OG_MODE_FX64> { typedef uint64_t elem; typedef uint64_t acc; };
template <> struct og_mode<OG_MODE_FX32> { typedef uint32_t elem; typedef uint64_t acc; };
template <> struct og_mode<OG_MODE_FX16> { typedef uint16_t elem; typedef uint64_t acc; };
template <> struct og_mode<OG_MODE_FX8>  { typedef uint8_t  elem; typedef uint64_t acc; };
template <> struct og_mode<OG_MODE_Q32>  { typedef uint32_t elem; typedef uint64_t acc; };
template <> struct og_mode<OG_MODE_Q16>  { typedef uint16_t elem; typedef uint64_t acc; };
template <> struct og_mode<OG_MODE_Q8>   { typedef uint8_t  elem; typedef uint64_t acc; };

/* The reference's next-rank expression for each variant, from the gathered
 * sum (pageRank.c:1016, :1278, :1412, :1544, :1676, :1944, :2083, :2222). */
template <int MODE>
__device__ __forceinline__ float og_next_rank(typename og_mode<MODE>::acc s, const og_qparams *qp)
{
    const float base = OG_BASE_PR, damp = OG_DAMP;
    if constexpr (MODE == OG_MODE_F32) return base + (damp * s);
    else if constexpr (MODE == OG_MODE_FX64)
        return (float)((double)base + ((double)damp * ((double)s / 4294967296.0)));
    else if constexpr (MODE == OG_MODE_FX32) return base + (damp * ((float)s / 65536.0f));
    else if constexpr (MODE == OG_MODE_FX16) return base + (damp * ((float)s / 16384.0f));
    else if constexpr (MODE == OG_MODE_FX8) return base + (damp * ((float)s / 64.0f));
    else if constexpr (MODE == OG_MODE_Q32) return base + damp * (float)(qp->scale_d * (double)s);
    else return base + damp * (qp->scale_f * (float)s);
}

/* The contribution the next iteration gathers (pageRank.c:989-996 and the
 * fixed-point conversions of fixedPoint.h:29-36).  Quantized modes store
 * the fp32 quotient; og_quantize_kernel converts it once the scale is known. */
template <int MODE>
__device__ __forceinline__ void og_store_contrib(void *c_out, uint32_t v, float r, uint32_t deg)
{
    /* Stores are non-temporal: the next iteration reads them back through
     * L2, this one must not let them evict the lines being gathered. */
    if constexpr (MODE == OG_MODE_F32 || MODE >= OG_MODE_Q32)
        __builtin_nontemporal_store(deg ? r / (float)deg : 0.0f, &((float *)c_out)[v]);
    else
    {
        typedef typename og_mode<MODE>::elem E;
        E x = 0;
        if (deg)
        {
            float q = r / (float)deg;
            if constexpr (MODE == OG_MODE_FX64) x = og_fixed64_of(q);
            else if constexpr (MODE == OG_MODE_FX32)
                x = (uint32_t)og_x86_f2i64(q * 65536.0f + (q >= 0 ? 0.5f : -0.5f));
            else if constexpr (MODE == OG_MODE_FX16)
                x = (uint16_t)og_x86_f2i32(q * 16384.0f + (q >= 0 ? 0.5f : -0.5f));
            else
                x = (uint8_t)og_x86_f2i32(q * 64.0f + (q >= 0 ? 0.5f : -0.5f));
        }
        __builtin_nontemporal_store(x, &((E *)c_out)[v]);
    }
}

/* og_fixed64_of for 0 <= q < 2^32 in fp32 steps that are all exact: the whole
 * part and the fraction apart, the fraction scaled by 2^32, halves rounded up
 * (a q with a fraction below 2^-32 has no whole part).  A handful of
 * full-rate operations; the fp64 form's conversions would bound a sum over
 * converted values. */
__device__ __forceinline__ uint64_t og_fixed64_split(float q)
{
    if (__float_as_uint(q) >= 0x4F800000u) return og_fixed64_of(q);   /* 2^32 and above, negative, NaN */
    const float w = floorf(q);
    const float v = ldexpf(q - w, 32);
    const float t = floorf(v);
    return ((uint64_t)(uint32_t)w << 32) + ((uint32_t)t + (v - t >= 0.5f ? 1u : 0u));
}

#endif
