// engine_strip.hpp -- block-Jacobi strip solves and whole-wave lane shifts,
// and bounded field access, shared by the streaming and the resident solver
// kernels.
#pragma once
#include "engine_device.hpp"

namespace tea {

// Block-Jacobi strip solve of one column from its own diagonal and Ky values
// (diag[k] = diag_A at row k, ky[k] = Ky at row k, k = 0..len): the
// expressions of block_solve_strip.
template <typename T>
__device__ __forceinline__ void strip_solve_col(const T (&rhs)[STRIP], T (&z)[STRIP], int len,
                                                const T (&diag)[STRIP], const T (&ky)[STRIP + 1])
{
    T cp[STRIP], bfp[STRIP], dp[STRIP];
    cp[0] = (-ky[1]) / diag[0];
    dp[0] = rhs[0] / diag[0];
#pragma unroll
    for (int k = 1; k < STRIP; k++) {
        if (k < len) {
            bfp[k] = T(1.0) / (diag[k] - (-ky[k]) * cp[k - 1]);
            cp[k] = (-ky[k + 1]) * bfp[k];
            dp[k] = (rhs[k] - (-ky[k]) * dp[k - 1]) * bfp[k];
        }
    }
#pragma unroll
    for (int k = STRIP - 1; k >= 0; k--) {
        if (k == len - 1) z[k] = dp[k];
        else if (k < len - 1) z[k] = dp[k] - cp[k] * z[k + 1];
    }
}

// The two halves of strip_solve_col: the factors cp, bfp depend on the
// strip's diagonal and Ky only (the reference's block_init,
// tea_block_jacobi.cuknl:80-111), so a pass of several inner steps forms them
// once; strip_apply is the per-application part (block_solve_func,
// tea_block_jacobi.cuknl:9-42).  Same expressions, so the same values.
template <typename T>
__device__ __forceinline__ void strip_factor(int len, const T (&diag)[STRIP], const T (&ky)[STRIP + 1],
                                             T (&cp)[STRIP], T (&bfp)[STRIP])
{
    cp[0] = (-ky[1]) / diag[0];
    bfp[0] = T(0.0);
#pragma unroll
    for (int k = 1; k < STRIP; k++) {
        bfp[k] = cp[k] = T(0.0);
        if (k < len) {
            bfp[k] = T(1.0) / (diag[k] - (-ky[k]) * cp[k - 1]);
            cp[k] = (-ky[k + 1]) * bfp[k];
        }
    }
}

template <typename T>
__device__ __forceinline__ void strip_apply(const T (&rhs)[STRIP], T (&z)[STRIP], int len, T diag0,
                                            const T (&ky)[STRIP + 1], const T (&cp)[STRIP], const T (&bfp)[STRIP])
{
    T dp[STRIP];
    dp[0] = rhs[0] / diag0;
#pragma unroll
    for (int k = 1; k < STRIP; k++)
        if (k < len) dp[k] = (rhs[k] - (-ky[k]) * dp[k - 1]) * bfp[k];
#pragma unroll
    for (int k = STRIP - 1; k >= 0; k--) {
        if (k == len - 1) z[k] = dp[k];
        else if (k < len - 1) z[k] = dp[k] - cp[k] * z[k + 1];
    }
}

// strip_apply for FP32 with dp0 = rhs0 / diag0 formed as (float)(rhs0 * rd),
// rd = 1 / (double)diag0 rounded to double once per strip: the same float as
// the IEEE division.  The exact quotient of two floats lies at least about
// 2^-49 (relative) from every midpoint between floats (it is never one unless
// it is a float itself), and rhs0 * rd carries a relative error below 2^-52,
// so both round to the same float.
__device__ __forceinline__ void strip_apply_rd(const float (&rhs)[STRIP], float (&z)[STRIP], int len, double rd,
                                               const float (&ky)[STRIP + 1], const float (&cp)[STRIP],
                                               const float (&bfp)[STRIP])
{
    float dp[STRIP];
    dp[0] = (float)((double)rhs[0] * rd);
#pragma unroll
    for (int k = 1; k < STRIP; k++)
        if (k < len) dp[k] = (rhs[k] - (-ky[k]) * dp[k - 1]) * bfp[k];
#pragma unroll
    for (int k = STRIP - 1; k >= 0; k--) {
        if (k == len - 1) z[k] = dp[k];
        else if (k < len - 1) z[k] = dp[k] - cp[k] * z[k + 1];
    }
}

// Whole-wave lane shifts by one (DPP wave_shr:1 / wave_shl:1, VALU moves with
// no LDS round trip): lane l receives v from lane l-1 (from_below) or l+1
// (from_above); the end lane (lane 0, resp. the last lane), which has no
// source, receives 0 (bound_ctrl), so no copy of v has to be made first.
// The streaming pass never reads those end values.
__device__ __forceinline__ int dpp_shr1(int v) { return __builtin_amdgcn_mov_dpp(v, 0x138, 0xf, 0xf, true); }
__device__ __forceinline__ int dpp_shl1(int v) { return __builtin_amdgcn_mov_dpp(v, 0x130, 0xf, 0xf, true); }
__device__ __forceinline__ float lane_from_below(float v) { return __int_as_float(dpp_shr1(__float_as_int(v))); }
__device__ __forceinline__ float lane_from_above(float v) { return __int_as_float(dpp_shl1(__float_as_int(v))); }
__device__ __forceinline__ double lane_from_below(double v)
{
    const long long b = __double_as_longlong(v);
    const int lo = dpp_shr1((int)(b & 0xffffffffLL)), hi = dpp_shr1((int)(b >> 32));
    return __longlong_as_double(((long long)hi << 32) | (long long)(unsigned)lo);
}
__device__ __forceinline__ double lane_from_above(double v)
{
    const long long b = __double_as_longlong(v);
    const int lo = dpp_shl1((int)(b & 0xffffffffLL)), hi = dpp_shl1((int)(b >> 32));
    return __longlong_as_double(((long long)hi << 32) | (long long)(unsigned)lo);
}

// A field seen through a raw buffer resource of `bytes` bytes (gfx9
// descriptor word 3: 0x00020000): an offset at or beyond `bytes` reads 0 and
// writes nothing, with no memory access.
constexpr unsigned OOB = 0xFFFFFFF0u;
template <typename T> struct FieldBuf {
    __amdgpu_buffer_rsrc_t r;
    __device__ FieldBuf(const T *base, unsigned bytes)
        : r(__builtin_amdgcn_make_buffer_rsrc((void *)base, (short)0, (int)bytes, 0x00020000))
    {
    }
    // base: a uniform part of the offset (below `bytes`)
    __device__ __forceinline__ T load(unsigned off, unsigned base = 0) const
    {
        if constexpr (sizeof(T) == 4)
            return __builtin_bit_cast(T, __builtin_amdgcn_raw_buffer_load_b32(r, (int)off, (int)base, 0));
        else
            return __builtin_bit_cast(T, __builtin_amdgcn_raw_buffer_load_b64(r, (int)off, (int)base, 0));
    }
    __device__ __forceinline__ void store(unsigned off, T v, unsigned base = 0) const
    {
        if constexpr (sizeof(T) == 4)
            __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, v), r, (int)off, (int)base, 0);
        else
            __builtin_amdgcn_raw_buffer_store_b64(
                __builtin_bit_cast(decltype(__builtin_amdgcn_raw_buffer_load_b64(r, 0, 0, 0)), v), r, (int)off,
                (int)base, 0);
    }
};

}  // namespace tea
