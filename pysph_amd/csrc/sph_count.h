// What the list count pass decides about a lane's sixteen products (candidate
// x destination values d^2 - R^2 in cells, see k_nnps_count): the part without
// device intrinsics, so that it also compiles for the host.
#pragma once

#include <math.h>
#include <stdint.h>

#define NN_BAND (64.0f * 0x1p-24f)   // times M^2
#define NN_FAR 1e30f                 // value of an absent candidate or destination

// All three coordinates within lim of the cell's centre.  Each is tested by
// itself: fmaxf leaves a NaN out when its other operand is a number.
__host__ __device__ __forceinline__ bool nn_inside(float x, float y, float z, float lim)
{
    return fabsf(x) <= lim && fabsf(y) <= lim && fabsf(z) <= lim;
}

// A destination whose column the error band covers: its coordinates and its
// radius (in cells) within lim.  NaN fails.
__host__ __device__ __forceinline__ bool nn_regular(float x, float y, float z, float radius,
                                                    float lim)
{
    return nn_inside(x, y, z, lim) && fabsf(radius) <= lim;
}

// Cell sizes whose float reciprocal, and coordinates over it, keep their 24
// bits, and whose squares neither underflow nor overflow in the float
// predicate: the band's assumptions.  Other grids are decided by the predicate
// throughout.
__host__ __device__ __forceinline__ bool nn_cell_size(double cs)
{
    return cs >= 0x1p-60 && cs <= 0x1p60;
}

// bits 0..15: which of a lane's candidates exist, `left` of them or more
__host__ __device__ __forceinline__ uint32_t nn_present(int32_t left)
{
    return left >= 16 ? 0xffffu : left > 0 ? (1u << left) - 1u : 0u;
}

// The lane's hits: `bits` are the signs of D, and the pairs within the band
// -- with `all`, every pair -- are asked of the predicate hit(e).  `all` also
// clears the signs: with a non-finite operand even an absent candidate's D is
// a NaN of either sign.  (Without it every operand is finite, and an absent
// candidate's D is positive.)
template <typename V, typename Hit>
__host__ __device__ __forceinline__ uint32_t nn_decide(uint32_t bits, const V &D, float band,
                                                       bool all, bool none, int32_t left, Hit hit)
{
    uint32_t ask = none ? 0u : nn_present(left);
    if (all || none) bits = 0;
    if (!all) {
        uint32_t in = 0;
#pragma unroll
        for (int e = 15; e >= 0; --e) in = 2 * in + (fabsf(D[e >> 2][e & 3]) < band);
        ask &= in;
    }
    while (ask) {
        const int e = __builtin_ctz(ask);
        ask &= ask - 1;
        bits = (bits & ~(1u << e)) | ((uint32_t)hit(e) << e);
    }
    return bits;
}
