#pragma once
/*
 * What the tiled 1D marches (onedim.hip, spacetime.hip) share: blocks of four
 * wavefronts with a solution element per lane, the shift to the neighbouring
 * lane, and quotients that share a denominator's reciprocal.
 */

#include "common.hpp"

namespace scamd
{

constexpr int TBLOCK = 256;
constexpr int TWAVES = TBLOCK / 64;
constexpr int GROUP = 8; // steps between exchanges of overlapping wavefronts

__device__ inline double recip_of(double d)
{
    double y = __builtin_amdgcn_rcp(d);
    double e = __builtin_fma(-d, y, 1.0);
    y = __builtin_fma(y, e, y);
    e = __builtin_fma(-d, y, 1.0);
    return __builtin_fma(y, e, y);
}

// a / d; with FAST from r = recip_of(d) by the last three steps of the IEEE
// division, which is the division unless it scales its operands: never for
// 2^-500 <= d < 2^92 and a = 0 or 2^-922 <= |a| < 2^261.  The remainder is
// taken as d q - a, so a zero quotient keeps the sign of a (d is positive):
// from a - d q a negative zero would come out as a positive one.
template <bool FAST>
struct Quot
{
    double d;
    double r;
    __device__ explicit Quot(double den)
        : d(den)
        , r(FAST ? recip_of(den) : 0.0)
    {
    }
    __device__ Quot(double den, double rec)
        : d(den)
        , r(rec)
    {
    }
    __device__ double operator()(double a) const
    {
        if constexpr (FAST)
        {
            double const q = a * r;
            double const over = __builtin_fma(d, q, -a);
            return __builtin_fma(-over, r, q);
        }
        else
        {
            return a / d;
        }
    }
};

// v of the next lane (wave_shl:1) or the one before (wave_shr:1); the lane at
// the end of the wavefront keeps its own.
template <bool NEXT>
__device__ inline double shift_lane(double v)
{
    constexpr int CTRL = NEXT ? 0x130 : 0x138;
    int const l = __double2loint(v);
    int const h = __double2hiint(v);
    int const lo = __builtin_amdgcn_update_dpp(l, l, CTRL, 0xf, 0xf, false);
    int const hi = __builtin_amdgcn_update_dpp(h, h, CTRL, 0xf, 0xf, false);
    return __hiloint2double(hi, lo);
}

} /* end namespace scamd */
