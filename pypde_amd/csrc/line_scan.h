// Cross-lane scans of the banded line solves: the chunk transfers of a line
// combined over the lanes that hold it, by DPP moves (no LDS traffic).  Used by
// the lane-chunk recurrences (a wave per line) and by the fused stage kernels (a
// row of 16 lanes per line).
#pragma once
#include "common.h"

namespace pypde {

// Cross-lane moves for the lane-chunk scans.  dpp_f64<CTRL>: a DPP move of a
// double (two 32-bit moves); lanes whose source lies outside the pattern keep
// `old`.  Controls used: row_shr:d (0x110 + d) and row_shl:d (0x100 + d) move
// within rows of 16 lanes, wave_shr:1 (0x138) and wave_shl:1 (0x130) across the
// wave.  readlane_f64: one lane's value, for every lane.
template <int CTRL>
__device__ __forceinline__ double dpp_f64(double old, double x)
{
    const unsigned long long ov = __builtin_bit_cast(unsigned long long, old);
    const unsigned long long xv = __builtin_bit_cast(unsigned long long, x);
    const int lo = __builtin_amdgcn_update_dpp((int)(unsigned)ov, (int)(unsigned)xv, CTRL, 0xf, 0xf, false);
    const int hi = __builtin_amdgcn_update_dpp((int)(unsigned)(ov >> 32), (int)(unsigned)(xv >> 32), CTRL,
                                               0xf, 0xf, false);
    return __builtin_bit_cast(double, ((unsigned long long)(unsigned)hi << 32) | (unsigned)lo);
}

__device__ __forceinline__ double readlane_f64(double x, int l)
{
    const unsigned long long xv = __builtin_bit_cast(unsigned long long, x);
    const unsigned lo = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)xv, l);
    const unsigned hi = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)(xv >> 32), l);
    return __builtin_bit_cast(double, ((unsigned long long)hi << 32) | lo);
}

// Forward chain maps y -> A y + B; (A, B) after (Ap, Bp): A Ap, A Bp + B.
// One step of the inclusive scan within rows of 16 lanes: lane l composes the
// map of lane l - D of its row (when there is one) before its own.
template <int D>
__device__ __forceinline__ void fwd_row_step(double& A, double& B, int lane)
{
    const double Au = dpp_f64<0x110 + D>(1.0, A);
    const double Bu = dpp_f64<0x110 + D>(0.0, B);
    const double nb = A * Bu + B, na = A * Au;
    const bool in = (lane & 15) >= D;
    B = in ? nb : B;
    A = in ? na : A;
}

// Backward chain maps (Z1, Z2) -> s + M (Z1, Z2), M = [a1 b1; a2 b2]; a lane's
// map applied after the map of the lane above it (its input is that lane's
// output): own.s1 + own.a1 t.s1 + own.b1 t.s2, ...
struct BwdMap {
    double s1, s2, a1, b1, a2, b2;
};

__device__ __forceinline__ BwdMap bwd_compose(const BwdMap& x, const BwdMap& t)
{
    return BwdMap{x.s1 + x.a1 * t.s1 + x.b1 * t.s2, x.s2 + x.a2 * t.s1 + x.b2 * t.s2,
                  x.a1 * t.a1 + x.b1 * t.a2,         x.a1 * t.b1 + x.b1 * t.b2,
                  x.a2 * t.a1 + x.b2 * t.a2,         x.a2 * t.b1 + x.b2 * t.b2};
}

template <int D>
__device__ __forceinline__ void bwd_row_step(BwdMap& m, int lane)
{
    const BwdMap t{dpp_f64<0x100 + D>(0.0, m.s1), dpp_f64<0x100 + D>(0.0, m.s2),
                   dpp_f64<0x100 + D>(1.0, m.a1), dpp_f64<0x100 + D>(0.0, m.b1),
                   dpp_f64<0x100 + D>(0.0, m.a2), dpp_f64<0x100 + D>(1.0, m.b2)};
    const BwdMap c = bwd_compose(m, t);
    const bool in = (lane & 15) + D < 16;
    m.s1 = in ? c.s1 : m.s1; m.s2 = in ? c.s2 : m.s2;
    m.a1 = in ? c.a1 : m.a1; m.b1 = in ? c.b1 : m.b1;
    m.a2 = in ? c.a2 : m.a2; m.b2 = in ? c.b2 : m.b2;
}

}  // namespace pypde
