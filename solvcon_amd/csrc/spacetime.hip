/*
 * One-dimensional space-time CESE scalar engine on the GPU: the device
 * counterpart of solvcon's spacetime SolverBase (cpp/solvcon/spacetime/
 * core.hpp:706-1036, core.cpp:14-116) with the element kernels of
 * kernel/linear_scalar.hpp:45-87, kernel/inviscid_burgers.hpp:51-109 and the
 * default hooks of Kernel::reset (core.hpp:520-536).
 *
 * Layout as in the reference: coordinates xc[nx] (nx = 2*ncelm + 5, two
 * mirrored ghost points each side), so0/so1[nx][nvar] row-major, cfl[nx].
 * Solution element j of a plane sits at xindex 2 + 2j + odd, conservation
 * element j at 3 + 2j + odd; only variable 0 is marched.
 *
 * One half step is one kernel: each thread owns one conservation element,
 * forms the new so0 at its centre, the CFL number of the solution element
 * there and the new so1, and the threads of the first and last elements
 * also write the periodic ghost points (treat_boundary_so0/so1,
 * core.hpp:982-1004).  A march of several steps is tiled: segments with
 * halos, an element per lane in registers, up to 64 steps per launch.
 */

#include "common.hpp"
#include "lane1d.hpp"

#include <cfloat>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <string>
#include <utility>
#include <vector>

namespace scamd
{
namespace
{

constexpr unsigned ST_BLOCK = 256;

enum StKind : int
{
    K_DEFAULT = 0,
    K_LINEAR = 1,
    K_BURGERS = 2,
};

// Coordinates and variable-0 state as seen by one element evaluation; the
// accessors take an xindex.  The same code runs on global memory and on LDS.
struct StView
{
    double const * xc;
    double const * u;
    double const * ux;
    int64_t stride;
    double hdt;
    double qdt;

    __device__ double x(int64_t y) const { return xc[y]; }
    __device__ double xneg(int64_t y) const { return xc[y - 1]; }
    __device__ double xpos(int64_t y) const { return xc[y + 1]; }
    __device__ double xctr(int64_t y) const { return (xneg(y) + xpos(y)) / 2; }
    __device__ double dxneg(int64_t y) const { return x(y) - xneg(y); }
    __device__ double dxpos(int64_t y) const { return xpos(y) - x(y); }
    __device__ double so0(int64_t y) const { return u[y * stride]; }
    __device__ double so1(int64_t y) const { return ux[y * stride]; }
};

template <int K>
__device__ inline double se_xn(StView const & v, int64_t y)
{
    if constexpr (K == K_DEFAULT)
    {
        return 0.0;
    }
    else
    {
        double const displacement = 0.5 * (v.x(y) + v.xneg(y)) - v.xctr(y);
        return v.dxneg(y) * (v.so0(y) + displacement * v.so1(y));
    }
}

template <int K>
__device__ inline double se_xp(StView const & v, int64_t y)
{
    if constexpr (K == K_DEFAULT)
    {
        return 0.0;
    }
    else
    {
        double const displacement = 0.5 * (v.x(y) + v.xpos(y)) - v.xctr(y);
        return v.dxpos(y) * (v.so0(y) + displacement * v.so1(y));
    }
}

// tn (sign +1) and tp (sign -1): the flux through the temporal faces.
template <int K, int SIGN>
__device__ inline double se_t(StView const & v, int64_t y)
{
    if constexpr (K == K_DEFAULT)
    {
        return 0.0;
    }
    else if constexpr (K == K_LINEAR)
    {
        double const displacement = v.x(y) - v.xctr(y);
        double ret = v.so0(y);
        ret += displacement * v.so1(y);
        if constexpr (SIGN > 0)
        {
            ret += v.qdt * v.so1(y);
        }
        else
        {
            ret -= v.qdt * v.so1(y);
        }
        return v.hdt * ret;
    }
    else
    {
        double const displacement = v.x(y) - v.xctr(y);
        double const u = v.so0(y);
        double const u_2 = u * u;
        double ret = 0.5 * u_2;
        ret += displacement * u * v.so1(y);
        if constexpr (SIGN > 0)
        {
            ret += v.qdt * u_2 * v.so1(y);
        }
        else
        {
            ret -= v.qdt * u_2 * v.so1(y);
        }
        return v.hdt * ret;
    }
}

template <int K>
__device__ inline double se_so0p(StView const & v, int64_t y)
{
    if constexpr (K == K_DEFAULT)
    {
        return v.so0(y);
    }
    else
    {
        double ret = v.so0(y);
        ret += (v.x(y) - v.xctr(y)) * v.so1(y);
        ret -= v.hdt * v.so1(y);
        return ret;
    }
}

// update_cfl of the solution element at y with so0 value u0.
template <int K>
__device__ inline double se_cfl(StView const & v, int64_t y, double u0)
{
    if constexpr (K == K_DEFAULT)
    {
        return 0.0;
    }
    else
    {
        double const dn = v.dxneg(y);
        double const dp = v.dxpos(y);
        double const hdx = dp < dn ? dp : dn; // std::min(dxneg, dxpos)
        if constexpr (K == K_LINEAR)
        {
            return v.hdt / hdx;
        }
        else
        {
            return fabs(u0) * v.hdt / hdx;
        }
    }
}

// Celm::calc_so0 (core.hpp:645-653) of the CE centred at X.
template <int K>
__device__ inline double ce_so0(StView const & v, int64_t X)
{
    double const flux_ll = se_xp<K>(v, X - 1) + se_t<K, -1>(v, X - 1);
    double const flux_ur = se_xn<K>(v, X + 1) - se_t<K, -1>(v, X + 1);
    return (flux_ll + flux_ur) / (v.xpos(X) - v.xneg(X));
}

template <int A>
__device__ inline double alpha_pow(double a)
{
    if constexpr (A == 0)
    {
        return 1.0;
    }
    else if constexpr (A == 1)
    {
        return a;
    }
    else
    {
        return a * a;
    }
}

// Celm::calc_so1_alpha (core.hpp:655-672) with the new so0 value utp at X.
template <int K, int A>
__device__ inline double ce_so1(StView const & v, int64_t X, double utp)
{
    double const upn = se_so0p<K>(v, X - 1);
    double const upp = se_so0p<K>(v, X + 1);
    double const duxn = (utp - upn) / v.dxpos(X - 1);
    double const duxp = (upp - utp) / v.dxneg(X + 1);
    double const fan = alpha_pow<A>(fabs(duxn));
    double const fap = alpha_pow<A>(fabs(duxp));
    return (fap * duxn + fan * duxp) / (fap + fan + DBL_MIN);
}

struct Plane
{
    int64_t first; // xindex of the first conservation element
    int64_t count;
};

__host__ __device__ inline Plane ce_plane(int64_t ncelm, bool odd)
{
    // ic in [odd ? -1 : 0, ncelm), X = 3 + 2 ic + odd (core.hpp:950-957).
    return odd ? Plane{2, ncelm + 1} : Plane{3, ncelm};
}

__host__ __device__ inline Plane se_plane(int64_t ncelm, bool odd)
{
    // ic in [odd ? -1 : 0, nselm), y = 2 + 2 ic + odd (core.hpp:960-968).
    return odd ? Plane{1, ncelm + 2} : Plane{2, ncelm + 1};
}

struct StArgs
{
    int64_t ncelm;
    int64_t nvar;
    double hdt;
    double qdt;
    double const * xc;
    double * so0;
    double * so1;
    double * cfl;
};

__device__ inline StView view_of(StArgs const & a)
{
    return StView{a.xc, a.so0, a.so1, a.nvar, a.hdt, a.qdt};
}

template <int K>
__global__ void k_st_so0(StArgs a, Plane p)
{
    int64_t const k = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (k < p.count)
    {
        int64_t const X = p.first + 2 * k;
        a.so0[X * a.nvar] = ce_so0<K>(view_of(a), X);
    }
}

template <int K, int A>
__global__ void k_st_so1(StArgs a, Plane p)
{
    int64_t const k = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (k < p.count)
    {
        int64_t const X = p.first + 2 * k;
        StView const v = view_of(a);
        a.so1[X * a.nvar] = ce_so1<K, A>(v, X, v.so0(X));
    }
}

template <int K>
__global__ void k_st_cfl(StArgs a, Plane p)
{
    int64_t const k = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (k < p.count)
    {
        int64_t const y = p.first + 2 * k;
        StView const v = view_of(a);
        a.cfl[y] = se_cfl<K>(v, y, v.so0(y));
    }
}

// treat_boundary_so0/so1 (core.hpp:982-1004): periodic odd-plane ghosts.
__global__ void k_st_bnd(int64_t ncelm, int64_t nvar, double * arr)
{
    if (blockIdx.x == 0 && threadIdx.x == 0)
    {
        double const left_in = arr[3 * nvar];
        double const right_in = arr[(2 * ncelm + 1) * nvar];
        arr[1 * nvar] = right_in;
        arr[(2 * ncelm + 3) * nvar] = left_in;
    }
}

// One element of a fused half step.  First half (odd == false):
// march_half_so0(false), treat_boundary_so0, update_cfl(true),
// march_half_so1(false), treat_boundary_so1 (core.hpp:1006-1014); the
// solution element at X belongs to the odd plane, and the threads of the
// first and last CEs also write the ghost points 2 ncelm + 3 and 1.  Second
// half: march_half_so0(true), update_cfl(false), march_half_so1(true)
// (core.hpp:1016-1024).
template <int K, int A>
__device__ inline void st_half_elem(StView const & v, int64_t ncelm, bool odd, int64_t k, double * so0, double * so1,
                                    int64_t stride, double * cfl)
{
    int64_t const X = (odd ? 2 : 3) + 2 * k;
    double const s0 = ce_so0<K>(v, X);
    double const c = se_cfl<K>(v, X, s0);
    double const s1 = ce_so1<K, A>(v, X, s0);
    so0[X * stride] = s0;
    so1[X * stride] = s1;
    if (cfl != nullptr)
    {
        cfl[X] = c;
    }
    if (!odd)
    {
        if (k == ncelm - 1)
        {
            so0[1 * stride] = s0;
            so1[1 * stride] = s1;
            if (cfl != nullptr)
            {
                cfl[1] = se_cfl<K>(v, 1, s0);
            }
        }
        if (k == 0)
        {
            int64_t const g = 2 * ncelm + 3;
            so0[g * stride] = s0;
            so1[g * stride] = s1;
            if (cfl != nullptr)
            {
                cfl[g] = se_cfl<K>(v, g, s0);
            }
        }
    }
}

template <int K, int A>
__global__ void k_st_half(StArgs a, int odd)
{
    int64_t const k = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    int64_t const count = odd ? a.ncelm + 1 : a.ncelm;
    if (k < count)
    {
        st_half_elem<K, A>(view_of(a), a.ncelm, odd != 0, k, a.so0, a.so1, a.nvar, a.cfl);
    }
}

// The tiled march_alpha<A>.  The even rows 0, 2, ..., 2 ncelm + 2 (row 0 only
// stands before the ghost at 1) are a ring of ncelm + 2 elements.  Block b
// owns elements [b seg, (b + 1) seg), takes halo elements on each side (round
// the ring, as often as the window asks for), runs `steps` steps without other
// blocks and writes its own rows to (out0, out1).  A lane holds the even row r
// before the first half step and the odd row r + 1 after it, and hands its
// neighbour two values by a DPP shift; the stale values at a window's or
// wavefront's end spread by an element per step.  The odd ghosts take their
// values from the element on the other side of the seam, two lanes away,
// which moves a stale end two elements further at each seam it passes: so the
// halo (st_halo), and the GROUP + 2 elements by which neighbouring wavefronts
// overlap between their exchanges through LDS: every GROUP steps on a ring
// longer than the overlap, every step on a shorter one.
//
// The reciprocals of the widths are formed once per launch, and quotients
// taken from them (Quot) while values keep the range where that is the
// division: the new so0 zero or in [2^-301, 2^200], the one-sided gradients
// zero or in [2^-241, 2^45] (then the weights' sum is at least 2^-482, or the
// numerator zero), the widths in [2^-200, 2^60].  The lanes note values out of
// range and look at the notes once per exchange: then the wavefront goes back
// to the values it had after the last exchange and runs those steps with the
// divisions.  (A look in every half step stands in its serial chain: 0.34 us
// per half step instead of 0.28 at 1000 elements, 0.81 instead of 0.75 at
// 100000.)
//
// A short ring is bound by the latency of a half step, about 60 instructions:
// 0.28 us, against 1.3 us in one workgroup with the state in LDS (1000
// elements); 100000 elements take 0.75 us against 3.4 us with a launch per
// half step.
constexpr int ST_OVER = GROUP + 2;
constexpr int ST_STRIDE = 64 - 2 * ST_OVER;
constexpr int ST_ELEMS = (TWAVES - 1) * ST_STRIDE + 64; // of a window

// Halo elements of a window for `steps` steps on a ring of `ring` elements:
// one per step, two of rounding up, two per seam in the halo itself.
inline int64_t st_halo(int64_t steps, int64_t ring)
{
    int64_t h = steps + 2;
    for (int64_t was = 0; was != h;)
    {
        was = h;
        h = steps + 2 + 2 * (h / ring + 1);
    }
    return h;
}

struct StTile
{
    int64_t ncelm;
    int64_t seg;
    int64_t halo;
    int64_t steps;
    int group;
    int last;
    double hdt;
    double qdt;
    double const * xc;
    double const * in0;
    double const * in1;
    int64_t in_stride;
    double * out0;
    double * out1;
    int64_t out_stride;
    double * cfl;
};

// The geometry of one element: x - xctr, its half widths and the offsets of
// their midpoints.
struct StOwn
{
    double c, dl, dr, ml, mr;
    __device__ void set(double xneg, double x, double xpos)
    {
        double const ctr = (xneg + xpos) / 2;
        c = x - ctr;
        dl = xpos - x;
        dr = x - xneg;
        ml = 0.5 * (x + xpos) - ctr;
        mr = 0.5 * (x + xneg) - ctr;
    }
};

// What an element gives to the conservation elements on its right (fl) and on
// its left (fr), and its so0p (se_xp, se_xn, se_t and se_so0p above).
template <int K>
__device__ inline void st_own(StOwn const & o, double hdt, double qdt, double u, double ux, double & fl, double & fr,
                              double & up)
{
    if constexpr (K == K_DEFAULT)
    {
        fl = 0.0;
        fr = 0.0;
        up = u;
        return;
    }
    double t;
    if constexpr (K == K_LINEAR)
    {
        t = u;
        t += o.c * ux;
        t -= qdt * ux;
    }
    else
    {
        double const u2 = u * u;
        t = 0.5 * u2;
        t += o.c * u * ux;
        t -= qdt * u2 * ux;
    }
    t = hdt * t;
    fl = o.dl * (u + o.ml * ux) + t;
    fr = o.dr * (u + o.mr * ux) - t;
    up = u;
    up += o.c * ux;
    up -= hdt * ux;
}

// ce_so0 and ce_so1 from the elements' contributions; ok: whether the quotients
// are the divisions (FAST).
template <int A, bool FAST>
__device__ inline void st_join(double sum, double upl, double upr, Quot<FAST> const & wx, Quot<FAST> const & wl,
                               Quot<FAST> const & wr, double & s0, double & s1, bool & ok)
{
    s0 = wx(sum);
    double const dn = wl(s0 - upl);
    double const dp = wr(upr - s0);
    double const fan = alpha_pow<A>(fabs(dn));
    double const fap = alpha_pow<A>(fabs(dp));
    Quot<FAST> const w(fap + fan + DBL_MIN);
    s1 = w(fap * dn + fan * dp);
    if constexpr (FAST)
    {
        unsigned const a = static_cast<unsigned>(__builtin_amdgcn_frexp_exp(s0) + 300);
        unsigned const b = static_cast<unsigned>(__builtin_amdgcn_frexp_exp(dn) + 240);
        unsigned const c = static_cast<unsigned>(__builtin_amdgcn_frexp_exp(dp) + 240);
        double const nan = __builtin_fma(s0, 0.0, __builtin_fma(s1, 0.0, 0.0));
        ok = a <= 500 && b <= 285 && c <= 285 && nan == 0.0;
    }
}

__device__ inline bool st_width_ok(double v)
{
    int const e = __builtin_amdgcn_frexp_exp(v);
    return v - v == 0.0 && v > 0.0 && e >= -199 && e <= 60;
}

// se_cfl of the element with so0 value u0 and half widths dl, dr.
template <int K>
__device__ inline double st_cfl(StOwn const & o, double hdt, double u0)
{
    if constexpr (K == K_DEFAULT)
    {
        return 0.0;
    }
    double const hdx = o.dl < o.dr ? o.dl : o.dr;
    return K == K_LINEAR ? hdt / hdx : fabs(u0) * hdt / hdx;
}

template <int K, int A>
__global__ void __launch_bounds__(TBLOCK) k_st_tiled(StTile const t)
{
    __shared__ double edge[ST_ELEMS * 2];
    int const lane = threadIdx.x & 63;
    int const wave = threadIdx.x >> 6;
    int const elem = wave * ST_STRIDE + lane;
    bool const mine = (lane >= ST_OVER || wave == 0) && (lane < 64 - ST_OVER || wave == TWAVES - 1);
    int64_t const ring = t.ncelm + 2;
    int64_t const first = static_cast<int64_t>(blockIdx.x) * t.seg;
    int64_t const at = elem - t.halo; // place in the block's own range
    int64_t j = (first + at) % ring;
    j = j < 0 ? j + ring : j;
    int64_t const r = 2 * j;
    int64_t const nx = 2 * t.ncelm + 5;
    bool const own = mine && at >= 0 && at < t.seg && first + at < ring;
    bool const ghost_l = j == 0;        // its odd row is the ghost 1
    bool const ghost_r = j == ring - 1; // its odd row is the ghost 2 ncelm + 3
    bool const up_even = !ghost_l;
    bool const up_odd = !ghost_l && !ghost_r;
    double x[4];
#pragma unroll
    for (int k = 0; k < 4; ++k)
    {
        int64_t const y = r - 1 + k;
        x[k] = t.xc[y < 0 ? 0 : y < nx ? y : nx - 1];
    }
    // Row 0 is no solution element and takes no part.
    double u = ghost_l ? 0.0 : t.in0[r * t.in_stride];
    double ux = ghost_l ? 0.0 : t.in1[r * t.in_stride];
    // Every wavefront has read before one writes: a block alone on its ring
    // writes where it read.
    __syncthreads();
    StOwn even;
    StOwn odd;
    even.set(x[0], x[1], x[2]);
    odd.set(x[1], x[2], x[3]);
    double const wx0 = x[3] - x[1];
    double const wl0 = x[2] - x[1];
    double const wr0 = x[3] - x[2];
    double const wx1 = x[2] - x[0];
    double const wl1 = x[1] - x[0];
    bool const fixed = __all((!up_odd || (st_width_ok(wx0) && st_width_ok(wr0))) &&
                             (!up_even || (st_width_ok(wl0) && st_width_ok(wx1) && st_width_ok(wl1))));
    Quot<true> const qx0(wx0);
    Quot<true> const ql0(wl0);
    Quot<true> const qr0(wr0);
    Quot<true> const qx1(wx1);
    Quot<true> const ql1(wl1);
    bool const seam = __any(ghost_l || ghost_r);
    double v = 0.0; // the odd row
    double vx = 0.0;
    // One step; bad: whether a value left the range of the quotients.
    auto step = [&](auto fast, int64_t it, bool & bad)
    {
        constexpr bool FAST = decltype(fast)::value;
        bool const cfl_now = t.last != 0 && it + 1 == t.steps;
        double fl, fr, up;
        bool ok = true;
        st_own<K>(even, t.hdt, t.qdt, u, ux, fl, fr, up);
        {
            double const nf = shift_lane<true>(fr);
            double const nu = shift_lane<true>(up);
            st_join<A, FAST>(fl + nf, up, nu, Quot<FAST>(wx0, qx0.r), Quot<FAST>(wl0, ql0.r), Quot<FAST>(wr0, qr0.r), v, vx,
                             ok);
            bad = bad || !(ok || !up_odd);
        }
        if (seam)
        {
            // treat_boundary_so0 / so1: the ghost 2 ncelm + 3 takes row 3, two
            // lanes on, the ghost 1 row 2 ncelm + 1, two lanes back.
            double const a = shift_lane<true>(shift_lane<true>(v));
            double const b = shift_lane<true>(shift_lane<true>(vx));
            double const c = shift_lane<false>(shift_lane<false>(v));
            double const d = shift_lane<false>(shift_lane<false>(vx));
            v = ghost_r ? a : ghost_l ? c : v;
            vx = ghost_r ? b : ghost_l ? d : vx;
        }
        if (__builtin_expect(cfl_now, 0))
        {
            if (own)
            {
                t.cfl[r + 1] = st_cfl<K>(odd, t.hdt, v);
            }
        }
        st_own<K>(odd, t.hdt, t.qdt, v, vx, fl, fr, up);
        {
            double const nf = shift_lane<false>(fl);
            double const nu = shift_lane<false>(up);
            double w;
            double wx;
            st_join<A, FAST>(nf + fr, nu, up, Quot<FAST>(wx1, qx1.r), Quot<FAST>(wl1, ql1.r), Quot<FAST>(wl0, ql0.r), w, wx,
                             ok);
            bad = bad || !(ok || !up_even);
            u = up_even ? w : u;
            ux = up_even ? wx : ux;
        }
        if (__builtin_expect(cfl_now, 0))
        {
            if (own && up_even)
            {
                t.cfl[r] = st_cfl<K>(even, t.hdt, u);
            }
        }
    };
#pragma unroll 1
    for (int64_t it = 0; it < t.steps; it += t.group)
    {
        int64_t const end = it + t.group < t.steps ? it + t.group : t.steps;
        double const su = u;
        double const sux = ux;
        bool bad = !fixed;
        if (fixed)
        {
#pragma unroll 1
            for (int64_t k = it; k < end; ++k)
            {
                step(std::true_type{}, k, bad);
            }
        }
        if (__builtin_expect(__any(bad), 0))
        {
            u = su;
            ux = sux;
#pragma unroll 1
            for (int64_t k = it; k < end; ++k)
            {
                step(std::false_type{}, k, bad);
            }
        }
        if (end < t.steps)
        {
            if (mine)
            {
                edge[elem * 2] = u;
                edge[elem * 2 + 1] = ux;
            }
            __syncthreads();
            if (!mine)
            {
                u = edge[elem * 2];
                ux = edge[elem * 2 + 1];
            }
            __syncthreads();
        }
    }
    if (own)
    {
        if (up_even)
        {
            t.out0[r * t.out_stride] = u;
            t.out1[r * t.out_stride] = ux;
        }
        t.out0[(r + 1) * t.out_stride] = v;
        t.out1[(r + 1) * t.out_stride] = vx;
        // The outermost rows, which no march changes, go along.
        if (ghost_l || ghost_r)
        {
            int64_t const y = ghost_l ? 0 : r + 2;
            t.out0[y * t.out_stride] = t.in0[y * t.in_stride];
            t.out1[y * t.out_stride] = t.in1[y * t.in_stride];
        }
    }
}

// One element value (what: 0 xn, 1 xp, 2 tn, 3 tp, 4 so0p, 5 update_cfl,
// 6 calc_so0, 7 calc_so1_alpha) of variable iv at xindex y; store != 0 with
// what == 5 also writes cfl[y].
template <int K>
__global__ void k_st_eval(StArgs a, int what, int alpha, int64_t y, int64_t iv, int store, double * out)
{
    if (blockIdx.x != 0 || threadIdx.x != 0)
    {
        return;
    }
    StView const v{a.xc, a.so0 + iv, a.so1 + iv, a.nvar, a.hdt, a.qdt};
    double r = 0.0;
    switch (what)
    {
    case 0: r = se_xn<K>(v, y); break;
    case 1: r = se_xp<K>(v, y); break;
    case 2: r = se_t<K, 1>(v, y); break;
    case 3: r = se_t<K, -1>(v, y); break;
    case 4: r = se_so0p<K>(v, y); break;
    case 5:
        // update_cfl reads variable 0 (inviscid_burgers.hpp:104-108).
        r = se_cfl<K>(StView{a.xc, a.so0, a.so1, a.nvar, a.hdt, a.qdt}, y, a.so0[y * a.nvar]);
        if (store != 0)
        {
            a.cfl[y] = r;
        }
        break;
    case 6: r = ce_so0<K>(v, y); break;
    default:
        if (alpha == 0)
        {
            r = ce_so1<K, 0>(v, y, v.so0(y));
        }
        else if (alpha == 1)
        {
            r = ce_so1<K, 1>(v, y, v.so0(y));
        }
        else
        {
            r = ce_so1<K, 2>(v, y, v.so0(y));
        }
        break;
    }
    out[0] = r;
}

// get_so0p (core.hpp:812-824) of one plane.
template <int K>
__global__ void k_st_so0p(StArgs a, Plane p, int64_t iv, double * out)
{
    int64_t const k = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (k < p.count)
    {
        StView const v{a.xc, a.so0 + iv, a.so1 + iv, a.nvar, a.hdt, a.qdt};
        out[k] = se_so0p<K>(v, p.first + 2 * k);
    }
}

// Shortest decimal that reads back to v, the way the reference's messages
// print numbers (std::format "{}"): the shorter of the fixed and the
// scientific forms, fixed on a tie.
std::string fmt_num(double v)
{
    char fx[400];
    char sc[64];
    fx[0] = '\0';
    for (int k = 0; k <= 17; ++k)
    {
        std::snprintf(fx, sizeof(fx), "%.*f", k, v);
        if (std::strtod(fx, nullptr) == v)
        {
            break;
        }
    }
    for (int p = 0; p <= 16; ++p)
    {
        std::snprintf(sc, sizeof(sc), "%.*e", p, v);
        if (std::strtod(sc, nullptr) == v)
        {
            break;
        }
    }
    std::string const f(fx);
    std::string const e(sc);
    return (std::strtod(fx, nullptr) == v && f.size() <= e.size()) ? f : e;
}

} /* end namespace */

// Grid::init_from_array (core.cpp:48-98).
void st_grid_from(double const * xloc, int64_t n, double * xc)
{
    if (n < 2)
    {
        fail(SC_EVALUE, "Grid::init_from_array(xloc) invalid arguments: xloc.size()=" + std::to_string(n)
                            + " smaller than 2");
    }
    for (int64_t it = 0; it + 1 < n; ++it)
    {
        if (xloc[it] >= xloc[it + 1])
        {
            fail(SC_EVALUE, "Grid::init_from_array(xloc) invalid arguments: xloc[" + std::to_string(it)
                                + "]=" + fmt_num(xloc[it]) + " >= xloc[" + std::to_string(it + 1)
                                + "]=" + fmt_num(xloc[it + 1]));
        }
    }
    constexpr int64_t B = 2;
    int64_t const ncelm = n - 1;
    int64_t const nx = ncelm * 2 + (1 + B * 2);
    for (int64_t it = 0; it < n; ++it)
    {
        xc[it * 2 + B] = xloc[it];
    }
    for (int64_t it = 0; it < ncelm; ++it)
    {
        int64_t const ref = it * 2 + B + 1;
        xc[ref] = (xc[ref - 1] + xc[ref + 1]) / 2;
    }
    for (int64_t it = 1; it <= B; ++it)
    {
        xc[B - it] = xc[B] + xc[B] - xc[B + it];
        int64_t const ref = nx - B - 1;
        xc[ref + it] = xc[ref] + xc[ref] - xc[ref - it];
    }
}

// Grid::Grid(xmin, xmax, ncelm) (core.cpp:14-45).
void st_grid(double xmin, double xmax, int64_t ncelm, double * xc)
{
    std::string const head = "Grid::Grid(xmin=" + fmt_num(xmin) + ", xmax=" + fmt_num(xmax)
                             + ", ncelm=" + std::to_string(ncelm) + ")";
    if (ncelm < 1)
    {
        fail(SC_EVALUE, head + " invalid argument: ncelm smaller than 1");
    }
    if (xmin >= xmax)
    {
        fail(SC_EVALUE, head + " invalid arguments: xmin >= xmax");
    }
    double const xspace = (xmax - xmin) / static_cast<double>(ncelm);
    std::vector<double> xloc(static_cast<size_t>(ncelm + 1));
    xloc[0] = xmin;
    for (int64_t it = 1; it < ncelm; ++it)
    {
        xloc[it] = xloc[it - 1] + xspace;
    }
    xloc[ncelm] = xmax;
    st_grid_from(xloc.data(), ncelm + 1, xc);
}

struct StCore
{
    int kind = K_LINEAR;
    int64_t nx = 0;
    int64_t ncelm = 0;
    int64_t nvar = 1;
    double dt = 0.0;
    StreamHolder sh; // declared before the buffers: freed last
    hipStream_t stream = sh.s;
    DevBuf<double> xc, so0, so1, cfl;
    DevBuf<double> t0, t1; // variable 0 between the launches of the tiled march

    StCore(int k, int64_t n, int64_t nv, double time_increment)
        : kind(k)
        , nx(n)
        , ncelm((n - 5) / 2)
        , nvar(nv)
        , dt(time_increment)
    {
        AllocScope const scope(stream);
        xc.alloc(nx);
        so0.alloc(nx * nvar);
        so1.alloc(nx * nvar);
        cfl.alloc(nx);
        SC_HIP(hipMemsetAsync(xc.ptr, 0, xc.bytes(), stream));
        SC_HIP(hipMemsetAsync(so0.ptr, 0, so0.bytes(), stream));
        SC_HIP(hipMemsetAsync(so1.ptr, 0, so1.bytes(), stream));
        SC_HIP(hipMemsetAsync(cfl.ptr, 0, cfl.bytes(), stream));
    }

    ~StCore() = default;

    void sync() { SC_HIP(hipStreamSynchronize(stream)); }

    DevBuf<double> & buf(int which)
    {
        switch (which)
        {
        case 0: return xc;
        case 1: return so0;
        case 2: return so1;
        case 3: return cfl;
        default: fail(SC_EVALUE, "spacetime solver: unknown array id");
        }
    }

    // Field::set_time_increment (core.cpp:109-114).
    StArgs args() const { return StArgs{ncelm, nvar, 0.5 * dt, 0.25 * dt, xc.ptr, so0.ptr, so1.ptr, cfl.ptr}; }

    template <int K>
    void so0_pass(bool odd)
    {
        Plane const p = ce_plane(ncelm, odd);
        k_st_so0<K><<<grid_for(p.count, ST_BLOCK), ST_BLOCK, 0, stream>>>(args(), p);
        SC_HIP(hipGetLastError());
    }

    template <int K, int A>
    void so1_pass(bool odd)
    {
        Plane const p = ce_plane(ncelm, odd);
        k_st_so1<K, A><<<grid_for(p.count, ST_BLOCK), ST_BLOCK, 0, stream>>>(args(), p);
        SC_HIP(hipGetLastError());
    }

    template <int K>
    void cfl_pass(bool odd)
    {
        Plane const p = se_plane(ncelm, odd);
        k_st_cfl<K><<<grid_for(p.count, ST_BLOCK), ST_BLOCK, 0, stream>>>(args(), p);
        SC_HIP(hipGetLastError());
    }

    void bnd(double * arr)
    {
        k_st_bnd<<<1, 64, 0, stream>>>(ncelm, nvar, arr);
        SC_HIP(hipGetLastError());
    }

    template <int K, int A>
    void half(bool odd)
    {
        int64_t const count = odd ? ncelm + 1 : ncelm;
        k_st_half<K, A><<<grid_for(count, ST_BLOCK), ST_BLOCK, 0, stream>>>(args(), odd ? 1 : 0);
        SC_HIP(hipGetLastError());
    }

    template <int K, int A>
    void march_k(int64_t steps)
    {
        if (steps <= 0)
        {
            return;
        }
        // Launches of at most 64 steps, 24 where the blocks fill the chip and
        // the elements computed twice count, and on a ring of a few elements,
        // which is nearly all seam and needs a wide halo.  A ring that one
        // block owns is marched in place.  Others march between two pairs of
        // arrays, which change places after an odd number of launches; a state
        // of several variables, of which the other pair holds the first alone,
        // takes an even number, and for a single step the half-step kernels.
        // Per call of one and of two steps: 10 elements 13.8 and 14.7 us in
        // place, 14.8 and 17.0 by half steps and an even number; 250 elements
        // 14.9 and 15.1 in one launch, 15.7 and 17.6.
        int64_t const ring = ncelm + 2;
        int64_t const most = ring <= 32 || ring > 20000 ? 24 : 64;
        bool const alone = ring <= ST_ELEMS - 2 * st_halo(steps < most ? steps : most, ring);
        bool const swaps = !alone && nvar == 1;
        if (steps == 1 && !alone && !swaps)
        {
            half<K, A>(false);
            half<K, A>(true);
            return;
        }
        if (!alone && t0.ptr == nullptr)
        {
            AllocScope const scope(stream);
            t0.alloc(nx);
            t1.alloc(nx);
        }
        int64_t const launches = alone || swaps ? (steps + most - 1) / most : 2 * ((steps + 2 * most - 1) / (2 * most));
        for (int64_t k = 0; k < launches; ++k)
        {
            int64_t const n = steps * (k + 1) / launches - steps * k / launches;
            StTile t{};
            t.ncelm = ncelm;
            t.steps = n;
            t.group = ring > ST_OVER ? GROUP : 1;
            t.halo = st_halo(n, ring);
            t.seg = ST_ELEMS - 2 * t.halo;
            t.last = k + 1 == launches ? 1 : 0;
            t.hdt = 0.5 * dt;
            t.qdt = 0.25 * dt;
            t.xc = xc.ptr;
            bool const from = !alone && k % 2 != 0; // reads the other pair
            bool const to = !alone && k % 2 == 0;   // writes the other pair
            t.in0 = from ? t0.ptr : so0.ptr;
            t.in1 = from ? t1.ptr : so1.ptr;
            t.in_stride = from ? 1 : nvar;
            t.out0 = to ? t0.ptr : so0.ptr;
            t.out1 = to ? t1.ptr : so1.ptr;
            t.out_stride = to ? 1 : nvar;
            t.cfl = cfl.ptr;
            k_st_tiled<K, A><<<grid_for(ring, static_cast<unsigned>(t.seg)), TBLOCK, 0, stream>>>(t);
            SC_HIP(hipGetLastError());
        }
        if (swaps && launches % 2 != 0)
        {
            std::swap(so0, t0);
            std::swap(so1, t1);
        }
    }

    template <int K>
    void stage_k(int stage, int alpha, bool odd)
    {
        switch (stage)
        {
        case 0: so0_pass<K>(odd); break;
        case 1:
            if (alpha == 0)
            {
                so1_pass<K, 0>(odd);
            }
            else if (alpha == 1)
            {
                so1_pass<K, 1>(odd);
            }
            else
            {
                so1_pass<K, 2>(odd);
            }
            break;
        case 2: cfl_pass<K>(odd); break;
        case 3: bnd(so0.ptr); break;
        case 4: bnd(so1.ptr); break;
        case 5:
        case 6:
            if (alpha == 0)
            {
                half<K, 0>(stage == 6);
            }
            else if (alpha == 1)
            {
                half<K, 1>(stage == 6);
            }
            else
            {
                half<K, 2>(stage == 6);
            }
            break;
        default: fail(SC_EVALUE, "spacetime solver: unknown stage");
        }
    }

    void stage(int st, int alpha, bool odd)
    {
        switch (kind)
        {
        case K_DEFAULT: stage_k<K_DEFAULT>(st, alpha, odd); break;
        case K_LINEAR: stage_k<K_LINEAR>(st, alpha, odd); break;
        default: stage_k<K_BURGERS>(st, alpha, odd); break;
        }
    }

    template <int K>
    void march_a(int alpha, int64_t steps)
    {
        if (alpha == 0)
        {
            march_k<K, 0>(steps);
        }
        else if (alpha == 1)
        {
            march_k<K, 1>(steps);
        }
        else
        {
            march_k<K, 2>(steps);
        }
    }

    void march(int alpha, int64_t steps)
    {
        switch (kind)
        {
        case K_DEFAULT: march_a<K_DEFAULT>(alpha, steps); break;
        case K_LINEAR: march_a<K_LINEAR>(alpha, steps); break;
        default: march_a<K_BURGERS>(alpha, steps); break;
        }
    }

    double eval(int what, int alpha, int64_t y, int64_t iv, int store)
    {
        DevBuf<double> out;
        out.alloc(1);
        switch (kind)
        {
        case K_DEFAULT:
            k_st_eval<K_DEFAULT><<<1, 64, 0, stream>>>(args(), what, alpha, y, iv, store, out.ptr);
            break;
        case K_LINEAR:
            k_st_eval<K_LINEAR><<<1, 64, 0, stream>>>(args(), what, alpha, y, iv, store, out.ptr);
            break;
        default: k_st_eval<K_BURGERS><<<1, 64, 0, stream>>>(args(), what, alpha, y, iv, store, out.ptr); break;
        }
        SC_HIP(hipGetLastError());
        double r = 0.0;
        SC_HIP(hipMemcpyAsync(&r, out.ptr, sizeof(double), hipMemcpyDeviceToHost, stream));
        sync();
        return r;
    }

    void so0p(int64_t iv, bool odd, double * host, int64_t n)
    {
        // get_so0p walks the nselm - odd solution elements from index 0.
        Plane const r{odd ? 3 : 2, ncelm + 1 - (odd ? 1 : 0)};
        if (n != r.count)
        {
            fail(SC_EVALUE, "get_so0p: output size mismatch");
        }
        DevBuf<double> out;
        out.alloc(r.count);
        switch (kind)
        {
        case K_DEFAULT:
            k_st_so0p<K_DEFAULT><<<grid_for(r.count, ST_BLOCK), ST_BLOCK, 0, stream>>>(args(), r, iv, out.ptr);
            break;
        case K_LINEAR:
            k_st_so0p<K_LINEAR><<<grid_for(r.count, ST_BLOCK), ST_BLOCK, 0, stream>>>(args(), r, iv, out.ptr);
            break;
        default:
            k_st_so0p<K_BURGERS><<<grid_for(r.count, ST_BLOCK), ST_BLOCK, 0, stream>>>(args(), r, iv, out.ptr);
            break;
        }
        SC_HIP(hipGetLastError());
        SC_HIP(hipMemcpyAsync(host, out.ptr, out.bytes(), hipMemcpyDeviceToHost, stream));
        sync();
    }
};

} /* end namespace scamd */

using scamd::guard;
using scamd::StCore;

extern "C"
{

int scst_grid(double xmin, double xmax, int64_t ncelm, double * xc, int64_t nx)
{
    return guard(
        [&]()
        {
            if (ncelm >= 1 && nx != 2 * ncelm + 5)
            {
                scamd::fail(scamd::SC_EVALUE, "Grid: coordinate buffer size mismatch");
            }
            scamd::st_grid(xmin, xmax, ncelm, xc);
        });
}

int scst_grid_from(double const * xloc, int64_t n, double * xc, int64_t nx)
{
    return guard(
        [&]()
        {
            if (n >= 2 && nx != 2 * (n - 1) + 5)
            {
                scamd::fail(scamd::SC_EVALUE, "Grid: coordinate buffer size mismatch");
            }
            scamd::st_grid_from(xloc, n, xc);
        });
}

int scst_create(int kind, double const * xc, int64_t nx, int64_t nvar, double time_increment, void ** out)
{
    return guard(
        [&]()
        {
            if (kind < 0 || kind > 2)
            {
                scamd::fail(scamd::SC_EVALUE, "spacetime solver: unknown kernel kind");
            }
            if (nx < 7 || (nx - 5) % 2 != 0)
            {
                scamd::fail(scamd::SC_EVALUE, "spacetime solver: coordinate count must be 2*ncelm+5 with ncelm >= 1");
            }
            if (nvar < 1)
            {
                scamd::fail(scamd::SC_EVALUE, "spacetime solver: nvar must be at least 1");
            }
            auto * h = new StCore(kind, nx, nvar, time_increment);
            SC_HIP(hipMemcpyAsync(h->xc.ptr, xc, h->xc.bytes(), hipMemcpyHostToDevice, h->stream));
            h->sync();
            *out = h;
        });
}

int scst_clone(void * h, void ** out)
{
    return guard(
        [&]()
        {
            auto & a = *static_cast<StCore *>(h);
            scamd::AllocScope const alloc_scope_(a.stream);
            auto * b = new StCore(a.kind, a.nx, a.nvar, a.dt);
            for (int w = 0; w < 4; ++w)
            {
                SC_HIP(hipMemcpyAsync(b->buf(w).ptr, a.buf(w).ptr, a.buf(w).bytes(), hipMemcpyDeviceToDevice,
                                      a.stream));
            }
            a.sync();
            b->sync();
            *out = b;
        });
}

void scst_destroy(void * h) { delete static_cast<StCore *>(h); }

int scst_set_time_increment(void * h, double time_increment)
{
    static_cast<StCore *>(h)->dt = time_increment;
    return 0;
}

int scst_upload(void * h, int which, double const * host, int64_t count)
{
    return guard(
        [&]()
        {
            auto & a = *static_cast<StCore *>(h);
            scamd::AllocScope const alloc_scope_(a.stream);
            auto & b = a.buf(which);
            if (count != b.count)
            {
                scamd::fail(scamd::SC_EVALUE, "spacetime solver: array size mismatch");
            }
            scamd::copy_up(b.ptr, host, b.bytes(), a.stream);
        });
}

int scst_download(void * h, int which, double * host, int64_t count)
{
    return guard(
        [&]()
        {
            auto & a = *static_cast<StCore *>(h);
            scamd::AllocScope const alloc_scope_(a.stream);
            auto & b = a.buf(which);
            if (count != b.count)
            {
                scamd::fail(scamd::SC_EVALUE, "spacetime solver: array size mismatch");
            }
            scamd::copy_down(host, b.ptr, b.bytes(), a.stream);
        });
}

int scst_stage(void * h, int stage, int alpha, int odd_plane)
{
    return guard(
        [&]()
        {
            if (alpha < 0 || alpha > 2)
            {
                scamd::fail(scamd::SC_EVALUE, "alpha must be 0, 1 or 2");
            }
            auto & a = *static_cast<StCore *>(h);
            scamd::AllocScope const alloc_scope_(a.stream);
            a.stage(stage, alpha, odd_plane != 0);
            a.sync();
        });
}

int scst_march(void * h, int alpha, int64_t steps)
{
    return guard(
        [&]()
        {
            if (alpha < 0 || alpha > 2)
            {
                scamd::fail(scamd::SC_EVALUE, "alpha must be 0, 1 or 2");
            }
            auto & a = *static_cast<StCore *>(h);
            scamd::AllocScope const alloc_scope_(a.stream);
            a.march(alpha, steps);
            a.sync();
        });
}

int scst_march_async(void * h, int alpha, int64_t steps)
{
    return guard(
        [&]()
        {
            if (alpha < 0 || alpha > 2)
            {
                scamd::fail(scamd::SC_EVALUE, "alpha must be 0, 1 or 2");
            }
            static_cast<StCore *>(h)->march(alpha, steps);
        });
}

int scst_sync(void * h)
{
    return guard([&]() { static_cast<StCore *>(h)->sync(); });
}

int scst_eval(void * h, int what, int alpha, int64_t xindex, int64_t iv, int store, double * out)
{
    return guard(
        [&]()
        {
            auto & a = *static_cast<StCore *>(h);
            scamd::AllocScope const alloc_scope_(a.stream);
            if (what < 0 || what > 7)
            {
                scamd::fail(scamd::SC_EVALUE, "spacetime solver: unknown element value");
            }
            if (iv < 0 || iv >= a.nvar)
            {
                scamd::fail(scamd::SC_EINDEX, "out of nvar range");
            }
            int64_t const lo = what >= 6 ? 2 : 1;
            if (xindex < lo || xindex >= a.nx - lo)
            {
                scamd::fail(scamd::SC_EINDEX, "spacetime solver: element index out of range");
            }
            *out = a.eval(what, alpha, xindex, iv, store);
        });
}

int scst_so0p(void * h, int64_t iv, int odd_plane, double * host_out, int64_t n)
{
    return guard(
        [&]()
        {
            auto & a = *static_cast<StCore *>(h);
            scamd::AllocScope const alloc_scope_(a.stream);
            if (iv < 0 || iv >= a.nvar)
            {
                scamd::fail(scamd::SC_EINDEX, "get_so0p(): out of nvar range");
            }
            a.so0p(iv, odd_plane != 0, host_out, n);
        });
}

} /* end extern "C" */
