/*
 * The face-lane form of the fused substep (calc_soln, bc_soln / bc_dsoln,
 * calc_cfl, calc_dsoln; euler_march.cpp:219-302, euler_bc.cpp:143-320,
 * euler_solution.cpp:114-159, euler_gradient.cpp:23-130): LANES lanes of a
 * wavefront work on one cell, lane f on its face f and on its fundamental
 * gradient element f, where k_cell of euler.hip gives a cell one lane.
 *
 * A cell's work is a chain of about 2500 (triangle) to 13000 (hexahedron)
 * instructions in k_cell, and its straight-line code is as long.  Here the
 * faces run side by side: the chain and the code are three to four times
 * shorter, a lane holds one neighbour's row instead of re-reading all of
 * them, and the registers allow more wavefronts per SIMD.
 *
 * Every sum keeps the reference's order.  Sums over faces, sub-faces
 * and gradient elements go through a few LDS words per cell.  Lanes beyond a cell's faces (or elements) repeat its
 * last one, so they store the same values and need no masks.
 *
 * The lanes repeat what belongs to the cell and not to a face: 1.5 (tetrahedra)
 * to 2 times (triangles) the instructions per cell of k_cell, the VALU 60%
 * busy on large meshes.  So it runs where the chip is not full (lane_cells):
 * the 8100-cell mixed block takes 12 us per substep against 159 with a kernel
 * pair per type, 18432 triangles 9.2 against 13.  Registers (200 in 2D, 250 in
 * 3D) allow two wavefronts per SIMD; compiled for three it spills and takes
 * 1.3 times as long.
 *
 * A wavefront runs the fast form (FastChk) and, when one of its cells
 * reports a value outside the range where that is exact, the exact form
 * over the same cells: one launch, no second kernel.  The later launches of
 * that march run the exact form alone, as k_cell's pairs do: a state that has
 * blown up then takes 11 us per substep on 18432 triangles and 59 on 110000
 * tetrahedra (26 and 131 with both forms tried in every launch, most of it the
 * atomics that count the passes).
 */

#include "euler_march.hpp"

#include <algorithm>

namespace scamd
{
namespace
{

template <int T>
constexpr int lanes_of()
{
    return Traits<T>::NF <= 4 ? 4 : 8;
}

template <int T>
constexpr int sub_max()
{
    return T == CT_TRI || T == CT_QUAD ? 2 : T == CT_TET ? 3 : 4;
}

// LDS words (doubles) per cell: the larger of the flux terms of
// every sub-face and the weighted gradients of every element; odd, so the
// cells of a wavefront start in different banks.
template <int T>
constexpr int lane_words()
{
    using TR = Traits<T>;
    int const a = TR::NFGE * (TR::ND + 2) * TR::ND;
    int const b = TR::NF * (1 + sub_max<T>()) * (TR::ND + 2);
    int const w = a > b ? a : b;
    return w % 2 == 0 ? w + 1 : w;
}

// Between LDS writes and reads of other lanes of the same wavefront.  The
// LDS operations of a wavefront complete in order; this keeps the compiler
// from moving them across.
__device__ inline void wave_lds()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// The v-th face (0-based) of gradient element e, e a lane's own: a table of
// 4-bit entries.
template <int T, int V>
__device__ inline int span_face(int e)
{
    constexpr auto table = []() constexpr {
        unsigned long long t = 0;
        for (int k = 0; k < Traits<T>::NFGE; ++k)
        {
            t |= static_cast<unsigned long long>(Traits<T>::fge(k, V) - 1) << (4 * k);
        }
        return t;
    };
    constexpr unsigned long long t = table();
    return static_cast<int>((static_cast<unsigned>(t) >> (4 * e)) & 15u);
}

// Hides the Jacobian's scalars from loop-invariant code motion, which would
// hoist every entry of every row out of the sub-face loop into registers,
// and forms the simple ones again.
template <bool FAST>
__device__ inline void renew(JacS<2, FAST> & j)
{
    asm volatile("" : "+v"(j.ga), "+v"(j.u2), "+v"(j.u3), "+v"(j.u4), "+v"(j.v1), "+v"(j.v2), "+v"(j.vs), "+v"(j.getot), "+v"(j.pr));
    j.ga1 = j.ga - 1;
    j.ga3 = j.ga - 3;
    j.ga1h = j.ga1 / 2;
    j.v1o2 = j.v1 * j.v1;
    j.v2o2 = j.v2 * j.v2;
}

template <bool FAST>
__device__ inline void renew(JacS<3, FAST> & j)
{
    asm volatile("" : "+v"(j.ga), "+v"(j.u2), "+v"(j.u3), "+v"(j.u4), "+v"(j.u5), "+v"(j.v1), "+v"(j.v2), "+v"(j.v3), "+v"(j.vs), "+v"(j.getot), "+v"(j.pr));
    j.ga1 = j.ga - 1;
    j.ga3 = j.ga - 3;
    j.ga1h = j.ga1 / 2;
    j.v1o2 = j.v1 * j.v1;
    j.v2o2 = j.v2 * j.v2;
    j.v3o2 = j.v3 * j.v3;
}

// One cell per group of lanes; l is the lane in the group, xs the group's
// LDS words.  Returns false (in any lane of the group) when the fast form
// may differ from the exact one, or is not wanted (only).
template <int T, int MODE, bool FAST>
__device__ inline bool lane_cell(KP const & p, GV const & g, int64_t i, int l, double * xs, bool only)
{
    using TR = Traits<T>;
    using LY = Layout<T>;
    constexpr int ND = TR::ND;
    constexpr int NF = TR::NF;
    constexpr int NEQ = ND + 2;
    constexpr int NFGE = TR::NFGE;
    constexpr int NS = sub_max<T>();
    constexpr int L = lanes_of<T>();
    int const f = l < NF ? l : NF - 1;
    int const e = l < NFGE ? l : NFGE - 1;
    FastChk chk;
    auto recip = [&](double d) -> double
    {
        if constexpr (FAST)
        {
            chk.den(d);
            return div_recip(d);
        }
        return 0.0;
    };
    auto quot = [&](double a, double d, double r) -> double
    {
        if constexpr (FAST)
        {
            return div_fast(a, d, r, chk);
        }
        return a / d;
    };

    int64_t const n = g.n;
    int64_t const row = p.G + g.off + i;
    double const * geo = g.geo + i;
    double const hdt = p.hdt;
    double const qdt = p.qdt;

    // Where the exact-only switch is looked at: in 3D before the loads, in 2D
    // when they have come, where its own load hides behind them.  There it
    // costs a normal 2D substep 0.02 to 0.1 us (before the loads 0.25 to 0.45
    // of 7 to 9 us), but one that has blown up 1 us; in 3D, where the flux
    // terms weigh more, 7 us of 59 for 110000 tetrahedra.
    if constexpr (FAST && ND == 3)
    {
        if (__builtin_expect(only, 0))
        {
            return false;
        }
    }
    // This face's neighbour row and geometry.
    int64_t const j = __builtin_nontemporal_load(g.nbr + f * n + i);
    double js[NEQ];
    double j1[NEQ][ND];
    double cj[ND];
    double bc[ND];
#pragma unroll
    for (int k = 0; k < NEQ; ++k)
    {
        js[k] = p.s0c[j * NEQ + k];
    }
#pragma unroll
    for (int k = 0; k < NEQ; ++k)
    {
#pragma unroll
        for (int d = 0; d < ND; ++d)
        {
            j1[k][d] = p.s1c[j * (NEQ * ND) + k * ND + d];
        }
    }
    double const jgam = p.gam[j];
#pragma unroll
    for (int d = 0; d < ND; ++d)
    {
        cj[d] = p.cen[j * ND + d];
        bc[d] = __builtin_nontemporal_load(geo + (LY::FB + f * ND + d) * n);
    }
    double const bvol = __builtin_nontemporal_load(geo + (LY::FV + 1 + f) * n);
    int const nsub = TR::nsub(f);
    double const * gc = geo + (LY::FC + TR::soff(f) * ND) * n;
    double const * gn = geo + (LY::FN + TR::soff(f) * ND) * n;
    double sc[ND];
    double sn[ND];
#pragma unroll
    for (int d = 0; d < ND; ++d)
    {
        sc[d] = __builtin_nontemporal_load(gc + d * n);
        sn[d] = __builtin_nontemporal_load(gn + d * n);
    }

    // This face's terms of the flux integral, in LDS: the neighbour's CE, then
    // the flux through each sub-face.  The sub-face loop stays a loop: its
    // Jacobian rows are formed again in each pass, which costs less than the
    // registers and the code of holding every sub-face's solution.
#pragma unroll
    for (int k = 0; k < NEQ; ++k)
    {
        double fusp = js[k];
#pragma unroll
        for (int d = 0; d < ND; ++d)
        {
            fusp += (bc[d] - cj[d]) * j1[k][d];
        }
        xs[f * (1 + NS) * NEQ + k] = fusp * bvol;
    }
    if constexpr (FAST && ND == 2)
    {
        if (__builtin_expect(only, 0))
        {
            return false;
        }
    }
    JacS<ND, FAST> jac;
    jac.set(jgam, js, &chk);
    double st[NEQ];
    solt_of<ND>(jac, j1, st);
    double e0[ND]; // the energy row's density column, which divides
    {
        double jr[NEQ][ND];
        double fr[ND];
        jac.template row<NEQ - 1>(jr, fr);
#pragma unroll
        for (int d = 0; d < ND; ++d)
        {
            e0[d] = jr[0][d];
        }
    }
    FastChk unused;
    jac.chk = &unused;
#pragma unroll 1
    for (int s = 0; s < NS; ++s)
    {
        // The next sub-face's geometry is loaded a pass ahead.
        int const nx = s + 1 < nsub ? s + 1 : nsub - 1;
        double scn[ND];
        double snn[ND];
#pragma unroll
        for (int d = 0; d < ND; ++d)
        {
            scn[d] = __builtin_nontemporal_load(gc + (nx * ND + d) * n);
            snn[d] = __builtin_nontemporal_load(gn + (nx * ND + d) * n);
        }
        double us[NEQ];
#pragma unroll
        for (int k = 0; k < NEQ; ++k)
        {
            us[k] = qdt * st[k];
#pragma unroll
            for (int d = 0; d < ND; ++d)
            {
                us[k] += (sc[d] - cj[d]) * j1[k][d];
            }
        }
        double * const xf = xs + (f * (1 + NS) + 1 + s) * NEQ;
        renew(jac);
        static_for<0, NEQ>([&](auto kc) {
            constexpr int k = decltype(kc)::value;
            double jr[NEQ][ND];
            double fr[ND];
            jac.template row<k>(jr, fr);
            if constexpr (k == NEQ - 1)
            {
#pragma unroll
                for (int d = 0; d < ND; ++d)
                {
                    jr[0][d] = e0[d];
                }
            }
            double dot = 0.0;
#pragma unroll
            for (int d2 = 0; d2 < ND; ++d2)
            {
                double dfcn = fr[d2];
#pragma unroll
                for (int m = 0; m < NEQ; ++m)
                {
                    if (!FAST || !jac_zero(ND, k, m, d2))
                    {
                        dfcn += jr[m][d2] * us[m];
                    }
                }
                dot += dfcn * sn[d2];
            }
            xf[k] = s < nsub ? hdt * dot : 0.0;
        });
#pragma unroll
        for (int d = 0; d < ND; ++d)
        {
            sc[d] = scn[d];
            sn[d] = snn[d];
        }
    }
    wave_lds();
    // Lane k adds the terms of equation k, face by face, and the cell's lanes
    // share the sums.
    double const cvol = __builtin_nontemporal_load(geo + LY::FV * n);
    double const rcv = recip(cvol);
    double u0[NEQ];
    constexpr int NP = (NEQ + L - 1) / L; // passes
    double un[NP];
#pragma unroll
    for (int q = 0; q < NP; ++q)
    {
        int const k = l + q * L < NEQ ? l + q * L : NEQ - 1;
        double acc = 0.0;
#pragma unroll
        for (int t = 0; t < NF * (1 + NS); ++t)
        {
            double const x = xs[t * NEQ + k];
            acc = t % (1 + NS) == 0 ? acc + x : acc - x;
        }
        un[q] = quot(acc, cvol, rcv);
    }
    wave_lds();
#pragma unroll
    for (int q = 0; q < NP; ++q)
    {
        xs[l + q * L < NEQ ? l + q * L : NEQ - 1] = un[q];
    }
    wave_lds();
#pragma unroll
    for (int k = 0; k < NEQ; ++k)
    {
        u0[k] = xs[k];
    }
    wave_lds();

    // calc_cfl, in every lane of the cell.
    double const dist = __builtin_nontemporal_load(geo + LY::FD * n);
    double const ga = p.gam[row];
    double const ga1 = ga - 1.0;
    double momsq = 0.0;
#pragma unroll
    for (int d = 0; d < ND; ++d)
    {
        momsq += u0[1 + d] * u0[1 + d];
    }
    double const ke = momsq / (2.0 * u0[0]);
    double const pr = ga1 * (u0[NEQ - 1] - ke);
    double const pra = (pr + fabs(pr)) / 2.0;
    double const wspd = sqrt(ga * pra / u0[0]) + sqrt(momsq) / u0[0];
    double const co = hdt * wspd / dist;
    double const cflc = (co - 1.0) * pra / (pra + TINYJ) + 1.0;
    double const epre = u0[NEQ - 1];
    u0[NEQ - 1] = pra / ga1 + ke + TINYJ;
    if (l == 0)
    {
        __builtin_nontemporal_store(co, p.cflo + row);
        __builtin_nontemporal_store(cflc, p.cflc + row);
#pragma unroll
        for (int k = 0; k < NEQ; ++k)
        {
            __builtin_nontemporal_store(u0[k], p.s0n + row * NEQ + k);
        }
    }
    if constexpr (FAST)
    {
#pragma unroll
        for (int k = 0; k < NEQ; ++k)
        {
            chk.finite(u0[k]);
        }
    }

    // calc_dsoln: the gradient element's points, its centroid, the
    // displacements and the solution differences.
    double const acfl = fabs(cflc);
    double const sgm0 = p.sigma0 / acfl;
    double const tau = p.taumin + acfl * p.tauscale;
    double ice[ND];
    double gp[ND];
#pragma unroll
    for (int d = 0; d < ND; ++d)
    {
        ice[d] = p.cen[row * ND + d];
        gp[d] = bc[d] + tau * (cj[d] - bc[d]);
        xs[f * ND + d] = gp[d];
    }
    wave_lds();
    double avg[ND];
#pragma unroll
    for (int d = 0; d < ND; ++d)
    {
        avg[d] = 0.0;
#pragma unroll
        for (int q = 0; q < NF; ++q)
        {
            avg[d] += xs[q * ND + d];
        }
        avg[d] /= NF;
    }
    int sp[ND];
    sp[0] = span_face<T, 0>(e);
    sp[1] = span_face<T, 1>(e);
    if constexpr (ND == 3)
    {
        sp[2] = span_face<T, 2>(e);
    }
    double sub[ND];
    double dst[ND][ND];
#pragma unroll
    for (int d = 0; d < ND; ++d)
    {
        sub[d] = avg[d];
    }
#pragma unroll
    for (int v = 0; v < ND; ++v)
    {
#pragma unroll
        for (int d = 0; d < ND; ++d)
        {
            double const x = xs[sp[v] * ND + d];
            sub[d] += x;
            dst[v][d] = x - avg[d];
        }
    }
    double const vob = ge_det<ND>(dst);
    wave_lds();
    xs[e * (ND + 1)] = vob;
#pragma unroll
    for (int d = 0; d < ND; ++d)
    {
        xs[e * (ND + 1) + 1 + d] = sub[d] / static_cast<double>(ND + 1) * vob;
    }
    wave_lds();
    double voc = 0.0;
    double cnd[ND];
#pragma unroll
    for (int d = 0; d < ND; ++d)
    {
        cnd[d] = 0.0;
    }
#pragma unroll
    for (int q = 0; q < NFGE; ++q)
    {
        voc += xs[q * (ND + 1)];
#pragma unroll
        for (int d = 0; d < ND; ++d)
        {
            cnd[d] += xs[q * (ND + 1) + 1 + d];
        }
    }
    double const rvoc = recip(voc);
    double jdis[ND];
    wave_lds();
#pragma unroll
    for (int d = 0; d < ND; ++d)
    {
        cnd[d] = quot(cnd[d], voc, rvoc);
        xs[f * (ND + NEQ) + d] = gp[d] - cnd[d];
        jdis[d] = (gp[d] - cj[d]) + ice[d] - cnd[d];
    }
#pragma unroll
    for (int k = 0; k < NEQ; ++k)
    {
        double val = js[k] + hdt * st[k] - u0[k];
#pragma unroll
        for (int d = 0; d < ND; ++d)
        {
            val += jdis[d] * j1[k][d];
        }
        xs[f * (ND + NEQ) + ND + k] = val;
    }
    wave_lds();
    double ud[ND][NEQ];
#pragma unroll
    for (int v = 0; v < ND; ++v)
    {
#pragma unroll
        for (int d = 0; d < ND; ++d)
        {
            dst[v][d] = xs[sp[v] * (ND + NEQ) + d];
        }
#pragma unroll
        for (int k = 0; k < NEQ; ++k)
        {
            ud[v][k] = xs[sp[v] * (ND + NEQ) + ND + k];
        }
    }
    double adj[ND][ND];
    ge_adj<ND>(dst, adj);
    double const det = ge_det<ND>(dst);
    double const rdet = recip(det);
    double gk[NEQ][ND];
    wave_lds();
#pragma unroll
    for (int k = 0; k < NEQ; ++k)
    {
        double sq = 0.0;
#pragma unroll
        for (int a = 0; a < ND; ++a)
        {
            double r = 0.0;
#pragma unroll
            for (int b = 0; b < ND; ++b)
            {
                r += adj[a][b] * ud[b][k];
            }
            gk[k][a] = quot(r, det, rdet);
        }
#pragma unroll
        for (int d = 0; d < ND; ++d)
        {
            sq += gk[k][d] * gk[k][d];
        }
        xs[e * NEQ + k] = 1.0 / sqrt(sq + ALMOST_ZERO);
    }
    wave_lds();
    // Lane k weights the elements of equation k: the quotients by the sum and
    // the limiter once per equation instead of in every lane.
    constexpr double ofg1 = 1.0 / NFGE;
#pragma unroll
    for (int q = 0; q < NP; ++q)
    {
        int const k = l + q * L < NEQ ? l + q * L : NEQ - 1;
        double w[NFGE];
        double wacc = 0.0;
#pragma unroll
        for (int t = 0; t < NFGE; ++t)
        {
            w[t] = xs[t * NEQ + k];
            wacc += w[t];
        }
        double rwa = 0.0;
        if constexpr (FAST)
        {
            rwa = div_recip(wacc); // no scaling acts in these quotients (see k_cell)
        }
        double wmax = 0.0;
        double wmin = 0.0;
#pragma unroll
        for (int t = 0; t < NFGE; ++t)
        {
            double x;
            if constexpr (FAST)
            {
                x = w[t] * rwa;
                double const rem = __builtin_fma(-wacc, x, w[t]);
                x = __builtin_fma(rem, rwa, x);
            }
            else
            {
                x = w[t] / wacc;
            }
            x -= ofg1;
            w[t] = x;
            wmax = fmax(wmax, x);
            wmin = fmin(wmin, x);
        }
        double const sm = fmin((1.0 - ofg1) / (wmax + ALMOST_ZERO), -ofg1 / (wmin - ALMOST_ZERO));
        double const smax = fmin(sm, sgm0);
        wave_lds();
#pragma unroll
        for (int t = 0; t < NFGE; ++t)
        {
            xs[t * NEQ + k] = ofg1 + smax * w[t];
        }
    }
    wave_lds();
    double wk[NEQ];
#pragma unroll
    for (int k = 0; k < NEQ; ++k)
    {
        wk[k] = xs[e * NEQ + k];
    }
    wave_lds();
#pragma unroll
    for (int k = 0; k < NEQ; ++k)
    {
#pragma unroll
        for (int d = 0; d < ND; ++d)
        {
            xs[(e * NEQ + k) * ND + d] = wk[k] * gk[k][d];
        }
    }
    wave_lds();
#pragma unroll
    for (int o = 0; o < NEQ * ND; o += L)
    {
        int const c = o + l < NEQ * ND ? o + l : NEQ * ND - 1;
        double out = 0.0;
#pragma unroll
        for (int q = 0; q < NFGE; ++q)
        {
            out += xs[q * (NEQ * ND) + c];
        }
        p.s1n[row * (NEQ * ND) + c] = out;
        if constexpr (FAST)
        {
            chk.finite(out);
        }
        if constexpr ((MODE & M_STNEXT) != 0)
        {
            wave_lds();
            xs[c] = out; // element 0's words, read by this lane only
            wave_lds();
        }
    }
    if constexpr ((MODE & M_STNEXT) != 0)
    {
        // so0t of this row for the level being written.
        double s1w[NEQ][ND];
#pragma unroll
        for (int k = 0; k < NEQ; ++k)
        {
#pragma unroll
            for (int d = 0; d < ND; ++d)
            {
                s1w[k][d] = xs[k * ND + d];
            }
        }
        JacS<ND, FAST> rj;
        rj.set(ga, u0, &chk);
        double rst[NEQ];
        solt_of<ND>(rj, s1w, rst);
        if constexpr (FAST)
        {
            chk.finite(rst[NEQ - 1]);
        }
        if (l == 0)
        {
#pragma unroll
            for (int k = 0; k < NEQ; ++k)
            {
                __builtin_nontemporal_store(rst[k], p.stn + row * NEQ + k);
            }
        }
    }
    // bc_soln (from the pre-CFL state) and bc_dsoln (from so1c) of this lane's
    // face when it is a boundary face; last, when few values are live.
    u0[NEQ - 1] = epre;
    if (j < p.G)
    {
        int32_t const kind = p.gkind[j];
        if (kind >= 0)
        {
            double mat[ND][ND];
#pragma unroll
            for (int a = 0; a < ND; ++a)
            {
#pragma unroll
                for (int b = 0; b < ND; ++b)
                {
                    mat[a][b] = p.gmat[(a * ND + b) * p.G + j];
                }
            }
            double o0[NEQ];
            bc_order0<ND>(kind, mat, p.inlet + static_cast<int64_t>(p.ginl[j]) * (ND + 3), u0, o0);
            double in1[NEQ][ND];
#pragma unroll
            for (int k = 0; k < NEQ; ++k)
            {
                p.s0n[j * NEQ + k] = o0[k];
#pragma unroll
                for (int d = 0; d < ND; ++d)
                {
                    in1[k][d] = p.s1c[row * (NEQ * ND) + k * ND + d];
                }
            }
            double o1[NEQ][ND];
            bc_order1<ND>(kind, mat, in1, o1);
#pragma unroll
            for (int k = 0; k < NEQ; ++k)
            {
#pragma unroll
                for (int d = 0; d < ND; ++d)
                {
                    p.s1n[j * (NEQ * ND) + k * ND + d] = o1[k][d];
                }
            }
            if constexpr ((MODE & M_STNEXT) != 0)
            {
                JacS<ND, FAST> gj;
                gj.set(p.gam[j], o0, &chk);
                double gst[NEQ];
                solt_of<ND>(gj, o1, gst);
                if constexpr (FAST)
                {
                    chk.finite(gst[NEQ - 1]);
                }
#pragma unroll
                for (int k = 0; k < NEQ; ++k)
                {
                    p.stn[j * NEQ + k] = gst[k];
                }
            }
        }
    }

    if constexpr (FAST)
    {
        return chk.ok();
    }
    return true;
}

// The cells of one block of a type group.
template <int T, int MODE>
__device__ inline void lane_block(KP const & p, GV const & g, unsigned blk, double * lds, bool only)
{
    constexpr int L = lanes_of<T>();
    constexpr int CELLS = BLK / L;
    int const l = threadIdx.x & (L - 1);
    int const c = threadIdx.x / L;
    int64_t const i = static_cast<int64_t>(blk) * CELLS + c;
    if (i >= g.cnt)
    {
        return;
    }
    double * const xs = lds + c * lane_words<T>();
    bool const ok = lane_cell<T, MODE, true>(p, g, i, l, xs, only);
    if (__builtin_expect(__any(!ok), 0))
    {
        // Exact passes run: the wavefronts that found out, then one per launch.
        if (only ? blk == 0 && threadIdx.x == 0 : __builtin_amdgcn_readfirstlane(threadIdx.x) == threadIdx.x)
        {
            atomicAdd(p.redo + 1, 1ull);
            p.redo[2] = 1;
        }
        // Keeps the exact form's loads its own.
        asm volatile("" ::: "memory");
        wave_lds();
        lane_cell<T, MODE, false>(p, g, i, l, xs, true);
    }
}

template <int ND>
constexpr int lds_words()
{
    if (ND == 2)
    {
        return std::max(BLK / lanes_of<CT_TRI>() * lane_words<CT_TRI>(), BLK / lanes_of<CT_QUAD>() * lane_words<CT_QUAD>());
    }
    return std::max(std::max(BLK / lanes_of<CT_TET>() * lane_words<CT_TET>(), BLK / lanes_of<CT_HEX>() * lane_words<CT_HEX>()),
                    std::max(BLK / lanes_of<CT_PRISM>() * lane_words<CT_PRISM>(),
                             BLK / lanes_of<CT_PYRAMID>() * lane_words<CT_PYRAMID>()));
}

// The march's exact-only switch (k_cell): read first, so that it is there when
// it is looked at.
__device__ inline bool exact_only(KP const & p)
{
    return p.redo[2] != 0;
}

// A single type group.
template <int T, int MODE>
__global__ void __launch_bounds__(BLK) k_lane(KP const p, GV const g)
{
    constexpr int L = lanes_of<T>();
    __shared__ double lds[BLK / L * lane_words<T>()];
    bool const only = exact_only(p);
    lane_block<T, MODE>(p, g, xcd_block(blockIdx.x, gridDim.x), lds, only);
}

// Every type group of a mesh, with the first group's switch and count for all.
template <int ND>
__global__ void __launch_bounds__(BLK) k_lane_all(KP const p, LaneGroups const lg)
{
    __shared__ double lds[lds_words<ND>()];
    bool const only = exact_only(p);
    unsigned const b = xcd_block(blockIdx.x, gridDim.x);
    int k = 0;
    for (int q = 1; q < lg.ng; ++q)
    {
        k = b >= lg.blk0[q] ? q : k;
    }
    GV const g = lg.g[k];
    unsigned const blk = b - lg.blk0[k];
    if constexpr (ND == 2)
    {
        if (lg.type[k] == CT_TRI)
        {
            lane_block<CT_TRI, 0>(p, g, blk, lds, only);
        }
        else
        {
            lane_block<CT_QUAD, 0>(p, g, blk, lds, only);
        }
    }
    else
    {
        switch (lg.type[k])
        {
        case CT_TET: lane_block<CT_TET, 0>(p, g, blk, lds, only); break;
        case CT_HEX: lane_block<CT_HEX, 0>(p, g, blk, lds, only); break;
        case CT_PRISM: lane_block<CT_PRISM, 0>(p, g, blk, lds, only); break;
        default: lane_block<CT_PYRAMID, 0>(p, g, blk, lds, only); break;
        }
    }
}

unsigned lane_blocks(int32_t type, int64_t cnt)
{
    return grid_for(cnt, BLK / (type == CT_TRI || type == CT_QUAD || type == CT_TET ? 4 : 8));
}

template <int MODE>
void launch_mode(int ndim, KP const & p, LaneGroups const & lg, hipStream_t stream)
{
    unsigned const nb = lg.blk0[lg.ng];
    if (lg.ng == 1)
    {
        GV const & g = lg.g[0];
        switch (lg.type[0])
        {
        case CT_TRI: k_lane<CT_TRI, MODE><<<nb, BLK, 0, stream>>>(p, g); break;
        case CT_QUAD: k_lane<CT_QUAD, MODE><<<nb, BLK, 0, stream>>>(p, g); break;
        case CT_TET: k_lane<CT_TET, MODE><<<nb, BLK, 0, stream>>>(p, g); break;
        case CT_HEX: k_lane<CT_HEX, MODE><<<nb, BLK, 0, stream>>>(p, g); break;
        case CT_PRISM: k_lane<CT_PRISM, MODE><<<nb, BLK, 0, stream>>>(p, g); break;
        case CT_PYRAMID: k_lane<CT_PYRAMID, MODE><<<nb, BLK, 0, stream>>>(p, g); break;
        default: fail(SC_ERUNTIME, "EulerCore: unsupported cell type in group");
        }
    }
    else if constexpr (MODE != 0)
    {
        fail(SC_ERUNTIME, "EulerCore: several groups in one launch do not chain so0t");
    }
    else if (ndim == 2)
    {
        k_lane_all<2><<<nb, BLK, 0, stream>>>(p, lg);
    }
    else
    {
        k_lane_all<3><<<nb, BLK, 0, stream>>>(p, lg);
    }
    SC_HIP(hipGetLastError());
}

} /* end namespace */

void lane_add(LaneGroups & lg, int32_t type, GV const & g)
{
    if (g.cnt <= 0)
    {
        return;
    }
    if (lg.ng == LANE_GROUPS)
    {
        fail(SC_ERUNTIME, "EulerCore: more type groups than cell types");
    }
    lg.type[lg.ng] = type;
    lg.g[lg.ng] = g;
    lg.blk0[lg.ng + 1] = lg.blk0[lg.ng] + lane_blocks(type, g.cnt);
    ++lg.ng;
}

void lane_launch(int ndim, int mode, KP const & p, LaneGroups const & lg, hipStream_t stream)
{
    if (lg.ng == 0)
    {
        return;
    }
    if (mode == M_STNEXT)
    {
        launch_mode<M_STNEXT>(ndim, p, lg, stream);
    }
    else
    {
        launch_mode<0>(ndim, p, lg, stream);
    }
}

} /* end namespace scamd */
