// mhh_tend.hip -- fused tendency of one dry-CBL substep: buoyancy
// (src/thermo_dry.cxx:163-180), 2i5 advection (src/advec_2i5.cxx:150-728) and
// Smagorinsky diffusion without a surface model (include/diff_kernels.h:144-484)
// of u, v, w and one scalar, accumulated onto ut, vt, wt, st in the order the
// reference driver applies them (src/model.cxx:388-414): buoyancy, horizontal
// advection, vertical advection, diffusion.
//
// Layout of the work.  A block owns a 64 x 4 column tile and marches upward
// through a chunk of levels.  At level k the LDS holds
//     u, v at k-1 and k,  w at k and k+1,  s at k      (halo 3 in x and y)
//     evisc at k-1, k, k+1                              (halo 1)
// rotating as k advances, so every plane is read from HBM once per chunk;
// the +-3 vertical neighbours of the thread's own column come from register
// queues.  Block ids are swizzled so that the tiles one XCD works on are
// neighbours: their halos are then served by that XCD's L2.
#include <algorithm>

#include "mhh_batch.h"
#include "mhh_stencil.h"
#include "mhh_tend.h"

namespace
{
    using namespace mhh;

    constexpr int TX = 64, TY = 4;
    constexpr int H = 3;                  // horizontal halo of the 2i5 stencil
    constexpr int PW = TX + 2*H, PH = TY + 2*H, PN = PW*PH;
    constexpr int EW = TX + 2, EH = TY + 2, EN = EW*EH;
    constexpr double grav = 9.81;        // include/constants.h:29

    // Per-thread share of a plane: elements tid, tid+256, tid+512 (halo-3
    // planes, 700 elements) or tid, tid+256 (halo-1 planes, 396 elements).
    constexpr int NQ3 = (PN + TX*TY - 1)/(TX*TY);
    constexpr int NQ1 = (EN + TX*TY - 1)/(TX*TY);

    // LIM: the pass also takes the two time-step inputs of the substep from
    // the fields it holds anyway, as block maxima in red_cfl / red_dn: the
    // 2i5 CFL rate (Advec_2i5::get_cfl without dt, src/advec_2i5.cxx:954-971;
    // u, v from the halo-3 planes, w from the column queue) and dnmul
    // (include/diff_kernels.h:486-511, from evisc at the point).
    template<typename TF, int MODE, bool LIM, bool SFC>
    __device__ __forceinline__ void tend_2i5_smag2_g(
            TF* __restrict__ ut, TF* __restrict__ vt, TF* __restrict__ wt, TF* __restrict__ st,
            const TF* __restrict__ u, const TF* __restrict__ v, const TF* __restrict__ w,
            const TF* __restrict__ s, const TF* __restrict__ evisc,
            const Level<TF>* __restrict__ lev, const TF* __restrict__ p, const TF* __restrict__ dpbar,
            Tend_args<TF> a, Gd g, double* __restrict__ red_cfl, double* __restrict__ red_dn, Wall_flux<TF> wfx,
            const Bid& bid_)
    {
        __shared__ __align__(16) TF lds[7*PN + 3*EN];

        // XCD-aware tile order: block b runs on XCD b % 8; give each XCD a
        // contiguous range of tiles (i fastest, then j, then the k chunk).
        const int nb = bid_.nx;
        const int ntiles = a.nti*a.ntj*a.nkc;
        const int tile = (bid_.x % 8)*(nb/8) + bid_.x/8;
        if (tile >= ntiles)
        {
            if (LIM && threadIdx.x == 0 && threadIdx.y == 0) { red_cfl[1 + bid_.x] = 0.; red_dn[1 + bid_.x] = 0.; }
            return;
        }
        const int ti = tile % a.nti;
        const int tj = (tile / a.nti) % a.ntj;
        const int kc = tile / (a.nti*a.ntj);

        const int tx = threadIdx.x, ty = threadIdx.y, tid = tx + TX*ty;
        const int i0 = g.istart + ti*TX, j0 = g.jstart + tj*TY;
        const int i = i0 + tx, j = j0 + ty;
        const bool active = i < g.iend && j < g.jend;
        const int kb = g.kstart + kc*a.kchunk;
        const int ke = min(kb + a.kchunk, g.kend);
        const int kk = g.ijcells;
        // Threads outside the domain compute on the clamped column (in bounds)
        // and store nothing.
        const int ij = min(i, g.iend-1) + min(j, g.jend-1)*g.icells;

        TF* Up = lds;        TF* Uc = Up + PN;
        TF* Vp = Uc + PN;    TF* Vc = Vp + PN;
        TF* Wc = Vc + PN;    TF* Wn = Wc + PN;
        TF* Sc = Wn + PN;
        TF* Ep = Sc + PN;    TF* Ec = Ep + EN;   TF* En = Ec + EN;

        load_plane(Up, u, kb-1, i0, j0, H, PW, PN, g, tid);
        load_plane(Vp, v, kb-1, i0, j0, H, PW, PN, g, tid);
        load_plane(Wc, w, kb, i0, j0, H, PW, PN, g, tid);
        load_plane(Ep, evisc, kb-1, i0, j0, 1, EW, EN, g, tid);
        load_plane(Ec, evisc, kb, i0, j0, 1, EW, EN, g, tid);

        // Column queues: q[m] holds level k-3+m of the thread's own column
        // (levels past the field repeat its top level: the stencils of the
        // faces near the top wall never reach them).
        const uint32_t oij = uint32_t(ij)*sizeof(TF);    // column offset within a level
        TF qu[7], qv[7], qw[7], qs[7];
        #pragma unroll
        for (int m = 0; m < 7; ++m)
        {
            const size_t kq = size_t(min(max(kb - 3 + m, 0), g.kcells - 1))*kk;
            qu[m] = ldo(u + kq, oij); qv[m] = ldo(v + kq, oij);
            qw[m] = ldo(w + kq, oij); qs[m] = ldo(s + kq, oij);
        }

        const int c = (ty + H)*PW + (tx + H);     // centre in the halo-3 planes
        const int ce = (ty + 1)*EW + (tx + 1);    // centre in the halo-1 planes
        const TF dxi = a.dxi, dyi = a.dyi, visc = a.visc;

        // Planes of the first level of the chunk go straight to LDS; the planes
        // of every next level are fetched into registers while the current one
        // is computed (software pipelining over k).
        load_plane(Uc, u, kb, i0, j0, H, PW, PN, g, tid);
        load_plane(Vc, v, kb, i0, j0, H, PW, PN, g, tid);
        load_plane(Wn, w, kb+1, i0, j0, H, PW, PN, g, tid);
        load_plane(Sc, s, kb, i0, j0, H, PW, PN, g, tid);
        load_plane(En, evisc, kb+1, i0, j0, 1, EW, EN, g, tid);
        TF ru[NQ3], rv[NQ3], rw[NQ3], rs[NQ3], re[NQ1];
        uint32_t o3[NQ3], o1[NQ1];
        plane_offsets<TF>(o3, i0, j0, H, PW, PN, g, tid);
        plane_offsets<TF>(o1, i0, j0, 1, EW, EN, g, tid);

        // Bottom-face terms of the first level of the chunk; every later level
        // takes them from the top face of the level below.
        TF bu_c, bu_u, bv_c, bv_u, bw_c, bw_u, bs_c, bs_u;   // advective
        TF du_b, dv_b, dw_b, ds_b;                          // diffusive
        __syncthreads();
        {
            const Level<TF> L = ld_const(lev, kb), Lm = ld_const(lev, kb-1);
            const TF rhh = TF(0.5)*L.rhoh;
            vface_c(kb, g.kstart, g.kend, rhh*(Wc[c-1] + Wc[c]),
                    qu[0], qu[1], qu[2], qu[3], qu[4], qu[5], bu_c, bu_u);
            vface_c(kb, g.kstart, g.kend, rhh*(Wc[c-PW] + Wc[c]),
                    qv[0], qv[1], qv[2], qv[3], qv[4], qv[5], bv_c, bv_u);
            vface_c(kb, g.kstart, g.kend, L.rhoh*Wc[c],
                    qs[0], qs[1], qs[2], qs[3], qs[4], qs[5], bs_c, bs_u);
            vface_w(kb-1, g.kstart, g.kend, TF(0.5)*Lm.rho,
                    qw[0], qw[1], qw[2], qw[3], qw[4], qw[5], bw_c, bw_u);
            const TF eu = TF(0.25)*(Ep[ce-1] + Ep[ce] + Ec[ce-1] + Ec[ce]) + visc;
            du_b = L.rhoh * eu*((qu[3]-qu[2])*L.dzhi + (Wc[c]-Wc[c-1])*dxi);
            const TF ev = TF(0.25)*(Ep[ce-EW] + Ep[ce] + Ec[ce-EW] + Ec[ce]) + visc;
            dv_b = L.rhoh * ev*((qv[3]-qv[2])*L.dzhi + (Wc[c]-Wc[c-PW])*dyi);
            dw_b = Lm.rho * (Ep[ce] + visc)*(qw[3]-qw[2])*Lm.dzi;
            const TF es = TF(0.5)*(Ep[ce]+Ec[ce]) * a.tPr_i + a.svisc;
            ds_b = L.rhoh * es*(qs[3]-qs[2])*L.dzhi;
            if (SFC && kb == g.kstart)
            {
                du_b = -L.rhoh*wfx.ub[ij];
                dv_b = -L.rhoh*wfx.vb[ij];
                ds_b = -L.rhoh*wfx.sb[ij];
            }
        }
        // TEND_DEFER: p of the own column one level down, carried from level
        // to level
        TF pb = MODE == TEND_DEFER ? ldo(p + size_t(kb-1)*kk, oij) : TF(0);
        double cm = 0., dm = 0.;   // LIM: running maxima of the CFL rate and dnmul
        // Every load of the preamble has landed: the waits inside the loop then
        // only count the loads issued in the loop.
        __builtin_amdgcn_s_waitcnt(0);

        for (int k = kb; k < ke; ++k)
        {
            const size_t kofs = size_t(k)*kk;
            TF* __restrict__ utk = ut + kofs; TF* __restrict__ vtk = vt + kofs;
            TF* __restrict__ wtk = wt + kofs; TF* __restrict__ stk = st + kofs;
            // Issue order sets what a wait covers (loads complete in order):
            // the tendencies of this level first, then the column values of
            // level k+4 (used by the next level), then the planes of the next
            // level, which stay in flight until the end of this one.  Every
            // level issues the same loads (the last one of the chunk fetches
            // clamped, unused planes), so the waits are the same on every pass.
            TF tu = TF(0), tv = TF(0), tw = TF(0), ts = TF(0);
            if (MODE != TEND_FRESH)
            {
                tu = ldo(utk, oij); tv = ldo(vtk, oij); tw = ldo(wtk, oij); ts = ldo(stk, oij);
            }
            TF pc = TF(0), pw = TF(0), ps = TF(0);
            if (MODE == TEND_DEFER)
            {
                // p at the point and its west and south neighbours
                const TF* __restrict__ pk = p + kofs;
                pc = ldo(pk, oij); pw = ldo(pk, oij - uint32_t(sizeof(TF)));
                ps = ldo(pk, oij - uint32_t(g.icells*sizeof(TF)));
            }
            __builtin_amdgcn_sched_barrier(0);
            const size_t kq = size_t(min(k + 4, g.kcells - 1))*kk;
            const TF nu = ldo(u + kq, oij), nv = ldo(v + kq, oij), nw = ldo(w + kq, oij), ns = ldo(s + kq, oij);
            __builtin_amdgcn_sched_barrier(0);
            {
                const int k1 = min(k + 1, g.kcells - 1), k2 = min(k + 2, g.kcells - 1);
                fetch_plane(ru, u, k1, o3, g);
                fetch_plane(rv, v, k1, o3, g);
                fetch_plane(rw, w, k2, o3, g);
                fetch_plane(rs, s, k1, o3, g);
                fetch_plane(re, evisc, k2, o1, g);
            }
            __syncthreads();

            const Level<TF> L = ld_const(lev, k);
            // L.cfac, L.wfac: dzi/rhoref and dzhi/rhorefh, the divisions of the
            // reference's "/ rhoref[k] * dzi[k]" taken out of the per-point work
            const TF cf = L.cfac, wf = L.wfac;
            // the 1/2 of the face-velocity interpolations, folded into the
            // grid factors and densities
            const TF dxih = TF(0.5)*dxi, dyih = TF(0.5)*dyi, rhph = TF(0.5)*L.rhohp;
            const TF dxi2 = TF(2.)*a.dxidxi, dyi2 = TF(2.)*a.dyidyi;
            // the south-west edge viscosity (i-1/2, j-1/2) is u's south and v's west edge
            const TF evsw = TF(0.25)*(Ec[ce-1-EW] + Ec[ce-EW] + Ec[ce-1] + Ec[ce]) + visc;

            // the deferred end of the previous substep, all four at once so
            // that the p values are dead before the stencils (tw is used
            // above the bottom wall only)
            if (MODE == TEND_DEFER)
            {
                TF dpz = pc - pb;
                if (dpbar) dpz += ld_const(dpbar, k);   // mixed mode: the FP64 mean's part
                tu = mul_rn(fma(pw - pc, dxi, tu), a.cA);
                tv = mul_rn(fma(ps - pc, dyi, tv), a.cA);
                tw = mul_rn(fma(-dpz, L.dzhi, tw), a.cA);
                ts = mul_rn(ts, a.cA);
                // FP64: keep the compiler from sinking these into the blocks
                // that use them, which would keep the p values live through
                // the stencils and spill (FP32 has registers to spare and runs
                // faster with the loads waited for later)
                if constexpr (sizeof(TF) == 8)
                    __asm__ volatile("" : "+v"(tu), "+v"(tv), "+v"(tw), "+v"(ts));
                pb = pc;
            }

            // -------------------------------------------------------------- u
            {
                tu += hflux_2i5_one(Uc[c] + Uc[c+1], Uc[c-1] + Uc[c], Uc, c, 1, dxih)
                    + hflux_2i5_one(Vc[c-1+PW] + Vc[c+PW], Vc[c-1] + Vc[c], Uc, c, PW, dyih);
                TF tc, tq;
                vface_c(k+1, g.kstart, g.kend, rhph*(Wn[c-1] + Wn[c]),
                        qu[1], qu[2], qu[3], qu[4], qu[5], qu[6], tc, tq);
                const TF evisce = Ec[ce] + visc;
                const TF eviscw = Ec[ce-1] + visc;
                const TF eviscn = TF(0.25)*(Ec[ce-1] + Ec[ce] + Ec[ce-1+EW] + Ec[ce+EW]) + visc;
                const TF eviscs = evsw;
                const TF evisct = TF(0.25)*(Ec[ce-1] + Ec[ce] + En[ce-1] + En[ce]) + visc;
                const TF hor =
                         + ( evisce*(Uc[c+1]-Uc[c  ])
                           - eviscw*(Uc[c  ]-Uc[c-1]) ) * dxi2
                         + ( eviscn*((Uc[c+PW]-Uc[c   ])*dyi + (Vc[c+PW]-Vc[c-1+PW])*dxi)
                           - eviscs*((Uc[c   ]-Uc[c-PW])*dyi + (Vc[c   ]-Vc[c-1   ])*dxi) ) * dyi;
                const TF dt = (SFC && k == g.kend-1) ? -L.rhohp*wfx.ut[ij]
                            : L.rhohp * evisct*((qu[4]-qu[3])*L.dzhip + (Wn[c]-Wn[c-1])*dxi);
                // vertical advection (centred, upwind) and diffusion share the factor
                tu += hor + ( ( tq - bu_u ) - ( tc - bu_c ) + ( dt - du_b ) ) * cf;
                bu_c = tc; bu_u = tq; du_b = dt;
                if (active) sto(utk, oij, tu);
            }
            // -------------------------------------------------------------- v
            {
                tv += hflux_2i5_one(Uc[c+1-PW] + Uc[c+1], Uc[c-PW] + Uc[c], Vc, c, 1, dxih)
                    + hflux_2i5_one(Vc[c] + Vc[c+PW], Vc[c-PW] + Vc[c], Vc, c, PW, dyih);
                TF tc, tq;
                vface_c(k+1, g.kstart, g.kend, rhph*(Wn[c-PW] + Wn[c]),
                        qv[1], qv[2], qv[3], qv[4], qv[5], qv[6], tc, tq);
                const TF evisce = TF(0.25)*(Ec[ce-EW] + Ec[ce] + Ec[ce+1-EW] + Ec[ce+1]) + visc;
                const TF eviscw = evsw;
                const TF eviscn = Ec[ce] + visc;
                const TF eviscs = Ec[ce-EW] + visc;
                const TF evisct = TF(0.25)*(Ec[ce-EW] + Ec[ce] + En[ce-EW] + En[ce]) + visc;
                const TF hor =
                         + ( evisce*((Vc[c+1]-Vc[c  ])*dxi + (Uc[c+1]-Uc[c+1-PW])*dyi)
                           - eviscw*((Vc[c  ]-Vc[c-1])*dxi + (Uc[c  ]-Uc[c  -PW])*dyi) ) * dxi
                         + ( eviscn*(Vc[c+PW]-Vc[c   ])
                           - eviscs*(Vc[c   ]-Vc[c-PW]) ) * dyi2;
                const TF dt = (SFC && k == g.kend-1) ? -L.rhohp*wfx.vt[ij]
                            : L.rhohp * evisct*((qv[4]-qv[3])*L.dzhip + (Wn[c]-Wn[c-PW])*dyi);
                tv += hor + ( ( tq - bv_u ) - ( tc - bv_c ) + ( dt - dv_b ) ) * cf;
                bv_c = tc; bv_u = tq; dv_b = dt;
                if (active) sto(vtk, oij, tv);
            }
            // -------------------------------------------------------------- w
            {
                // faces at the cell centres k (top) and k-1 (bottom, carried)
                TF tc, tq;
                vface_w(k, g.kstart, g.kend, TF(0.5)*L.rho, qw[1], qw[2], qw[3], qw[4], qw[5], qw[6], tc, tq);
                const TF dt = L.rho * (Ec[ce] + visc)*(qw[4]-qw[3])*L.dzi;
                if (k > g.kstart)
                {
                    if (a.buoyancy)
                        tw += L.gthi * (i2(qs[2], qs[3]) - L.threfh_rel);
                    tw += hflux_2i5_one(Up[c+1] + Uc[c+1], Up[c] + Uc[c], Wc, c, 1, dxih)
                        + hflux_2i5_one(Vp[c+PW] + Vc[c+PW], Vp[c] + Vc[c], Wc, c, PW, dyih);
                    const TF evisce = TF(0.25)*(Ep[ce] + Ec[ce] + Ep[ce+1] + Ec[ce+1]) + visc;
                    // the west and south edge viscosities in diff_w's own
                    // order (include/diff_kernels.h:350-392), at every level
                    const TF eviscw = TF(0.25)*(Ep[ce-1] + Ec[ce-1] + Ep[ce] + Ec[ce]) + visc;
                    const TF eviscn = TF(0.25)*(Ep[ce] + Ec[ce] + Ep[ce+EW] + Ec[ce+EW]) + visc;
                    const TF eviscs = TF(0.25)*(Ep[ce-EW] + Ec[ce-EW] + Ep[ce] + Ec[ce]) + visc;
                    tw += + ( evisce*((Wc[c+1]-Wc[c  ])*dxi + (Uc[c+1]-Up[c+1])*L.dzhi)
                            - eviscw*((Wc[c  ]-Wc[c-1])*dxi + (Uc[c  ]-Up[c  ])*L.dzhi) ) * dxi
                          + ( eviscn*((Wc[c+PW]-Wc[c   ])*dyi + (Vc[c+PW]-Vp[c+PW])*L.dzhi)
                            - eviscs*((Wc[c   ]-Wc[c-PW])*dyi + (Vc[c   ]-Vp[c   ])*L.dzhi) ) * dyi
                          + ( ( tq - bw_u ) - ( tc - bw_c ) + TF(2.)*( dt - dw_b ) ) * wf;
                    if (active) sto(wtk, oij, tw);
                }
                bw_c = tc; bw_u = tq; dw_b = dt;
            }
            // -------------------------------------------------------------- s
            {
                ts += hflux_2i5_one(Uc[c+1], Uc[c], Sc, c, 1, dxi)
                    + hflux_2i5_one(Vc[c+PW], Vc[c], Sc, c, PW, dyi);
                TF tc, tq;
                vface_c(k+1, g.kstart, g.kend, L.rhohp*Wn[c],
                        qs[1], qs[2], qs[3], qs[4], qs[5], qs[6], tc, tq);
                // 1/(2 tPr): the two-point average and the Prandtl number in one factor
                const TF htPr = TF(0.5)*a.tPr_i, sv = a.svisc;
                const TF evisce = (Ec[ce   ]+Ec[ce+1 ]) * htPr + sv;
                const TF eviscw = (Ec[ce-1 ]+Ec[ce   ]) * htPr + sv;
                const TF eviscn = (Ec[ce   ]+Ec[ce+EW]) * htPr + sv;
                const TF eviscs = (Ec[ce-EW]+Ec[ce   ]) * htPr + sv;
                const TF evisct = (Ec[ce   ]+En[ce   ]) * htPr + sv;
                const TF hor =
                         + ( evisce*(Sc[c+1]-Sc[c  ])
                           - eviscw*(Sc[c  ]-Sc[c-1]) ) * a.dxidxi
                         + ( eviscn*(Sc[c+PW]-Sc[c   ])
                           - eviscs*(Sc[c   ]-Sc[c-PW]) ) * a.dyidyi;
                const TF dt = (SFC && k == g.kend-1) ? -L.rhohp*wfx.st[ij]
                            : L.rhohp * evisct*(qs[4]-qs[3])*L.dzhip;
                ts += hor + ( ( tq - bs_u ) - ( tc - bs_c ) + ( dt - ds_b ) ) * cf;
                bs_c = tc; bs_u = tq; ds_b = dt;
                if (active) sto(stk, oij, ts);
            }
            if (LIM && active)
            {
                // the expressions of visc_tile_g's limits, w at k-2 .. k+3 = qw[1 .. 6]
                dm = fmax(dm, static_cast<double>(fabs(Ec[ce]*a.tPrfac_i*(a.dxidxi + a.dyidyi + L.dzi*L.dzi))));
                TF wpart;
                if (k == g.kstart || k == g.kend-1)
                    wpart = fabs(i2(qw[3], qw[4]))*L.dzi;
                else if (k == g.kstart+1 || k == g.kend-2)
                    wpart = fabs(i4ws(qw[2], qw[3], qw[4], qw[5]))*L.dzi;
                else
                    wpart = fabs(i6ws(qw[1], qw[2], qw[3], qw[4], qw[5], qw[6]))*L.dzi;
                const TF val = fabs(i6ws(Uc[c-2], Uc[c-1], Uc[c], Uc[c+1], Uc[c+2], Uc[c+3]))*dxi
                             + fabs(i6ws(Vc[c-2*PW], Vc[c-PW], Vc[c], Vc[c+PW], Vc[c+2*PW], Vc[c+3*PW]))*dyi
                             + wpart;
                cm = fmax(cm, static_cast<double>(val));
            }
            __syncthreads();

            // rotate the plane ring, store the prefetched planes, advance the queues
            TF* x;
            x = Up; Up = Uc; Uc = x;
            x = Vp; Vp = Vc; Vc = x;
            x = Wc; Wc = Wn; Wn = x;
            x = Ep; Ep = Ec; Ec = En; En = x;
            store_plane(Uc, ru, PN, tid);
            store_plane(Vc, rv, PN, tid);
            store_plane(Wn, rw, PN, tid);
            store_plane(Sc, rs, PN, tid);
            store_plane(En, re, EN, tid);
            #pragma unroll
            for (int m = 0; m < 6; ++m)
            {
                qu[m] = qu[m+1]; qv[m] = qv[m+1]; qw[m] = qw[m+1]; qs[m] = qs[m+1];
            }
            qu[6] = nu; qv[6] = nv; qw[6] = nw; qs[6] = ns;
        }
        if (LIM)
        {
            // block maxima, in the plane ring's LDS (no longer read)
            __syncthreads();
            double* smc = reinterpret_cast<double*>(lds);
            double* smd = smc + TX*TY;
            smc[tid] = cm; smd[tid] = dm;
            __syncthreads();
            for (int st2 = TX*TY/2; st2 > 0; st2 >>= 1)
            {
                if (tid < st2) { smc[tid] = fmax(smc[tid], smc[tid + st2]); smd[tid] = fmax(smd[tid], smd[tid + st2]); }
                __syncthreads();
            }
            if (tid == 0) { red_cfl[1 + bid_.x] = smc[0]; red_dn[1 + bid_.x] = smd[0]; }
        }
    }

    template<typename TF, int MODE, bool LIM, bool SFC>
    struct tend_2i5_smag2_k
    {
        static constexpr int NT = TX*TY, MINB = 2;
        TF* ut; TF* vt; TF* wt; TF* st; const TF* u; const TF* v; const TF* w; const TF* s; const TF* evisc;
        const Level<TF>* lev; const TF* p; const TF* dpbar; Tend_args<TF> a; Gd g; double* red_cfl;
        double* red_dn; Wall_flux<TF> wfx;
        __device__ __forceinline__ void operator()(const Bid& bid_) const
        {
            tend_2i5_smag2_g<TF, MODE, LIM, SFC>(ut, vt, wt, st, u, v, w, s, evisc, lev, p, dpbar, a, g,
                red_cfl, red_dn, wfx, bid_);
        }
    };

    template<typename TF>
    int tend(mhh_ctx* c, const Prof<TF>& p, const mhh_smag_params& par, int buoyancy,
             double* cfl_rate = nullptr, double* dnmul = nullptr)
    {
        const Gd& g = c->gd;
        if (c->f.nscalars < 1)
            return fail(MHH_ESTATE, "the fused tendency needs scalar 0");
        if (g.igc < 3 || g.jgc < 3)
            return fail(MHH_EINVAL, "the fused tendency needs igc = jgc >= 3");
        const bool sfc = par.surface_model != 0;
        if (sfc && (!c->f.u_fluxbot || !c->f.v_fluxbot || !c->f.s_fluxbot[0] || !c->f.u_fluxtop || !c->f.v_fluxtop
                    || !c->f.s_fluxtop[0]))
            return fail(MHH_ESTATE, "the surface-model variant needs the flux planes of u, v and scalar 0 bound");
        Wall_flux<TF> wfl{static_cast<const TF*>(c->f.u_fluxbot), static_cast<const TF*>(c->f.v_fluxbot),
                          static_cast<const TF*>(c->f.s_fluxbot[0]), static_cast<const TF*>(c->f.u_fluxtop),
                          static_cast<const TF*>(c->f.v_fluxtop), static_cast<const TF*>(c->f.s_fluxtop[0])};
        if (buoyancy && !p.threfh)
            return fail(MHH_ESTATE, "buoyancy needs mhh_set_base_state()");
        if (!p.lev)
            return fail(MHH_ESTATE, "the fused tendency needs the grid profiles");
        Tend_args<TF> a{};
        a.dxi = TF(1.)/TF(g.dx); a.dyi = TF(1.)/TF(g.dy);
        a.dxidxi = TF(1./(g.dx*g.dx)); a.dyidyi = TF(1./(g.dy*g.dy));
        a.visc = TF(par.visc); a.svisc = TF(par.svisc[0]); a.tPr_i = TF(1)/TF(par.tPr);
        a.tPrfac_i = TF(1)/std::min(TF(1.), TF(par.tPr));
        a.buoyancy = buoyancy;
        // a pending deferred RK3 update is completed in this pass
        const int mode = !c->defer_pending ? TEND_ADD : c->defer_cA == 0. ? TEND_FRESH : TEND_DEFER;
        a.cA = TF(c->defer_cA);
        if (mode == TEND_DEFER && !c->f.p)
            return fail(MHH_ESTATE, "a deferred tendency update needs p bound");
        const TF* dpb = c->mixed ? reinterpret_cast<const TF*>(c->dpbar) : nullptr;
        a.nti = (g.itot + TX - 1)/TX;
        a.ntj = (g.jtot + TY - 1)/TY;
        a.kchunk = c->tend_kchunk > 0 ? c->tend_kchunk : march_kchunk(c, a.nti*a.ntj, g.ktot, MARCH_LEAST_TEND);
        a.nkc = (g.ktot + a.kchunk - 1)/a.kchunk;
        const int ntiles = a.nti*a.ntj*a.nkc;
        const int nblocks = (ntiles + 7)/8*8;
        const bool lim = cfl_rate && dnmul;
        double* rc = nullptr; double* rd = nullptr;
        if (lim)
        {
            MHH_CHECK(ensure_reduction(c, 2*nblocks + 1));
            rc = c->red; rd = c->red + nblocks + 1;
        }
        { mhh::Timer _t(c, "tend_2i5_smag2");
#define MHH_TEND2(M, L, S) launch(c, tend_2i5_smag2_k<TF, M, L, S>{ \
                static_cast<TF*>(c->f.ut), static_cast<TF*>(c->f.vt), static_cast<TF*>(c->f.wt), \
                static_cast<TF*>(c->f.st[0]), \
                static_cast<const TF*>(c->f.u), static_cast<const TF*>(c->f.v), static_cast<const TF*>(c->f.w), \
                static_cast<const TF*>(c->f.s[0]), static_cast<const TF*>(c->f.evisc), p.lev, \
                static_cast<const TF*>(c->f.p), dpb, a, g, rc, rd, wfl}, nblocks, dim3(TX, TY))
#define MHH_TEND(M, L) do { if (sfc) MHH_TEND2(M, L, true); else MHH_TEND2(M, L, false); } while (0)
          if (lim)
          {
              if (mode == TEND_DEFER) MHH_TEND(TEND_DEFER, true);
              else if (mode == TEND_FRESH) MHH_TEND(TEND_FRESH, true);
              else MHH_TEND(TEND_ADD, true);
          }
          else
          {
              if (mode == TEND_DEFER) MHH_TEND(TEND_DEFER, false);
              else if (mode == TEND_FRESH) MHH_TEND(TEND_FRESH, false);
              else MHH_TEND(TEND_ADD, false);
          }
#undef MHH_TEND
#undef MHH_TEND2
        }
        c->defer_pending = false;
        MHH_CHECK(check_launch("tend_2i5_smag2"));
        if (!lim) return 0;
        MHH_CHECK(reduce_max_partials_at(c, rc, nblocks, cfl_rate));
        return reduce_max_partials_at(c, rd, nblocks, dnmul);
    }
}

extern "C" {

int mhh_tendency_2i5_smag2_limits(mhh_ctx* c, const mhh_smag_params* par, int buoyancy,
                                  double* cfl_rate, double* dnmul)
{
    MHH_REQUIRE_BOUND(c);
    if (!par || !cfl_rate || !dnmul) return mhh::fail(MHH_EINVAL, "null argument");
    if (!c->f.evisc) return mhh::fail(MHH_ESTATE, "evisc field is not bound");
    if (buoyancy && !c->have_base_state) return mhh::fail(MHH_ESTATE, "buoyancy needs mhh_set_base_state()");
    if (c->fluxlimit[0])
        return mhh::fail(MHH_ESTATE, "the fused tendency has no flux limiter: use mhh_advec_2i5_exec for limited scalars");
    return c->precision == MHH_FP64 ? tend<double>(c, c->pd, *par, buoyancy, cfl_rate, dnmul)
                                    : tend<float>(c, c->pf, *par, buoyancy, cfl_rate, dnmul);
}

int mhh_tendency_2i5_smag2(mhh_ctx* c, const mhh_smag_params* par, int buoyancy)
{
    MHH_REQUIRE_BOUND(c);
    if (!par) return mhh::fail(MHH_EINVAL, "null smag params");
    if (!c->f.evisc) return mhh::fail(MHH_ESTATE, "evisc field is not bound");
    if (buoyancy && !c->have_base_state) return mhh::fail(MHH_ESTATE, "buoyancy needs mhh_set_base_state()");
    if (c->fluxlimit[0])
        return mhh::fail(MHH_ESTATE, "the fused tendency has no flux limiter: use mhh_advec_2i5_exec for limited scalars");
    return c->precision == MHH_FP64 ? tend<double>(c, c->pd, *par, buoyancy) : tend<float>(c, c->pf, *par, buoyancy);
}

} // extern "C"
