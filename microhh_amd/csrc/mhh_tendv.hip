// mhh_tendv.hip -- the fused tendency pass with the eddy viscosity computed in
// it: Diff_smag2::exec_viscosity (strain2, N2 and the Richardson-limited
// closure of calc_evisc, include/diff_kernels.h:34-142, src/thermo_dry.cxx:
// 66-79, src/diff_smag2.cxx:148-269, with the wall mirror and the cyclic
// update of evisc), then buoyancy (src/thermo_dry.cxx:163-180), 2i5
// advection (src/advec_2i5.cxx:150-728) and Smagorinsky diffusion
// (include/diff_kernels.h:144-484) of u, v, w and scalar 0, accumulated onto
// the tendencies in the order of src/model.cxx:388-414.  The buoyant
// closure, with the default boundary or the surface model (the surface
// layer's gradients and N2 at kstart, optionally Mason damping, and the
// prescribed wall fluxes of the tendencies).
//
// Layout of the work.  A block owns a 32 x 8 column tile and marches upward
// through a chunk of levels.  At level k the LDS holds
//     u, v at k-1 .. k+2,  w, theta at k .. k+2             (halo 3 in x and y)
//     evisc at k-1, k, k+1                                    (halo 1)
// evisc at k+1 is computed at the start of level k from the planes at k .. k+2
// (strain2 and N2 never go to memory), so the viscosity costs no pass of its
// own and the tendencies no read of evisc; evisc is still written once (the
// field the time step and the diagnostics read).  The planes run two levels
// ahead of the tendencies, so the column values of the vertical stencils
// (loaded a level before their planes) are still in the L2 when the planes
// arrive.  14 halo-3 planes and 3 halo-1 planes: 68 KB in FP64, two blocks
// per CU.  The body of a level (the four tendencies, the chunk's first
// faces, the time-step maxima) is the one of the tendency pass in
// mhh_tend.hip, with the same expressions in the same order, and the
// viscosity shares its expressions with the viscosity pass (mhh_stencil.h):
// one pass and two passes agree to the bit.
#include <algorithm>

#include "mhh_batch.h"
#include "mhh_stencil.h"
#include "mhh_tend.h"

namespace
{
    using namespace mhh;

    constexpr int VX = 32, VY = 8;
    static_assert(VX*VY == TEND_NT, "one thread per column of the tile");
    constexpr int H = 3;                                   // horizontal halo of the 2i5 stencil
    constexpr int QW = VX + 2*H, QH = VY + 2*H, QN = QW*QH;   // halo-3 planes
    constexpr int FW = VX + 2, FH = VY + 2, FN = FW*FH;        // halo-1 planes (evisc)
    constexpr int NQ3 = (QN + TEND_NT - 1)/TEND_NT;
    constexpr int NQ1 = (FN + TEND_NT - 1)/TEND_NT;
    static_assert(NQ1 == 2 && FN - TEND_NT <= TEND_NT/2, "two rounds, the second for half the waves");

    // strain2_acc accessors: the plane ring (u, v at k-1, k, k+1 and w at k,
    // k+1 around the point, QW wide) and global memory.
    template<typename TF>
    struct Plane_acc
    {
        const TF* um; const TF* uc; const TF* up; const TF* vm; const TF* vc; const TF* vp;
        const TF* wc; const TF* wp; int c;
        __device__ __forceinline__ TF u(int di, int dj, int dk) const
        { return (dk < 0 ? um : dk > 0 ? up : uc)[c + di + dj*QW]; }
        __device__ __forceinline__ TF v(int di, int dj, int dk) const
        { return (dk < 0 ? vm : dk > 0 ? vp : vc)[c + di + dj*QW]; }
        __device__ __forceinline__ TF w(int di, int dj, int dk) const
        { return (dk > 0 ? wp : wc)[c + di + dj*QW]; }
    };

    template<typename TF>
    struct Col_acc
    {
        const TF* uu; const TF* vv; const TF* ww; int ijk, jj, kk;
        __device__ __forceinline__ TF u(int di, int dj, int dk) const { return uu[ijk + di + dj*jj + dk*kk]; }
        __device__ __forceinline__ TF v(int di, int dj, int dk) const { return vv[ijk + di + dj*jj + dk*kk]; }
        __device__ __forceinline__ TF w(int di, int dj, int dk) const { return ww[ijk + di + dj*jj + dk*kk]; }
    };

    // The surface layer's fields the viscosity reads with the surface model:
    // du/dz, dv/dz, db/dz at the wall and the roughness length z0m, one value
    // per column.
    template<typename TF>
    struct Sfc_in
    {
        const TF* dudz; const TF* dvdz; const TF* dbdz; const TF* z0m;
    };

    // mlen^2 at level k of column ij: the Smagorinsky length, with Mason
    // damping towards the surface for SFC = 2 (as the viscosity pass).
    template<typename TF, int SFC>
    __device__ __forceinline__ TF mlen2_at(const TF* __restrict__ mlen0, const TF* __restrict__ zc,
                                           const Sfc_in<TF>& sf, int ij, int k)
    {
        const TF ml = ld_const(mlen0, k);
        if (SFC == 2) return mason_sq<TF, 2>(ml, ld_const(zc, k), sf.z0m[ij]);
        return ml*ml;
    }

    // The interior column whose periodic image column (gi, gj) is: the
    // surface layer's planes are read there, as the viscosity pass reads them
    // for the interior column before it copies evisc to the images.
    __device__ __forceinline__ int interior_image(int gi, int gj, const Gd& g)
    {
        const int ii = gi < g.istart ? gi + g.itot : gi >= g.iend ? gi - g.itot : gi;
        const int jj = gj < g.jstart ? gj + g.jtot : gj >= g.jend ? gj - g.jtot : gj;
        return ii + jj*g.icells;
    }

    // evisc at column ij, level k (kstart <= k < kend) from global memory,
    // with the expressions of the viscosity pass and of the plane ring; ijs:
    // the column of the surface planes (the interior image of ij).
    template<typename TF, int SFC>
    __device__ __forceinline__ TF evisc_col(const TF* __restrict__ u, const TF* __restrict__ v,
                                            const TF* __restrict__ w, const TF* __restrict__ th,
                                            const Level<TF>* __restrict__ lev, const TF* __restrict__ mlen0,
                                            const TF* __restrict__ zc, const Sfc_in<TF>& sf,
                                            TF dxi, TF dyi, TF tPr_i, const Gd& g, int ij, int ijs, int k)
    {
        const int kk = g.ijcells, ijk = ij + k*kk;
        const Level<TF> L = ld_const(lev, k);
        const TF mlen2 = mlen2_at<TF, SFC>(mlen0, zc, sf, ijs, k);
        const Col_acc<TF> acc{u, v, w, ijk, g.icells, kk};
        if (SFC && k == g.kstart)
            return evisc_ri(strain2_surface_acc(acc, sf.dudz[ijs], sf.dvdz[ijs], dxi, dyi, L.dzi),
                            sf.dbdz[ijs]*tPr_i, mlen2);
        return evisc_ri(strain2_acc(acc, dxi, dyi, L.dzi, L.dzhi, L.dzhip),
                        L.n2fac*(th[ijk+kk] - th[ijk-kk])*tPr_i, mlen2);
    }

    // LIM: the pass also returns the block maxima of the 2i5 CFL rate
    // (Advec_2i5::get_cfl without dt, src/advec_2i5.cxx:954-971) and of dnmul
    // (include/diff_kernels.h:486-511), as the tendency pass without the
    // viscosity does.
    template<typename TF, int MODE, bool LIM, int SFC>
    __device__ __forceinline__ void tend_visc_g(
            TF* __restrict__ ut, TF* __restrict__ vt, TF* __restrict__ wt, TF* __restrict__ st,
            TF* __restrict__ evisc,
            const TF* __restrict__ u, const TF* __restrict__ v, const TF* __restrict__ w,
            const TF* __restrict__ s, const Level<TF>* __restrict__ lev, const TF* __restrict__ mlen0,
            const TF* __restrict__ zc, const TF* __restrict__ p, const TF* __restrict__ dpbar,
            Tend_args<TF> a, Gd g, double* __restrict__ red_cfl, double* __restrict__ red_dn,
            Wall_flux<TF> wfx, Sfc_in<TF> sf, const Bid& bid_)
    {
        __shared__ __align__(16) TF lds[14*QN + 3*FN];

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

        const int tx = threadIdx.x, ty = threadIdx.y, tid = tx + VX*ty;
        const int i0 = g.istart + ti*VX, j0 = g.jstart + tj*VY;
        const int i = i0 + tx, j = j0 + ty;
        const bool active = i < g.iend && j < g.jend;
        const int kb = g.kstart + kc*a.kchunk;
        const int ke = min(kb + a.kchunk, g.kend);
        const int kk = g.ijcells;
        const int ktop = g.kcells - 1;
        // Threads outside the domain compute on the clamped column (in bounds)
        // and store nothing.
        const int ij = min(i, g.iend-1) + min(j, g.jend-1)*g.icells;

        // the plane ring, named by level relative to k
        TF* Up = lds;        TF* Uc = Up + QN;   TF* Un = Uc + QN;   TF* Uq = Un + QN;
        TF* Vp = Uq + QN;    TF* Vc = Vp + QN;   TF* Vn = Vc + QN;   TF* Vq = Vn + QN;
        TF* Wc = Vq + QN;    TF* Wn = Wc + QN;   TF* Wq = Wn + QN;
        TF* Sc = Wq + QN;    TF* Sn = Sc + QN;   TF* Sq = Sn + QN;
        TF* Ep = Sq + QN;    TF* Ec = Ep + FN;   TF* En = Ec + FN;

        load_plane(Up, u, kb-1, i0, j0, H, QW, QN, g, tid);
        load_plane(Uc, u, kb, i0, j0, H, QW, QN, g, tid);
        load_plane(Un, u, kb+1, i0, j0, H, QW, QN, g, tid);
        load_plane(Uq, u, min(kb+2, ktop), i0, j0, H, QW, QN, g, tid);
        load_plane(Vp, v, kb-1, i0, j0, H, QW, QN, g, tid);
        load_plane(Vc, v, kb, i0, j0, H, QW, QN, g, tid);
        load_plane(Vn, v, kb+1, i0, j0, H, QW, QN, g, tid);
        load_plane(Vq, v, min(kb+2, ktop), i0, j0, H, QW, QN, g, tid);
        load_plane(Wc, w, kb, i0, j0, H, QW, QN, g, tid);
        load_plane(Wn, w, kb+1, i0, j0, H, QW, QN, g, tid);
        load_plane(Wq, w, min(kb+2, ktop), i0, j0, H, QW, QN, g, tid);
        load_plane(Sc, s, kb, i0, j0, H, QW, QN, g, tid);
        load_plane(Sn, s, kb+1, i0, j0, H, QW, QN, g, tid);
        load_plane(Sq, s, min(kb+2, ktop), i0, j0, H, QW, QN, g, tid);

        const TF dxi = a.dxi, dyi = a.dyi, visc = a.visc;
        // evisc of the chunk's first level and of the one below at the
        // tile's halo-1 positions, from global memory (the plane ring starts
        // at kb); below kstart the wall mirror (with the surface model a value
        // that no tendency reads: the wall fluxes replace the terms).  Positions beyond the last
        // interior column plus one feed only threads outside the domain: they
        // are clamped into the field.
        #pragma unroll
        for (int q = 0; q < NQ1; ++q)
        {
            const int idx = tid + q*TEND_NT;
            if (idx < FN)
            {
                const int pj = idx / FW, pi = idx - pj*FW;
                const int gi = min(i0 - 1 + pi, g.iend), gj = min(j0 - 1 + pj, g.jend);
                const int ijq = gi + gj*g.icells, ijs = SFC ? interior_image(gi, gj, g) : ijq;
                const TF ec = evisc_col<TF, SFC>(u, v, w, s, lev, mlen0, zc, sf, dxi, dyi, a.tPr_i, g, ijq, ijs, kb);
                Ec[idx] = ec;
                Ep[idx] = kb == g.kstart ? ec
                        : evisc_col<TF, SFC>(u, v, w, s, lev, mlen0, zc, sf, dxi, dyi, a.tPr_i, g, ijq, ijs, kb-1);
            }
        }

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

        const int c = (ty + H)*QW + (tx + H);     // centre in the halo-3 planes
        const int ce = (ty + 1)*FW + (tx + 1);    // centre in the halo-1 planes

        // the planes of level k+3 are fetched into registers while level k is
        // computed (software pipelining over k)
        TF ru[NQ3], rv[NQ3], rw[NQ3], rs[NQ3];
        uint32_t o3[NQ3];
        plane_offsets<TF>(o3, i0, j0, H, QW, QN, g, tid);

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
            vface_c(kb, g.kstart, g.kend, rhh*(Wc[c-QW] + Wc[c]),
                    qv[0], qv[1], qv[2], qv[3], qv[4], qv[5], bv_c, bv_u);
            vface_c(kb, g.kstart, g.kend, L.rhoh*Wc[c],
                    qs[0], qs[1], qs[2], qs[3], qs[4], qs[5], bs_c, bs_u);
            vface_w(kb-1, g.kstart, g.kend, TF(0.5)*Lm.rho,
                    qw[0], qw[1], qw[2], qw[3], qw[4], qw[5], bw_c, bw_u);
            const TF eu = TF(0.25)*(Ep[ce-1] + Ep[ce] + Ec[ce-1] + Ec[ce]) + visc;
            du_b = L.rhoh * eu*((qu[3]-qu[2])*L.dzhi + (Wc[c]-Wc[c-1])*dxi);
            const TF ev = TF(0.25)*(Ep[ce-FW] + Ep[ce] + Ec[ce-FW] + Ec[ce]) + visc;
            dv_b = L.rhoh * ev*((qv[3]-qv[2])*L.dzhi + (Wc[c]-Wc[c-QW])*dyi);
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
            // level k+4 (used by the next level); the planes of level k+3
            // follow after the viscosity and stay in flight until the end of
            // the level.  Every level issues the same loads (the last ones of
            // the chunk fetch clamped, unused planes), so the waits are the
            // same on every pass.
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
            __syncthreads();

            // evisc at level k+1 into En: strain2 from u, v at k .. k+2 and w
            // at k+1, k+2, N2 from theta at k and k+2; at the top wall the
            // mirror of level k (with the surface model unread: the wall flux
            // replaces the terms)
            if (k + 1 < g.kend)
            {
                const Level<TF> L1 = ld_const(lev, k + 1);
                // the second round has work for two of the four waves (84 of the
                // 340 positions): for waves 0 and 1 at even levels and 2 and 3 at
                // odd ones, so that no SIMD runs both rounds at every level (384 x 320 x
                // 160 FP64 1115 us with waves 0 and 1 always, 1098 now)
                #pragma unroll 1
                for (int q = 0; q < NQ1; ++q)
                {
                    const int idx = q == 0 ? tid : TEND_NT + ((tid + (k & 1)*(TEND_NT/2)) & (TEND_NT - 1));
                    if (idx < FN)
                    {
                        const int pj = idx / FW, pi = idx - pj*FW;
                        const int c3 = (pj + H - 1)*QW + (pi + H - 1);
                        const int ijq = SFC == 2 ? interior_image(min(i0 - 1 + pi, g.iend), min(j0 - 1 + pj, g.jend), g) : 0;
                        const TF s2 = strain2_acc(Plane_acc<TF>{Uc, Un, Uq, Vc, Vn, Vq, Wn, Wq, c3},
                                                  dxi, dyi, L1.dzi, L1.dzhi, L1.dzhip);
                        En[idx] = evisc_ri(s2, L1.n2fac*(Sq[c3] - Sc[c3])*a.tPr_i,
                                           mlen2_at<TF, SFC>(mlen0, zc, sf, ijq, k + 1));
                    }
                }
            }
            else
            {
                #pragma unroll
                for (int q = 0; q < NQ1; ++q)
                {
                    const int idx = tid + q*TEND_NT;
                    if (idx < FN) En[idx] = Ec[idx];
                }
            }
            __syncthreads();
            // the planes of level k+3, in flight until the end of the level
            // (issued after the viscosity, whose registers they would take)
            {
                const int k3 = min(k + 3, ktop);
                fetch_plane(ru, u, k3, o3, g);
                fetch_plane(rv, v, k3, o3, g);
                fetch_plane(rw, w, k3, o3, g);
                fetch_plane(rs, s, k3, o3, g);
            }

            const Level<TF> L = ld_const(lev, k);
            // L.cfac, L.wfac: dzi/rhoref and dzhi/rhorefh, the divisions of the
            // reference's "/ rhoref[k] * dzi[k]" taken out of the per-point work
            const TF cf = L.cfac, wf = L.wfac;
            // the 1/2 of the face-velocity interpolations, folded into the
            // grid factors and densities
            const TF dxih = TF(0.5)*dxi, dyih = TF(0.5)*dyi, rhph = TF(0.5)*L.rhohp;
            const TF dxi2 = TF(2.)*a.dxidxi, dyi2 = TF(2.)*a.dyidyi;
            // the south-west edge viscosity (i-1/2, j-1/2) is u's south and v's west edge
            const TF evsw = TF(0.25)*(Ec[ce-1-FW] + Ec[ce-FW] + Ec[ce-1] + Ec[ce]) + visc;

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
                    + hflux_2i5_one(Vc[c-1+QW] + Vc[c+QW], Vc[c-1] + Vc[c], Uc, c, QW, dyih);
                TF tc, tq;
                vface_c(k+1, g.kstart, g.kend, rhph*(Wn[c-1] + Wn[c]),
                        qu[1], qu[2], qu[3], qu[4], qu[5], qu[6], tc, tq);
                const TF evisce = Ec[ce] + visc;
                const TF eviscw = Ec[ce-1] + visc;
                const TF eviscn = TF(0.25)*(Ec[ce-1] + Ec[ce] + Ec[ce-1+FW] + Ec[ce+FW]) + visc;
                const TF eviscs = evsw;
                const TF evisct = TF(0.25)*(Ec[ce-1] + Ec[ce] + En[ce-1] + En[ce]) + visc;
                const TF hor =
                         + ( evisce*(Uc[c+1]-Uc[c  ])
                           - eviscw*(Uc[c  ]-Uc[c-1]) ) * dxi2
                         + ( eviscn*((Uc[c+QW]-Uc[c   ])*dyi + (Vc[c+QW]-Vc[c-1+QW])*dxi)
                           - eviscs*((Uc[c   ]-Uc[c-QW])*dyi + (Vc[c   ]-Vc[c-1   ])*dxi) ) * dyi;
                const TF dt = (SFC && k == g.kend-1) ? -L.rhohp*wfx.ut[ij]
                            : L.rhohp * evisct*((qu[4]-qu[3])*L.dzhip + (Wn[c]-Wn[c-1])*dxi);
                // vertical advection (centred, upwind) and diffusion share the factor
                tu += hor + ( ( tq - bu_u ) - ( tc - bu_c ) + ( dt - du_b ) ) * cf;
                bu_c = tc; bu_u = tq; du_b = dt;
                if (active) sto(utk, oij, tu);
            }
            // -------------------------------------------------------------- v
            {
                tv += hflux_2i5_one(Uc[c+1-QW] + Uc[c+1], Uc[c-QW] + Uc[c], Vc, c, 1, dxih)
                    + hflux_2i5_one(Vc[c] + Vc[c+QW], Vc[c-QW] + Vc[c], Vc, c, QW, dyih);
                TF tc, tq;
                vface_c(k+1, g.kstart, g.kend, rhph*(Wn[c-QW] + Wn[c]),
                        qv[1], qv[2], qv[3], qv[4], qv[5], qv[6], tc, tq);
                const TF evisce = TF(0.25)*(Ec[ce-FW] + Ec[ce] + Ec[ce+1-FW] + Ec[ce+1]) + visc;
                const TF eviscw = evsw;
                const TF eviscn = Ec[ce] + visc;
                const TF eviscs = Ec[ce-FW] + visc;
                const TF evisct = TF(0.25)*(Ec[ce-FW] + Ec[ce] + En[ce-FW] + En[ce]) + visc;
                const TF hor =
                         + ( evisce*((Vc[c+1]-Vc[c  ])*dxi + (Uc[c+1]-Uc[c+1-QW])*dyi)
                           - eviscw*((Vc[c  ]-Vc[c-1])*dxi + (Uc[c  ]-Uc[c  -QW])*dyi) ) * dxi
                         + ( eviscn*(Vc[c+QW]-Vc[c   ])
                           - eviscs*(Vc[c   ]-Vc[c-QW]) ) * dyi2;
                const TF dt = (SFC && k == g.kend-1) ? -L.rhohp*wfx.vt[ij]
                            : L.rhohp * evisct*((qv[4]-qv[3])*L.dzhip + (Wn[c]-Wn[c-QW])*dyi);
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
                        + hflux_2i5_one(Vp[c+QW] + Vc[c+QW], Vp[c] + Vc[c], Wc, c, QW, dyih);
                    const TF evisce = TF(0.25)*(Ep[ce] + Ec[ce] + Ep[ce+1] + Ec[ce+1]) + visc;
                    // the west and south edge viscosities in diff_w's own
                    // order (include/diff_kernels.h:350-392), at every level
                    const TF eviscw = TF(0.25)*(Ep[ce-1] + Ec[ce-1] + Ep[ce] + Ec[ce]) + visc;
                    const TF eviscn = TF(0.25)*(Ep[ce] + Ec[ce] + Ep[ce+FW] + Ec[ce+FW]) + visc;
                    const TF eviscs = TF(0.25)*(Ep[ce-FW] + Ec[ce-FW] + Ep[ce] + Ec[ce]) + visc;
                    tw += + ( evisce*((Wc[c+1]-Wc[c  ])*dxi + (Uc[c+1]-Up[c+1])*L.dzhi)
                            - eviscw*((Wc[c  ]-Wc[c-1])*dxi + (Uc[c  ]-Up[c  ])*L.dzhi) ) * dxi
                          + ( eviscn*((Wc[c+QW]-Wc[c   ])*dyi + (Vc[c+QW]-Vp[c+QW])*L.dzhi)
                            - eviscs*((Wc[c   ]-Wc[c-QW])*dyi + (Vc[c   ]-Vp[c   ])*L.dzhi) ) * dyi
                          + ( ( tq - bw_u ) - ( tc - bw_c ) + TF(2.)*( dt - dw_b ) ) * wf;
                    if (active) sto(wtk, oij, tw);
                }
                bw_c = tc; bw_u = tq; dw_b = dt;
            }
            // -------------------------------------------------------------- s
            {
                ts += hflux_2i5_one(Uc[c+1], Uc[c], Sc, c, 1, dxi)
                    + hflux_2i5_one(Vc[c+QW], Vc[c], Sc, c, QW, dyi);
                TF tc, tq;
                vface_c(k+1, g.kstart, g.kend, L.rhohp*Wn[c],
                        qs[1], qs[2], qs[3], qs[4], qs[5], qs[6], tc, tq);
                // 1/(2 tPr): the two-point average and the Prandtl number in one factor
                const TF htPr = TF(0.5)*a.tPr_i, sv = a.svisc;
                const TF evisce = (Ec[ce   ]+Ec[ce+1 ]) * htPr + sv;
                const TF eviscw = (Ec[ce-1 ]+Ec[ce   ]) * htPr + sv;
                const TF eviscn = (Ec[ce   ]+Ec[ce+FW]) * htPr + sv;
                const TF eviscs = (Ec[ce-FW]+Ec[ce   ]) * htPr + sv;
                const TF evisct = (Ec[ce   ]+En[ce   ]) * htPr + sv;
                const TF hor =
                         + ( evisce*(Sc[c+1]-Sc[c  ])
                           - eviscw*(Sc[c  ]-Sc[c-1]) ) * a.dxidxi
                         + ( eviscn*(Sc[c+QW]-Sc[c   ])
                           - eviscs*(Sc[c   ]-Sc[c-QW]) ) * a.dyidyi;
                const TF dt = (SFC && k == g.kend-1) ? -L.rhohp*wfx.st[ij]
                            : L.rhohp * evisct*(qs[4]-qs[3])*L.dzhip;
                ts += hor + ( ( tq - bs_u ) - ( tc - bs_c ) + ( dt - ds_b ) ) * cf;
                bs_c = tc; bs_u = tq; ds_b = dt;
                if (active) sto(stk, oij, ts);
            }
            if (active)
            {
                // evisc of the point, with the periodic images and the ghost
                // levels beyond the walls (the mirror of ev with the default
                // boundary; with the surface model the value they hold, and
                // its images): the field as the viscosity pass leaves it
                const TF ev = Ec[ce];
                TF* __restrict__ ek = evisc + kofs;
                sto(ek, oij, ev);
                put_images(ek, i, j, ev, g);
                if (k == g.kstart || k == g.kend-1)
                {
                    TF* __restrict__ wl = evisc + size_t(k == g.kstart ? k-1 : k+1)*kk;
                    if (!SFC) wl[i + j*g.icells] = ev;
                    put_images(wl, i, j, SFC ? wl[i + j*g.icells] : ev, g);
                }
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
                             + fabs(i6ws(Vc[c-2*QW], Vc[c-QW], Vc[c], Vc[c+QW], Vc[c+2*QW], Vc[c+3*QW]))*dyi
                             + wpart;
                cm = fmax(cm, static_cast<double>(val));
            }
            __syncthreads();

            // rotate the plane ring, store the prefetched planes, advance the queues
            TF* x;
            x = Up; Up = Uc; Uc = Un; Un = Uq; Uq = x;
            x = Vp; Vp = Vc; Vc = Vn; Vn = Vq; Vq = x;
            x = Wc; Wc = Wn; Wn = Wq; Wq = x;
            x = Sc; Sc = Sn; Sn = Sq; Sq = x;
            x = Ep; Ep = Ec; Ec = En; En = x;
            store_plane(Uq, ru, QN, tid);
            store_plane(Vq, rv, QN, tid);
            store_plane(Wq, rw, QN, tid);
            store_plane(Sq, rs, QN, tid);
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
            double* smd = smc + TEND_NT;
            smc[tid] = cm; smd[tid] = dm;
            __syncthreads();
            for (int st2 = TEND_NT/2; st2 > 0; st2 >>= 1)
            {
                if (tid < st2) { smc[tid] = fmax(smc[tid], smc[tid + st2]); smd[tid] = fmax(smd[tid], smd[tid + st2]); }
                __syncthreads();
            }
            if (tid == 0) { red_cfl[1 + bid_.x] = smc[0]; red_dn[1 + bid_.x] = smd[0]; }
        }
    }


    template<typename TF, int MODE, bool LIM, int SFC>
    struct tend_visc_k
    {
        static constexpr int NT = TEND_NT, MINB = 2;
        TF* ut; TF* vt; TF* wt; TF* st; TF* evisc; const TF* u; const TF* v; const TF* w; const TF* s;
        const Level<TF>* lev; const TF* mlen0; const TF* zc; const TF* p; const TF* dpbar; Tend_args<TF> a; Gd g;
        double* red_cfl; double* red_dn; Wall_flux<TF> wfx; Sfc_in<TF> sf;
        __device__ __forceinline__ void operator()(const Bid& bid_) const
        {
            tend_visc_g<TF, MODE, LIM, SFC>(ut, vt, wt, st, evisc, u, v, w, s, lev, mlen0, zc, p, dpbar, a, g,
                                            red_cfl, red_dn, wfx, sf, bid_);
        }
    };

    // Copy of a plane (the surface gradients kept for the viscosity).
    template<typename TF>
    struct copy_plane_k
    {
        static constexpr int NT = 256, MINB = 0;
        TF* dst; const TF* src; int n;
        __device__ __forceinline__ void operator()(const Bid& bid_) const
        {
            const int i = bid_.x*256 + static_cast<int>(threadIdx.x);
            if (i < n) dst[i] = src[i];
        }
    };

    template<typename TF> const TF* mlen_of(const mhh_ctx* c);
    template<> const double* mlen_of<double>(const mhh_ctx* c) { return c->mlen_d; }
    template<> const float* mlen_of<float>(const mhh_ctx* c) { return c->mlen_f; }

    // Whether the pass applies: the buoyant closure, and grids whose ghost
    // columns are each one periodic image (the pass writes evisc's images
    // itself); with the surface model its gradient, roughness and flux
    // planes bound.
    bool applies(const mhh_ctx* c, const mhh_smag_params& par)
    {
        const Gd& g = c->gd;
        const mhh_field_set& f = c->f;
        if (par.surface_model && (!f.dudz || !f.dvdz || !f.dbdz || !f.z0m || !f.u_fluxbot || !f.v_fluxbot
                                  || !f.u_fluxtop || !f.v_fluxtop || !f.s_fluxbot[0] || !f.s_fluxtop[0]))
            return false;
        return par.thermo && f.nscalars > 0 && c->have_base_state
            && g.igc >= 3 && g.jgc >= 3 && g.kgc == 1 && g.itot >= 2*g.igc && g.jtot >= 2*g.jgc
            && !c->fluxlimit[0];
    }

    template<typename TF>
    int tend_visc(mhh_ctx* c, const Prof<TF>& p, const mhh_smag_params& par, int buoyancy,
                  double* cfl_rate, double* dnmul)
    {
        const Gd& g = c->gd;
        if (buoyancy && !p.threfh)
            return fail(MHH_ESTATE, "buoyancy needs mhh_set_base_state()");
        if (!p.lev)
            return fail(MHH_ESTATE, "the fused tendency needs the grid profiles");
        MHH_CHECK(smag_prepare(c, par));
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
        a.nti = (g.itot + VX - 1)/VX;
        a.ntj = (g.jtot + VY - 1)/VY;
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
        const mhh_field_set& f = c->f;
        const int sfc = par.surface_model ? (par.swmason ? 2 : 1) : 0;
        Wall_flux<TF> wfl{static_cast<const TF*>(f.u_fluxbot), static_cast<const TF*>(f.v_fluxbot),
                          static_cast<const TF*>(f.s_fluxbot[0]), static_cast<const TF*>(f.u_fluxtop),
                          static_cast<const TF*>(f.v_fluxtop), static_cast<const TF*>(f.s_fluxtop[0])};
        // the surface gradients: those kept before the surface layer ran
        // (mhh_tendency_keep_surface_gradients), else the current ones
        const TF* kept = static_cast<const TF*>(c->sfc_keep);
        const size_t np = static_cast<size_t>(g.ijcells);
        Sfc_in<TF> sf{static_cast<const TF*>(f.dudz), static_cast<const TF*>(f.dvdz),
                      static_cast<const TF*>(f.dbdz), static_cast<const TF*>(f.z0m)};
        if (sfc && c->sfc_kept) { sf.dudz = kept; sf.dvdz = kept + np; sf.dbdz = kept + 2*np; }
        { mhh::Timer _t(c, "tend_visc");
#define MHH_TENDV2(M, L, S) launch(c, tend_visc_k<TF, M, L, S>{ \
                static_cast<TF*>(f.ut), static_cast<TF*>(f.vt), static_cast<TF*>(f.wt), \
                static_cast<TF*>(f.st[0]), static_cast<TF*>(f.evisc), \
                static_cast<const TF*>(f.u), static_cast<const TF*>(f.v), static_cast<const TF*>(f.w), \
                static_cast<const TF*>(f.s[0]), p.lev, mlen_of<TF>(c), p.z, \
                static_cast<const TF*>(f.p), dpb, a, g, rc, rd, wfl, sf}, nblocks, dim3(VX, VY))
#define MHH_TENDV(M, L) do { if (sfc == 2) MHH_TENDV2(M, L, 2); else if (sfc) MHH_TENDV2(M, L, 1); \
                             else MHH_TENDV2(M, L, 0); } while (0)
          if (lim)
          {
              if (mode == TEND_DEFER) MHH_TENDV(TEND_DEFER, true);
              else if (mode == TEND_FRESH) MHH_TENDV(TEND_FRESH, true);
              else MHH_TENDV(TEND_ADD, true);
          }
          else
          {
              if (mode == TEND_DEFER) MHH_TENDV(TEND_DEFER, false);
              else if (mode == TEND_FRESH) MHH_TENDV(TEND_FRESH, false);
              else MHH_TENDV(TEND_ADD, false);
          }
#undef MHH_TENDV
#undef MHH_TENDV2
        }
        c->defer_pending = false;
        c->sfc_kept = false;
        MHH_CHECK(check_launch("tend_visc"));
        if (!lim) return 0;
        MHH_CHECK(reduce_max_partials_at(c, rc, nblocks, cfl_rate));
        return reduce_max_partials_at(c, rd, nblocks, dnmul);
    }

    // The viscosity pass then the tendency pass, the viscosity from the kept
    // surface gradients when there are some.
    int two_passes(mhh_ctx* c, const mhh_smag_params* par, int buoyancy, double* cfl_rate, double* dnmul)
    {
        if (par->surface_model && c->sfc_kept)
        {
            mhh_field_set& f = c->f;
            const size_t np = static_cast<size_t>(c->gd.ijcells)*(c->precision == MHH_FP64 ? 8 : 4);
            void* cur[3] = {f.dudz, f.dvdz, f.dbdz};
            char* kept = static_cast<char*>(c->sfc_keep);
            f.dudz = kept; f.dvdz = kept + np; f.dbdz = kept + 2*np;
            const int rc = mhh_diff_smag2_exec_viscosity(c, par);
            f.dudz = cur[0]; f.dvdz = cur[1]; f.dbdz = cur[2];
            MHH_CHECK(rc);
        }
        else
            MHH_CHECK(mhh_diff_smag2_exec_viscosity(c, par));
        c->sfc_kept = false;
        return cfl_rate ? mhh_tendency_2i5_smag2_limits(c, par, buoyancy, cfl_rate, dnmul)
                        : mhh_tendency_2i5_smag2(c, par, buoyancy);
    }

    // One pass or two: the one pass where it applies and is chosen
    // (MHH_TUNE_VISC_SEPARATE = 2) or, by default, on grids of at least 256 x
    // 256 columns: on smaller ones (ensemble members) its 32 x 8 tiles and
    // the recomputed halo viscosity cost more than the second pass saves.
    bool one_pass(const mhh_ctx* c, const mhh_smag_params& par)
    {
        if (!applies(c, par) || c->visc_mode == 1) return false;
        return c->visc_mode == 2 || static_cast<long long>(c->gd.itot)*c->gd.jtot >= 256*256;
    }

    int run(mhh_ctx* c, const mhh_smag_params* par, int buoyancy, double* cfl_rate, double* dnmul)
    {
        if (!par) return fail(MHH_EINVAL, "null smag params");
        if (!c->f.evisc) return fail(MHH_ESTATE, "evisc field is not bound");
        if (buoyancy && !c->have_base_state) return fail(MHH_ESTATE, "buoyancy needs mhh_set_base_state()");
        if (!one_pass(c, *par))
            return two_passes(c, par, buoyancy, cfl_rate, dnmul);
        return c->precision == MHH_FP64 ? tend_visc<double>(c, c->pd, *par, buoyancy, cfl_rate, dnmul)
                                        : tend_visc<float>(c, c->pf, *par, buoyancy, cfl_rate, dnmul);
    }

    template<typename TF>
    int keep(mhh_ctx* c)
    {
        const mhh_field_set& f = c->f;
        if (!f.dudz || !f.dvdz || !f.dbdz)
            return fail(MHH_ESTATE, "mhh_tendency_keep_surface_gradients needs dudz, dvdz and dbdz bound");
        const int n = c->gd.ijcells;
        if (!c->sfc_keep)
            MHH_CHECK(check_hip(hipMalloc(&c->sfc_keep, sizeof(TF)*3*static_cast<size_t>(n)), "hipMalloc(sfc_keep)"));
        TF* k = static_cast<TF*>(c->sfc_keep);
        const int nb = (n + 255)/256;
        launch(c, copy_plane_k<TF>{k, static_cast<const TF*>(f.dudz), n}, nb, 256);
        launch(c, copy_plane_k<TF>{k + n, static_cast<const TF*>(f.dvdz), n}, nb, 256);
        launch(c, copy_plane_k<TF>{k + 2*static_cast<size_t>(n), static_cast<const TF*>(f.dbdz), n}, nb, 256);
        c->sfc_kept = true;
        return check_launch("keep_surface_gradients");
    }
}

extern "C" {

int mhh_tendency_2i5_smag2_visc(mhh_ctx* c, const mhh_smag_params* par, int buoyancy)
{
    MHH_REQUIRE_BOUND(c);
    return run(c, par, buoyancy, nullptr, nullptr);
}

int mhh_tendency_2i5_smag2_visc_limits(mhh_ctx* c, const mhh_smag_params* par, int buoyancy,
                                       double* cfl_rate, double* dnmul)
{
    MHH_REQUIRE_BOUND(c);
    if (!cfl_rate || !dnmul) return mhh::fail(MHH_EINVAL, "null argument");
    return run(c, par, buoyancy, cfl_rate, dnmul);
}

int mhh_tendency_2i5_smag2_visc_fused(const mhh_ctx* c, const mhh_smag_params* par, int* fused)
{
    if (!c || !par || !fused) return mhh::fail(MHH_EINVAL, "null argument");
    *fused = one_pass(c, *par) ? 1 : 0;
    return 0;
}

int mhh_tendency_keep_surface_gradients(mhh_ctx* c)
{
    MHH_REQUIRE_BOUND(c);
    return c->precision == MHH_FP64 ? keep<double>(c) : keep<float>(c);
}

}
