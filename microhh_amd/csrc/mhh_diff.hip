// mhh_diff.hip -- Smagorinsky (smag2) eddy viscosity and stress divergence,
// and constant-viscosity diffusion (diff_2).
//
// The viscosity kernel fuses strain2 (include/diff_kernels.h:34-142), N2
// (src/thermo_dry.cxx:66-79) and the evisc closure (src/diff_smag2.cxx:47-269)
// per point: S^2 and N^2 never go to memory, only evisc does.
#include <cmath>

#include "mhh_batch.h"
#include "mhh_stencil.h"

namespace
{
    using namespace mhh;

    constexpr double dsmall = 1.e-9;   // include/constants.h:97
    constexpr double kappa = 0.4;      // include/constants.h:28
    constexpr double grav = 9.81;      // include/constants.h:29

    __device__ __forceinline__ bool point(const Gd& g, int kfirst, int& i, int& j, int& k)
    {
        i = blockIdx.x*BX + threadIdx.x + g.istart;
        j = blockIdx.y*BY + threadIdx.y + g.jstart;
        k = blockIdx.z + kfirst;
        return i < g.iend && j < g.jend;
    }

    __device__ __forceinline__ bool point(const Bid& b, const Gd& g, int kfirst, int& i, int& j, int& k)
    {
        i = b.x*BX + threadIdx.x + g.istart;
        j = b.y*BY + threadIdx.y + g.jstart;
        k = b.z + kfirst;
        return i < g.iend && j < g.jend;
    }

    template<typename TF>
    struct Visc_args
    {
        TF* __restrict__ evisc;
        const TF* __restrict__ u;
        const TF* __restrict__ v;
        const TF* __restrict__ w;
        const TF* __restrict__ th;
        const TF* __restrict__ dudz;
        const TF* __restrict__ dvdz;
        const TF* __restrict__ dbdz;
        const TF* __restrict__ z0m;
        const TF* __restrict__ z;
        const TF* __restrict__ dzi;
        const TF* __restrict__ dzhi;
        const TF* __restrict__ thref;
        const TF* __restrict__ mlen0;
        TF dxi, dyi, tPr, visc, zsize;
    };

    // ---- plane-ring viscosity kernel ----
    // A block owns a 64 x 4 column tile and marches up a chunk of levels with
    // u, v at k-1, k, k+1 and w at k, k+1 in LDS (halo 1), so every plane is
    // read from HBM once per chunk; theta comes from a register queue.  With
    // `limits` it also returns the block maxima of the 2i5 CFL rate
    // (src/advec_2i5.cxx:59-148, without the dt factor) and of dnmul
    // (include/diff_kernels.h:486-511) for the time step.  The surface-model
    // variants take the wall gradients and N2 of the surface layer at kstart.
    constexpr int VTX = 64, VTY = 4;
    constexpr int VPW = VTX + 2, VPH = VTY + 2, VPN = VPW*VPH;
    constexpr int VNQ = (VPN + VTX*VTY - 1)/(VTX*VTY);

    // Accessor of the LDS plane ring for strain2_acc: u, v at k-1, k, k+1 and
    // w at k, k+1, each plane VPW wide.
    template<typename TF>
    struct Ring_acc
    {
        const TF* __restrict__ um; const TF* __restrict__ uc; const TF* __restrict__ up;
        const TF* __restrict__ vm; const TF* __restrict__ vc; const TF* __restrict__ vp;
        const TF* __restrict__ wc; const TF* __restrict__ wp; int c;
        __device__ __forceinline__ TF u(int di, int dj, int dk) const
        { return (dk < 0 ? um : dk > 0 ? up : uc)[c + di + dj*VPW]; }
        __device__ __forceinline__ TF v(int di, int dj, int dk) const
        { return (dk < 0 ? vm : dk > 0 ? vp : vc)[c + di + dj*VPW]; }
        __device__ __forceinline__ TF w(int di, int dj, int dk) const
        { return (dk > 0 ? wp : wc)[c + di + dj*VPW]; }
    };

    // The surface layer's fields for the surface-model variants: du/dz, dv/dz,
    // db/dz at the wall and the roughness length z0m, one value per column.
    template<typename TF>
    struct Visc_surface
    {
        const TF* dudz; const TF* dvdz; const TF* dbdz; const TF* z0m;
    };

    template<typename TF>
    __device__ __forceinline__ void vplane_load(TF* __restrict__ dst, const TF* __restrict__ src, int k,
                                                const int (&o)[VNQ], int tid, const Gd& g)
    {
        const TF* __restrict__ sk = src + static_cast<size_t>(k)*g.ijcells;
        #pragma unroll
        for (int q = 0; q < VNQ; ++q)
        {
            const int idx = tid + q*VTX*VTY;
            if (idx < VPN) dst[idx] = o[q] >= 0 ? sk[o[q]] : TF(0);
        }
    }

    template<typename TF>
    __device__ __forceinline__ TF vldo(const TF* __restrict__ base, uint32_t off)
    {
        return *reinterpret_cast<const TF*>(reinterpret_cast<const char*>(base) + off);
    }

    // Unconditional loads of the thread's share of plane k (k < kcells) at the
    // byte offsets ob (0 for elements past the plane or outside the field).
    template<typename TF>
    __device__ __forceinline__ void vplane_fetch(TF (&r)[VNQ], const TF* __restrict__ src, int k,
                                                 const uint32_t (&ob)[VNQ], const Gd& g)
    {
        const TF* __restrict__ sk = src + static_cast<size_t>(k)*g.ijcells;
        #pragma unroll
        for (int q = 0; q < VNQ; ++q) r[q] = vldo(sk, ob[q]);
    }

    template<typename TF>
    __device__ __forceinline__ void vplane_store(TF* __restrict__ dst, const TF (&r)[VNQ], int tid)
    {
        #pragma unroll
        for (int q = 0; q < VNQ-1; ++q)
            dst[tid + q*VTX*VTY] = r[q];
        const int idx = tid + (VNQ-1)*VTX*VTY;
        if (idx < VPN) dst[idx] = r[VNQ-1];
    }

    template<typename TF>
    struct Visc_scalars
    {
        TF dxi, dyi, tPr_i, visc, zsize, tPrfac_i, dxidxi, dyidyi;
    };

    // Viscosity of the default boundary (no surface model) over a 64 x 4 tile
    // marching up a chunk of levels: u, v at k-1, k, k+1 and w at k, k+1 in an
    // LDS plane ring (halo 1).  Pointers are __restrict__ kernel parameters,
    // so the per-level factors come in through scalar loads.  With `limits`
    // also the block maxima of the 2i5 CFL rate and of dnmul.
    // SFC: 0 the default boundary (van Driest damping in the neutral case, the
    // wall mirror of evisc), 1 the surface model (surface gradients and N2 at
    // kstart, no mirror), 2 the surface model with Mason damping.
    template<typename TF, bool thermo, bool limits, int SFC>
    __device__ __forceinline__ void visc_tile_g(
            TF* __restrict__ evisc, const TF* __restrict__ u, const TF* __restrict__ v,
            const TF* __restrict__ w, const TF* __restrict__ th, const Level<TF>* __restrict__ lev,
            const TF* __restrict__ mlen0, const TF* __restrict__ zc, Visc_scalars<TF> a, Gd g,
            int nti, int ntj, int nkc, int kchunk, int halo, double* __restrict__ red_cfl, double* __restrict__ red_dn,
            const Visc_surface<TF>& sf, const Bid& bid_)
    {
        static_assert(!(SFC && limits), "the fused limits cover the default boundary only");
        __shared__ TF lds[8*VPN];
        __shared__ double smc[limits ? VTX*VTY : 1], smd[limits ? VTX*VTY : 1];
        const int tid = threadIdx.x + VTX*threadIdx.y;
        // XCD-aware tile order, as in the fused tendency kernel
        const int nb = bid_.nx;
        const int tile = (bid_.x % 8)*(nb/8) + bid_.x/8;
        if (tile >= nti*ntj*nkc)
        {
            if (limits && tid == 0) { red_cfl[1 + bid_.x] = 0.; red_dn[1 + bid_.x] = 0.; }
            return;
        }
        const int ti = tile % nti, tj = (tile / nti) % ntj, kc = tile / (nti*ntj);
        const int i0 = g.istart + ti*VTX, j0 = g.jstart + tj*VTY;
        const int i = i0 + threadIdx.x, j = j0 + threadIdx.y;
        const bool active = i < g.iend && j < g.jend;
        const int kb = g.kstart + kc*kchunk, ke = min(kb + kchunk, g.kend);
        const int kk = g.ijcells;
        // threads outside the domain compute on the clamped column and store nothing
        const int ij = min(i, g.iend-1) + min(j, g.jend-1)*g.icells;
        const uint32_t oij = uint32_t(ij)*sizeof(TF);

        int o[VNQ];
        uint32_t ob[VNQ];
        #pragma unroll
        for (int q = 0; q < VNQ; ++q)
        {
            const int idx = tid + q*VTX*VTY;
            const int pj = idx / VPW, pi = idx - pj*VPW;
            const int gi = i0 - 1 + pi, gj = j0 - 1 + pj;
            o[q] = (idx < VPN && gi < g.icells && gj < g.jcells) ? gi + gj*g.icells : -1;
            ob[q] = o[q] >= 0 ? uint32_t(o[q])*sizeof(TF) : 0u;
        }
        TF* Um = lds;        TF* Uc = Um + VPN;   TF* Up = Uc + VPN;
        TF* Vm = Up + VPN;   TF* Vc = Vm + VPN;   TF* Vp = Vc + VPN;
        TF* Wc = Vp + VPN;   TF* Wp = Wc + VPN;
        vplane_load(Um, u, kb-1, o, tid, g); vplane_load(Uc, u, kb, o, tid, g); vplane_load(Up, u, kb+1, o, tid, g);
        vplane_load(Vm, v, kb-1, o, tid, g); vplane_load(Vc, v, kb, o, tid, g); vplane_load(Vp, v, kb+1, o, tid, g);
        vplane_load(Wc, w, kb, o, tid, g);   vplane_load(Wp, w, kb+1, o, tid, g);

        // theta at k-1, k+1 of the own column (N2, src/thermo_dry.cxx:66-79)
        TF t0 = TF(0), t1 = TF(0), t2 = TF(0);
        if (thermo)
        {
            t0 = vldo(th + size_t(kb-1)*kk, oij); t1 = vldo(th + size_t(kb)*kk, oij);
            t2 = vldo(th + size_t(kb+1)*kk, oij);
        }
        // van Driest wall friction velocities of the column (neutral case)
        TF u_tau_bot = TF(0), u_tau_top = TF(0);
        if (!thermo && !SFC)
        {
            const int kbot = ij + g.kstart*kk, ktop = ij + g.kend*kk;
            u_tau_bot = pow(sq(a.visc*(u[kbot] - u[kbot-kk])*ld_const(lev, g.kstart).dzhi)
                          + sq(a.visc*(v[kbot] - v[kbot-kk])*ld_const(lev, g.kstart).dzhi), TF(0.25));
            u_tau_top = pow(sq(a.visc*(u[ktop] - u[ktop-kk])*ld_const(lev, g.kend).dzhi)
                          + sq(a.visc*(v[ktop] - v[ktop-kk])*ld_const(lev, g.kend).dzhi), TF(0.25));
        }
        const int c = (threadIdx.y + 1)*VPW + (threadIdx.x + 1);
        double cm = 0., dm = 0.;
        TF ru[VNQ], rv[VNQ], rw[VNQ];
        // CFL: w of the own column at k-2 .. k+3 in a register queue (levels
        // outside the field repeat the nearest one; the wall stencils never
        // reach them)
        TF wq[6];
        if (limits)
        {
            #pragma unroll
            for (int m = 0; m < 6; ++m)
                wq[m] = vldo(w + size_t(min(max(kb - 2 + m, 0), g.kcells - 1))*kk, oij);
        }
        __builtin_amdgcn_s_waitcnt(0);

        for (int k = kb; k < ke; ++k)
        {
            // Issue order sets what a wait covers (loads complete in order): the
            // CFL stencil values this level needs beyond the LDS planes first
            // (u at i-2, i+2, i+3 and v at j-2, j+2, j+3, in the cache lines of
            // the planes, and w of the own column at k+4 for the queue), then
            // theta of level k+2, then the planes of level k+2, which stay in
            // flight until the end of the level.  Every level issues the same
            // loads (clamped levels).
            TF cu[3], cv[3], wn = TF(0);
            if (limits)
            {
                const TF* __restrict__ uk = u + size_t(k)*kk;
                const TF* __restrict__ vk = v + size_t(k)*kk;
                const int sz = int(sizeof(TF)), jb = g.icells*int(sizeof(TF));
                cu[0] = vldo(uk, oij - uint32_t(2*sz)); cu[1] = vldo(uk, oij + uint32_t(2*sz));
                cu[2] = vldo(uk, oij + uint32_t(3*sz));
                cv[0] = vldo(vk, oij - uint32_t(2*jb)); cv[1] = vldo(vk, oij + uint32_t(2*jb));
                cv[2] = vldo(vk, oij + uint32_t(3*jb));
                wn = vldo(w + size_t(min(k + 4, g.kcells - 1))*kk, oij);
                __builtin_amdgcn_sched_barrier(0);
            }
            const int k2 = min(k + 2, g.kcells - 1);
            TF tn = TF(0);
            if (thermo) tn = vldo(th + size_t(k2)*kk, oij);
            __builtin_amdgcn_sched_barrier(0);
            vplane_fetch(ru, u, k2, ob, g);
            vplane_fetch(rv, v, k2, ob, g);
            vplane_fetch(rw, w, k2, ob, g);
            __syncthreads();

            const Level<TF> L = ld_const(lev, k);
            const bool bot = SFC && k == g.kstart;
            const TF s2 = bot ? strain2_surface_acc(Ring_acc<TF>{Um, Uc, Up, Vm, Vc, Vp, Wc, Wp, c},
                                                    vldo(sf.dudz, oij), vldo(sf.dvdz, oij), a.dxi, a.dyi, L.dzi)
                              : strain2_acc(Ring_acc<TF>{Um, Uc, Up, Vm, Vc, Vp, Wc, Wp, c}, a.dxi, a.dyi,
                                            L.dzi, L.dzhi, L.dzhip);
            TF ev;
            // mlen^2: the Smagorinsky length, with Mason damping towards the
            // surface (per column: z0m)
            TF mlen2;
            if (SFC == 2)
                mlen2 = mason_sq<TF, thermo ? 2 : 1>(ld_const(mlen0, k), ld_const(zc, k), vldo(sf.z0m, oij));
            else
            {
                const TF mlen = ld_const(mlen0, k);
                mlen2 = mlen*mlen;
            }
            if (thermo)
            {
                // the Richardson-limited closure; N2 at kstart with the
                // surface model is db/dz of the surface layer
                const TF n2_tPr = (bot ? vldo(sf.dbdz, oij) : L.n2fac*(t2 - t0))*a.tPr_i;
                ev = evisc_ri(s2, n2_tPr, mlen2);
            }
            else if (SFC)
                ev = mlen2 * sqrt(s2);
            else
            {
                const TF A_vandriest = TF(26.);
                const TF zk = ld_const(zc, k);
                const TF fac_bot = TF(1.) - exp(-(        zk *u_tau_bot) / (A_vandriest*a.visc));
                const TF fac_top = TF(1.) - exp(-((a.zsize-zk)*u_tau_top) / (A_vandriest*a.visc));
                const TF fac = fmin(fac_bot, fac_top);
                ev = sq(fac * ld_const(mlen0, k)) * sqrt(s2);
            }
            if (active) *reinterpret_cast<TF*>(reinterpret_cast<char*>(evisc + size_t(k)*kk) + oij) = ev;
            if (halo && active)
            {
                // the wall mirror and the cyclic update of the pass, done here
                put_images(evisc + size_t(k)*kk, i, j, ev, g);
                if (k == g.kstart || k == g.kend-1)
                {
                    // the ghost level beyond the wall: the mirror of ev (default
                    // boundary) or, with the surface model, the value it holds;
                    // either way with its periodic images
                    TF* __restrict__ wl = evisc + size_t(k == g.kstart ? k-1 : k+1)*kk;
                    if (!SFC) wl[i + j*g.icells] = ev;
                    put_images(wl, i, j, SFC ? wl[i + j*g.icells] : ev, g);
                }
            }
            if (limits && active)
            {
                dm = fmax(dm, static_cast<double>(fabs(ev*a.tPrfac_i*(a.dxidxi + a.dyidyi + L.dzi*L.dzi))));
                // the 2i5 CFL rate as in cfl_g
                TF wpart;
                if (k == g.kstart || k == g.kend-1)
                    wpart = fabs(i2(wq[2], wq[3]))*L.dzi;
                else if (k == g.kstart+1 || k == g.kend-2)
                    wpart = fabs(i4ws(wq[1], wq[2], wq[3], wq[4]))*L.dzi;
                else
                    wpart = fabs(i6ws(wq[0], wq[1], wq[2], wq[3], wq[4], wq[5]))*L.dzi;
                const TF val = fabs(i6ws(cu[0], Uc[c-1], Uc[c], Uc[c+1], cu[1], cu[2]))*a.dxi
                             + fabs(i6ws(cv[0], Vc[c-VPW], Vc[c], Vc[c+VPW], cv[1], cv[2]))*a.dyi
                             + wpart;
                cm = fmax(cm, static_cast<double>(val));
            }
            __syncthreads();
            TF* x;
            x = Um; Um = Uc; Uc = Up; Up = x;
            x = Vm; Vm = Vc; Vc = Vp; Vp = x;
            x = Wc; Wc = Wp; Wp = x;
            vplane_store(Up, ru, tid);
            vplane_store(Vp, rv, tid);
            vplane_store(Wp, rw, tid);
            t0 = t1; t1 = t2; t2 = tn;
            if (limits)
            {
                #pragma unroll
                for (int m = 0; m < 5; ++m) wq[m] = wq[m+1];
                wq[5] = wn;
            }
        }
        if (limits)
        {
            smc[tid] = cm; smd[tid] = dm;
            __syncthreads();
            for (int st = VTX*VTY/2; st > 0; st >>= 1)
            {
                if (tid < st) { smc[tid] = fmax(smc[tid], smc[tid + st]); smd[tid] = fmax(smd[tid], smd[tid + st]); }
                __syncthreads();
            }
            if (tid == 0) { red_cfl[1 + bid_.x] = smc[0]; red_dn[1 + bid_.x] = smd[0]; }
        }
    }

    template<typename TF, bool thermo, bool limits, int SFC>
    struct visc_tile_k
    {
        static constexpr int NT = VTX*VTY, MINB = 0;
        TF* evisc; const TF* u; const TF* v; const TF* w; const TF* th; const Level<TF>* lev;
        const TF* mlen0; const TF* zc; Visc_scalars<TF> a; Gd g; int nti; int ntj; int nkc; int kchunk;
        int halo; double* red_cfl; double* red_dn; Visc_surface<TF> sf;
        __device__ __forceinline__ void operator()(const Bid& bid_) const
        {
            visc_tile_g<TF, thermo, limits, SFC>(evisc, u, v, w, th, lev, mlen0, zc, a, g, nti, ntj, nkc, kchunk,
                halo, red_cfl, red_dn, sf, bid_);
        }
    };

    // Mirror evisc over both walls (src/diff_smag2.cxx:193-205) for the interior
    // columns; the cyclic update that follows fills the horizontal ghosts.
    template<typename TF>
    __device__ __forceinline__ void mirror_walls_g(TF* __restrict__ evisc, Gd g, const Bid& bid_)
    {
        const int i = bid_.x*blockDim.x + threadIdx.x + g.istart;
        const int j = bid_.y*blockDim.y + threadIdx.y + g.jstart;
        if (i >= g.iend || j >= g.jend) return;
        const int ij = i + j*g.icells, kk = g.ijcells;
        evisc[ij + (g.kstart-1)*kk] = evisc[ij + g.kstart*kk];
        evisc[ij + g.kend*kk] = evisc[ij + (g.kend-1)*kk];
    }

    template<typename TF>
    struct mirror_walls_k
    {
        static constexpr int NT = 1024, MINB = 0;
        TF* evisc; Gd g;
        __device__ __forceinline__ void operator()(const Bid& bid_) const
        {
            mirror_walls_g<TF>(evisc, g, bid_);
        }
    };

    template<typename TF>
    struct Diff_args
    {
        TF* __restrict__ at;
        const TF* __restrict__ a;      // diffused scalar (diff_c)
        const TF* __restrict__ u;
        const TF* __restrict__ v;
        const TF* __restrict__ w;
        const TF* __restrict__ evisc;
        const TF* __restrict__ fluxbot;
        const TF* __restrict__ fluxtop;
        const TF* __restrict__ dzi;
        const TF* __restrict__ dzhi;
        const TF* __restrict__ rho;
        const TF* __restrict__ rhoh;
        TF dxi, dyi, dxidxi, dyidyi, visc, tPr;
    };

    // diff_u (include/diff_kernels.h:144-240).
    template<typename TF, bool sfc>
    __global__ void __launch_bounds__(BX*BY) diff_u_g(Diff_args<TF> a, Gd g)
    {
        int i, j, k;
        if (!point(g, g.kstart, i, j, k)) return;
        const int ii = 1, jj = g.icells, kk = g.ijcells;
        const int ij = i + j*jj, ijk = ij + k*kk;
        const TF* __restrict__ u = a.u; const TF* __restrict__ v = a.v; const TF* __restrict__ w = a.w;
        const TF* __restrict__ e = a.evisc;
        const TF visc = a.visc, dxi = a.dxi, dyi = a.dyi;
        const TF evisce = e[ijk   ] + visc;
        const TF eviscw = e[ijk-ii] + visc;
        const TF eviscn = TF(0.25)*(e[ijk-ii   ] + e[ijk   ] + e[ijk-ii+jj] + e[ijk+jj]) + visc;
        const TF eviscs = TF(0.25)*(e[ijk-ii-jj] + e[ijk-jj] + e[ijk-ii   ] + e[ijk   ]) + visc;
        const TF hor =
                 + ( evisce*(u[ijk+ii]-u[ijk   ])*dxi
                   - eviscw*(u[ijk   ]-u[ijk-ii])*dxi ) * TF(2.)*dxi
                 + ( eviscn*((u[ijk+jj]-u[ijk   ])*dyi  + (v[ijk+jj]-v[ijk-ii+jj])*dxi)
                   - eviscs*((u[ijk   ]-u[ijk-jj])*dyi  + (v[ijk   ]-v[ijk-ii   ])*dxi) ) * dyi;
        TF ver;
        if (sfc && k == g.kstart)
        {
            const TF evisct = TF(0.25)*(e[ijk-ii   ] + e[ijk   ] + e[ijk-ii+kk] + e[ijk+kk]) + visc;
            ver = ( a.rhoh[k+1] * evisct*((u[ijk+kk]-u[ijk   ])* a.dzhi[k+1] + (w[ijk+kk]-w[ijk-ii+kk])*dxi)
                  + a.rhoh[k  ] * a.fluxbot[ij] ) / a.rho[k] * a.dzi[k];
        }
        else if (sfc && k == g.kend-1)
        {
            const TF eviscb = TF(0.25)*(e[ijk-ii-kk] + e[ijk-kk] + e[ijk-ii   ] + e[ijk   ]) + visc;
            ver = (- a.rhoh[k+1] * a.fluxtop[ij]
                   - a.rhoh[k  ] * eviscb*((u[ijk   ]-u[ijk-kk])* a.dzhi[k] + (w[ijk   ]-w[ijk-ii   ])*dxi) ) / a.rho[k] * a.dzi[k];
        }
        else
        {
            const TF evisct = TF(0.25)*(e[ijk-ii   ] + e[ijk   ] + e[ijk-ii+kk] + e[ijk+kk]) + visc;
            const TF eviscb = TF(0.25)*(e[ijk-ii-kk] + e[ijk-kk] + e[ijk-ii   ] + e[ijk   ]) + visc;
            ver = ( a.rhoh[k+1] * evisct*((u[ijk+kk]-u[ijk   ])* a.dzhi[k+1] + (w[ijk+kk]-w[ijk-ii+kk])*dxi)
                  - a.rhoh[k  ] * eviscb*((u[ijk   ]-u[ijk-kk])* a.dzhi[k  ] + (w[ijk   ]-w[ijk-ii   ])*dxi) ) / a.rho[k] * a.dzi[k];
        }
        a.at[ijk] += hor + ver;
    }

    // diff_v (include/diff_kernels.h:242-340).
    template<typename TF, bool sfc>
    __global__ void __launch_bounds__(BX*BY) diff_v_g(Diff_args<TF> a, Gd g)
    {
        int i, j, k;
        if (!point(g, g.kstart, i, j, k)) return;
        const int ii = 1, jj = g.icells, kk = g.ijcells;
        const int ij = i + j*jj, ijk = ij + k*kk;
        const TF* __restrict__ u = a.u; const TF* __restrict__ v = a.v; const TF* __restrict__ w = a.w;
        const TF* __restrict__ e = a.evisc;
        const TF visc = a.visc, dxi = a.dxi, dyi = a.dyi;
        const TF evisce = TF(0.25)*(e[ijk   -jj] + e[ijk   ] + e[ijk+ii-jj] + e[ijk+ii]) + visc;
        const TF eviscw = TF(0.25)*(e[ijk-ii-jj] + e[ijk-ii] + e[ijk   -jj] + e[ijk   ]) + visc;
        const TF eviscn = e[ijk   ] + visc;
        const TF eviscs = e[ijk-jj] + visc;
        const TF hor =
                 + ( evisce*((v[ijk+ii]-v[ijk   ])*dxi + (u[ijk+ii]-u[ijk+ii-jj])*dyi)
                   - eviscw*((v[ijk   ]-v[ijk-ii])*dxi + (u[ijk   ]-u[ijk   -jj])*dyi) ) * dxi
                 + ( eviscn*(v[ijk+jj]-v[ijk   ])*dyi
                   - eviscs*(v[ijk   ]-v[ijk-jj])*dyi ) * TF(2.)*dyi;
        TF ver;
        if (sfc && k == g.kstart)
        {
            const TF evisct = TF(0.25)*(e[ijk   -jj] + e[ijk   ] + e[ijk+kk-jj] + e[ijk+kk]) + visc;
            ver = ( a.rhoh[k+1] * evisct*((v[ijk+kk]-v[ijk   ])*a.dzhi[k+1] + (w[ijk+kk]-w[ijk-jj+kk])*dyi)
                  + a.rhoh[k  ] * a.fluxbot[ij] ) / a.rho[k] * a.dzi[k];
        }
        else if (sfc && k == g.kend-1)
        {
            const TF eviscb = TF(0.25)*(e[ijk-kk-jj] + e[ijk-kk] + e[ijk   -jj] + e[ijk   ]) + visc;
            ver = (- a.rhoh[k+1] * a.fluxtop[ij]
                   - a.rhoh[k  ] * eviscb*((v[ijk   ]-v[ijk-kk])*a.dzhi[k] + (w[ijk   ]-w[ijk-jj   ])*dyi) ) / a.rho[k] * a.dzi[k];
        }
        else
        {
            const TF evisct = TF(0.25)*(e[ijk   -jj] + e[ijk   ] + e[ijk+kk-jj] + e[ijk+kk]) + visc;
            const TF eviscb = TF(0.25)*(e[ijk-kk-jj] + e[ijk-kk] + e[ijk   -jj] + e[ijk   ]) + visc;
            ver = ( a.rhoh[k+1] * evisct*((v[ijk+kk]-v[ijk   ])*a.dzhi[k+1] + (w[ijk+kk]-w[ijk-jj+kk])*dyi)
                  - a.rhoh[k  ] * eviscb*((v[ijk   ]-v[ijk-kk])*a.dzhi[k  ] + (w[ijk   ]-w[ijk-jj   ])*dyi) ) / a.rho[k] * a.dzi[k];
        }
        a.at[ijk] += hor + ver;
    }

    // diff_w (include/diff_kernels.h:342-390), half levels kstart+1..kend-1.
    template<typename TF>
    __global__ void __launch_bounds__(BX*BY) diff_w_g(Diff_args<TF> a, Gd g)
    {
        int i, j, k;
        if (!point(g, g.kstart+1, i, j, k)) return;
        const int ii = 1, jj = g.icells, kk = g.ijcells;
        const int ijk = i + j*jj + k*kk;
        const TF* __restrict__ u = a.u; const TF* __restrict__ v = a.v; const TF* __restrict__ w = a.w;
        const TF* __restrict__ e = a.evisc;
        const TF visc = a.visc, dxi = a.dxi, dyi = a.dyi, dzhik = a.dzhi[k];
        const TF evisce = TF(0.25)*(e[ijk   -kk] + e[ijk   ] + e[ijk+ii-kk] + e[ijk+ii]) + visc;
        const TF eviscw = TF(0.25)*(e[ijk-ii-kk] + e[ijk-ii] + e[ijk   -kk] + e[ijk   ]) + visc;
        const TF eviscn = TF(0.25)*(e[ijk   -kk] + e[ijk   ] + e[ijk+jj-kk] + e[ijk+jj]) + visc;
        const TF eviscs = TF(0.25)*(e[ijk-jj-kk] + e[ijk-jj] + e[ijk   -kk] + e[ijk   ]) + visc;
        const TF evisct = e[ijk   ] + visc;
        const TF eviscb = e[ijk-kk] + visc;
        a.at[ijk] +=
                 + ( evisce*((w[ijk+ii]-w[ijk   ])*dxi + (u[ijk+ii]-u[ijk+ii-kk])*dzhik)
                   - eviscw*((w[ijk   ]-w[ijk-ii])*dxi + (u[ijk   ]-u[ijk   -kk])*dzhik) ) * dxi
                 + ( eviscn*((w[ijk+jj]-w[ijk   ])*dyi + (v[ijk+jj]-v[ijk+jj-kk])*dzhik)
                   - eviscs*((w[ijk   ]-w[ijk-jj])*dyi + (v[ijk   ]-v[ijk   -kk])*dzhik) ) * dyi
                 + ( a.rho[k  ] * evisct*(w[ijk+kk]-w[ijk   ])*a.dzi[k  ]
                   - a.rho[k-1] * eviscb*(w[ijk   ]-w[ijk-kk])*a.dzi[k-1] ) / a.rhoh[k] * TF(2.)*dzhik;
    }

    // diff_c (include/diff_kernels.h:392-484).
    template<typename TF, bool sfc>
    __global__ void __launch_bounds__(BX*BY) diff_c_g(Diff_args<TF> a, Gd g)
    {
        int i, j, k;
        if (!point(g, g.kstart, i, j, k)) return;
        const int ii = 1, jj = g.icells, kk = g.ijcells;
        const int ij = i + j*jj, ijk = ij + k*kk;
        const TF* __restrict__ s = a.a;
        const TF* __restrict__ e = a.evisc;
        const TF visc = a.visc, tPr_i = TF(1)/a.tPr;
        const TF dxidxi = a.dxidxi, dyidyi = a.dyidyi;
        const TF evisce = TF(0.5)*(e[ijk   ]+e[ijk+ii]) * tPr_i + visc;
        const TF eviscw = TF(0.5)*(e[ijk-ii]+e[ijk   ]) * tPr_i + visc;
        const TF eviscn = TF(0.5)*(e[ijk   ]+e[ijk+jj]) * tPr_i + visc;
        const TF eviscs = TF(0.5)*(e[ijk-jj]+e[ijk   ]) * tPr_i + visc;
        const TF hor =
                 + ( evisce*(s[ijk+ii]-s[ijk   ])
                   - eviscw*(s[ijk   ]-s[ijk-ii]) ) * dxidxi
                 + ( eviscn*(s[ijk+jj]-s[ijk   ])
                   - eviscs*(s[ijk   ]-s[ijk-jj]) ) * dyidyi;
        TF ver;
        if (sfc && k == g.kstart)
        {
            const TF evisct = TF(0.5)*(e[ijk   ]+e[ijk+kk]) * tPr_i + visc;
            ver = ( a.rhoh[k+1] * evisct*(s[ijk+kk]-s[ijk   ])*a.dzhi[k+1]
                  + a.rhoh[k  ] * a.fluxbot[ij] ) / a.rho[k] * a.dzi[k];
        }
        else if (sfc && k == g.kend-1)
        {
            const TF eviscb = TF(0.5)*(e[ijk-kk]+e[ijk   ]) * tPr_i + visc;
            ver = (-a.rhoh[k+1] * a.fluxtop[ij]
                   - a.rhoh[k  ] * eviscb*(s[ijk   ]-s[ijk-kk])*a.dzhi[k] ) / a.rho[k] * a.dzi[k];
        }
        else
        {
            const TF evisct = TF(0.5)*(e[ijk   ]+e[ijk+kk]) * tPr_i + visc;
            const TF eviscb = TF(0.5)*(e[ijk-kk]+e[ijk   ]) * tPr_i + visc;
            ver = ( a.rhoh[k+1] * evisct*(s[ijk+kk]-s[ijk   ])*a.dzhi[k+1]
                  - a.rhoh[k  ] * eviscb*(s[ijk   ]-s[ijk-kk])*a.dzhi[k]  ) / a.rho[k] * a.dzi[k];
        }
        a.at[ijk] += hor + ver;
    }

    // calc_dnmul (include/diff_kernels.h:486-511), per-block maxima.
    template<typename TF>
    __global__ void __launch_bounds__(BX*BY) dnmul_g(const TF* __restrict__ evisc, const TF* __restrict__ dzi,
                                                     TF dxidxi, TF dyidyi, TF tPrfac_i, Gd g, double* __restrict__ red)
    {
        __shared__ double sm[BX*BY];
        const int tid = threadIdx.x + threadIdx.y*BX;
        const int i = blockIdx.x*BX + threadIdx.x + g.istart;
        const int j = blockIdx.y*BY + threadIdx.y + g.jstart;
        const int kb = g.kstart + blockIdx.z*RED_KCHUNK;
        const int ke = min(kb + RED_KCHUNK, g.kend);
        double m = 0.;
        if (i < g.iend && j < g.jend)
            for (int k = kb; k < ke; ++k)
            {
                const int ijk = i + j*g.icells + k*g.ijcells;
                m = fmax(m, static_cast<double>(fabs(evisc[ijk]*tPrfac_i*(dxidxi + dyidyi + dzi[k]*dzi[k]))));
            }
        sm[tid] = m;
        __syncthreads();
        for (int s = BX*BY/2; s > 0; s >>= 1)
        {
            if (tid < s) sm[tid] = fmax(sm[tid], sm[tid + s]);
            __syncthreads();
        }
        if (tid == 0)
            red[1 + blockIdx.x + gridDim.x*(blockIdx.y + gridDim.y*blockIdx.z)] = sm[0];
    }

    // A field read at offsets from a point of global memory.
    template<typename TF>
    struct Gacc2
    {
        const TF* __restrict__ f; int ijk, jj, kk;
        __device__ __forceinline__ TF operator()(int di, int dj, int dk) const { return f[ijk + di + dj*jj + dk*kk]; }
    };

    // Diff_2 (src/diff_2.cxx:39-85): the constant-viscosity Laplacian, one
    // point per thread; the expression is diff_2_pt (mhh_stencil.h), shared
    // with the fused 2nd-order tendency pass.
    template<typename TF>
    __global__ void __launch_bounds__(BX*BY) diff_2_c_g(TF* __restrict__ at, const TF* __restrict__ a, TF visc,
                                                        const TF* __restrict__ dzi, const TF* __restrict__ dzhi,
                                                        TF dxidxi, TF dyidyi, Gd g)
    {
        int i, j, k;
        if (!point(g, g.kstart, i, j, k)) return;
        const int jj = g.icells, kk = g.ijcells, ijk = i + j*jj + k*kk;
        at[ijk] += diff_2_pt(Gacc2<TF>{a, ijk, jj, kk}, visc, dxidxi, dyidyi, dzi[k], dzhi[k], dzhi[k+1]);
    }

    template<typename TF>
    __global__ void __launch_bounds__(BX*BY) diff_2_w_g(TF* __restrict__ wt, const TF* __restrict__ w, TF visc,
                                                        const TF* __restrict__ dzi, const TF* __restrict__ dzhi,
                                                        TF dxidxi, TF dyidyi, Gd g)
    {
        int i, j, k;
        if (!point(g, g.kstart+1, i, j, k)) return;
        const int jj = g.icells, kk = g.ijcells, ijk = i + j*jj + k*kk;
        wt[ijk] += diff_2_pt(Gacc2<TF>{w, ijk, jj, kk}, visc, dxidxi, dyidyi, dzhi[k], dzi[k-1], dzi[k]);
    }

    template<typename TF> TF*& mlen_ptr(mhh_ctx* c);
    template<> double*& mlen_ptr<double>(mhh_ctx* c) { return c->mlen_d; }
    template<> float*& mlen_ptr<float>(mhh_ctx* c) { return c->mlen_f; }

    template<typename TF>
    int ensure_mlen(mhh_ctx* c, double cs)
    {
        TF*& dev = mlen_ptr<TF>(c);
        if (dev && c->mlen_cs == cs) return 0;
        const Gd& g = c->gd;
        // mlen0 = cs*(dx*dy*dz)^(1/3) in the element type (src/diff_smag2.cxx:163, 214, 240).
        std::vector<TF> h(g.kcells, TF(0));
        for (int k = g.kstart; k < g.kend; ++k)
            h[k] = TF(cs)*std::pow(TF(g.dx)*TF(g.dy)*TF(c->h_dz[k]), TF(1./3.));
        if (!dev)
            MHH_CHECK(check_hip(hipMalloc(&dev, sizeof(TF)*g.kcells), "hipMalloc(mlen)"));
        MHH_CHECK(check_hip(hipMemcpy(dev, h.data(), sizeof(TF)*g.kcells, hipMemcpyHostToDevice), "hipMemcpy(mlen)"));
        c->mlen_cs = cs;
        return 0;
    }

    template<typename TF>
    const TF* dptr(void* p) { return static_cast<const TF*>(p); }

    // lim: also leave the CFL-rate and dnmul block maxima in the reduction
    // buffer (c->red[1..*nred] and c->red[*nred+2 ..]); no surface model only.
    template<typename TF>
    int viscosity(mhh_ctx* c, const Prof<TF>& p, const mhh_smag_params& par, bool lim = false, int* nred = nullptr)
    {
        const Gd& g = c->gd;
        if (par.thermo && (c->f.nscalars < 1 || !p.thref))
            return fail(MHH_ESTATE, "smag2 with thermo needs scalar 0 (th) and mhh_set_base_state()");
        if (par.surface_model && (!c->f.z0m || !c->f.dudz || !c->f.dvdz || (par.thermo && !c->f.dbdz)))
            return fail(MHH_ESTATE, "smag2 with a surface model needs dudz, dvdz, dbdz and z0m bound");
        MHH_CHECK(ensure_mlen<TF>(c, par.cs));

        Visc_args<TF> a;
        a.evisc = static_cast<TF*>(c->f.evisc);
        a.u = dptr<TF>(c->f.u); a.v = dptr<TF>(c->f.v); a.w = dptr<TF>(c->f.w);
        a.th = par.thermo ? dptr<TF>(c->f.s[0]) : nullptr;
        a.dudz = dptr<TF>(c->f.dudz); a.dvdz = dptr<TF>(c->f.dvdz);
        a.dbdz = dptr<TF>(c->f.dbdz); a.z0m = dptr<TF>(c->f.z0m);
        a.z = p.z; a.dzi = p.dzi; a.dzhi = p.dzhi; a.thref = p.thref;
        a.mlen0 = mlen_ptr<TF>(c);
        a.dxi = TF(1.)/TF(g.dx); a.dyi = TF(1.)/TF(g.dy);
        a.tPr = TF(par.tPr); a.visc = TF(par.visc);
        a.zsize = TF(c->h_zh[g.kend]);

        const bool sfc = par.surface_model != 0, th = par.thermo != 0, ms = par.swmason != 0;
        if (lim && sfc)
            return fail(MHH_EINVAL, "the fused time-step limits cover the default boundary only");
        // plane-ring kernel; with `limits` also the CFL and dnmul maxima
        const int nti = (g.itot + VTX - 1)/VTX, ntj = (g.jtot + VTY - 1)/VTY;
        const int kchunk = c->visc_kchunk > 0 ? c->visc_kchunk
                         : march_kchunk(c, nti*ntj, g.ktot, MARCH_LEAST_VISC, visc_most(sizeof(TF) == 8, lim, sfc, ms));
        const int nkc = (g.ktot + kchunk - 1)/kchunk;
        // the wall mirror and the cyclic update of the pass done inside it where
        // every ghost column is one periodic image and kgc = 1
        const int halo = g.itot >= 2*g.igc && g.jtot >= 2*g.jgc && g.kgc == 1;
        const int nblocks = (nti*ntj*nkc + 7)/8*8;
        double* rc = nullptr; double* rd = nullptr;
        if (lim)
        {
            MHH_CHECK(ensure_reduction(c, 2*nblocks + 1));
            rc = c->red; rd = c->red + nblocks + 1;
        }
        if (!p.lev)
            return fail(MHH_ESTATE, "the viscosity needs the grid profiles");
        Visc_scalars<TF> vs;
        vs.dxi = a.dxi; vs.dyi = a.dyi; vs.tPr_i = TF(1)/TF(par.tPr); vs.visc = a.visc; vs.zsize = a.zsize;
        vs.tPrfac_i = TF(1)/std::min(TF(1.), TF(par.tPr));
        vs.dxidxi = TF(1.)/(TF(g.dx)*TF(g.dx)); vs.dyidyi = TF(1.)/(TF(g.dy)*TF(g.dy));
        const Visc_surface<TF> sf{a.dudz, a.dvdz, a.dbdz, a.z0m};
        const dim3 vb(VTX, VTY);
        const TF* ml = mlen_ptr<TF>(c);
        {
            mhh::Timer _t(c, "evisc");
#define MHH_VISC_LAUNCH(T, L, S) launch(c, visc_tile_k<TF, T, L, S>{ \
                a.evisc, a.u, a.v, a.w, a.th, p.lev, ml, p.z, vs, g, nti, ntj, nkc, kchunk, halo, rc, rd, sf}, nblocks, vb)
            if (sfc && th && ms)  MHH_VISC_LAUNCH(true, false, 2);
            else if (sfc && th)   MHH_VISC_LAUNCH(true, false, 1);
            else if (sfc && ms)   MHH_VISC_LAUNCH(false, false, 2);
            else if (sfc)         MHH_VISC_LAUNCH(false, false, 1);
            else if (th && lim)   MHH_VISC_LAUNCH(true, true, 0);
            else if (th)          MHH_VISC_LAUNCH(true, false, 0);
            else if (lim)         MHH_VISC_LAUNCH(false, true, 0);
            else                  MHH_VISC_LAUNCH(false, false, 0);
#undef MHH_VISC_LAUNCH
        }
        if (lim) *nred = nblocks;
        MHH_CHECK(check_launch("evisc"));
        if (halo) return 0;

        if (!sfc)
        {
            const dim3 b2(64, 4), g2((g.itot + 63)/64, (g.jtot + 3)/4);
            { mhh::Timer _t(c, "mirror_walls"); launch(c, mirror_walls_k<TF>{a.evisc, g}, g2, b2); }
            MHH_CHECK(check_launch("mirror_walls"));
        }
        return mhh::cyclic_field(c, c->f.evisc, MHH_EDGE_BOTH);
    }

    template<typename TF>
    int diffuse(mhh_ctx* c, const Prof<TF>& p, const mhh_smag_params& par)
    {
        const Gd& g = c->gd;
        const bool sfc = par.surface_model != 0;
        if (sfc)
        {
            if (!c->f.u_fluxbot || !c->f.u_fluxtop || !c->f.v_fluxbot || !c->f.v_fluxtop)
                return fail(MHH_ESTATE, "smag2 with a surface model needs the u and v flux planes bound");
            for (int n = 0; n < c->f.nscalars; ++n)
                if (!c->f.s_fluxbot[n] || !c->f.s_fluxtop[n])
                    return fail(MHH_ESTATE, "smag2 with a surface model needs the scalar flux planes bound");
        }
        Diff_args<TF> a{};
        a.u = dptr<TF>(c->f.u); a.v = dptr<TF>(c->f.v); a.w = dptr<TF>(c->f.w);
        a.evisc = dptr<TF>(c->f.evisc);
        a.dzi = p.dzi; a.dzhi = p.dzhi; a.rho = p.rhoref; a.rhoh = p.rhorefh;
        a.dxi = TF(1.)/TF(g.dx); a.dyi = TF(1.)/TF(g.dy);
        a.dxidxi = TF(1./(g.dx*g.dx)); a.dyidyi = TF(1./(g.dy*g.dy));
        a.visc = TF(par.visc); a.tPr = TF(par.tPr);
        const dim3 blk(BX, BY);

        a.at = static_cast<TF*>(c->f.ut); a.fluxbot = dptr<TF>(c->f.u_fluxbot); a.fluxtop = dptr<TF>(c->f.u_fluxtop);
        if (sfc) { mhh::Timer _t(c, "diff_u"); diff_u_g<TF, true><<<grid3(g, g.kstart, g.kend), blk, 0, c->stream>>>(a, g); }
        else     { mhh::Timer _t(c, "diff_u"); diff_u_g<TF, false><<<grid3(g, g.kstart, g.kend), blk, 0, c->stream>>>(a, g); }

        a.at = static_cast<TF*>(c->f.vt); a.fluxbot = dptr<TF>(c->f.v_fluxbot); a.fluxtop = dptr<TF>(c->f.v_fluxtop);
        if (sfc) { mhh::Timer _t(c, "diff_v"); diff_v_g<TF, true><<<grid3(g, g.kstart, g.kend), blk, 0, c->stream>>>(a, g); }
        else     { mhh::Timer _t(c, "diff_v"); diff_v_g<TF, false><<<grid3(g, g.kstart, g.kend), blk, 0, c->stream>>>(a, g); }

        a.at = static_cast<TF*>(c->f.wt);
        { mhh::Timer _t(c, "diff_w"); diff_w_g<TF><<<grid3(g, g.kstart+1, g.kend), blk, 0, c->stream>>>(a, g); }

        for (int n = 0; n < c->f.nscalars; ++n)
        {
            a.at = static_cast<TF*>(c->f.st[n]); a.a = dptr<TF>(c->f.s[n]);
            a.fluxbot = dptr<TF>(c->f.s_fluxbot[n]); a.fluxtop = dptr<TF>(c->f.s_fluxtop[n]);
            a.visc = TF(par.svisc[n]);
            if (sfc) { mhh::Timer _t(c, "diff_c"); diff_c_g<TF, true><<<grid3(g, g.kstart, g.kend), blk, 0, c->stream>>>(a, g); }
            else     { mhh::Timer _t(c, "diff_c"); diff_c_g<TF, false><<<grid3(g, g.kstart, g.kend), blk, 0, c->stream>>>(a, g); }
        }
        return check_launch("diff_smag2");
    }

    template<typename TF>
    int dnmul(mhh_ctx* c, const Prof<TF>& p, double tPr, double* out)
    {
        const Gd& g = c->gd;
        const dim3 grd = grid_red(g);
        const int nb = static_cast<int>(grd.x*grd.y*grd.z);
        MHH_CHECK(ensure_reduction(c, nb));
        const TF dxi = TF(1.)/TF(g.dx), dyi = TF(1.)/TF(g.dy);
        { mhh::Timer _t(c, "dnmul"); dnmul_g<TF><<<grd, dim3(BX, BY), 0, c->stream>>>(dptr<TF>(c->f.evisc), p.dzi,
                TF(1.)/(TF(g.dx)*TF(g.dx)), TF(1.)/(TF(g.dy)*TF(g.dy)), TF(1)/std::min(TF(1.), TF(tPr)), g, c->red); }
        (void)dxi; (void)dyi;
        MHH_CHECK(check_launch("dnmul"));
        return reduce_max_partials(c, nb, out);
    }

    template<typename TF>
    int diff_2(mhh_ctx* c, const Prof<TF>& p, double visc, const double* svisc)
    {
        const Gd& g = c->gd;
        const TF dxidxi = TF(1/(g.dx*g.dx)), dyidyi = TF(1/(g.dy*g.dy));
        const dim3 blk(BX, BY);
        { mhh::Timer _t(c, "diff_2"); diff_2_c_g<TF><<<grid3(g, g.kstart, g.kend), blk, 0, c->stream>>>(static_cast<TF*>(c->f.ut), dptr<TF>(c->f.u),
                TF(visc), p.dzi, p.dzhi, dxidxi, dyidyi, g); }
        { mhh::Timer _t(c, "diff_2"); diff_2_c_g<TF><<<grid3(g, g.kstart, g.kend), blk, 0, c->stream>>>(static_cast<TF*>(c->f.vt), dptr<TF>(c->f.v),
                TF(visc), p.dzi, p.dzhi, dxidxi, dyidyi, g); }
        { mhh::Timer _t(c, "diff_2"); diff_2_w_g<TF><<<grid3(g, g.kstart+1, g.kend), blk, 0, c->stream>>>(static_cast<TF*>(c->f.wt), dptr<TF>(c->f.w),
                TF(visc), p.dzi, p.dzhi, dxidxi, dyidyi, g); }
        for (int n = 0; n < c->f.nscalars; ++n)
            { mhh::Timer _t(c, "diff_2"); diff_2_c_g<TF><<<grid3(g, g.kstart, g.kend), blk, 0, c->stream>>>(static_cast<TF*>(c->f.st[n]),
                    dptr<TF>(c->f.s[n]), TF(svisc ? svisc[n] : visc), p.dzi, p.dzhi, dxidxi, dyidyi, g); }
        return check_launch("diff_2");
    }
}

namespace mhh
{
    int smag_prepare(mhh_ctx* c, const mhh_smag_params& par)
    {
        return c->precision == MHH_FP64 ? ensure_mlen<double>(c, par.cs) : ensure_mlen<float>(c, par.cs);
    }
}

extern "C" {

int mhh_diff_smag2_exec_viscosity(mhh_ctx* c, const mhh_smag_params* par)
{
    MHH_REQUIRE_BOUND(c);
    if (!par) return mhh::fail(MHH_EINVAL, "null smag params");
    if (!c->f.evisc) return mhh::fail(MHH_ESTATE, "evisc field is not bound");
    return c->precision == MHH_FP64 ? viscosity<double>(c, c->pd, *par) : viscosity<float>(c, c->pf, *par);
}

int mhh_diff_smag2_exec_viscosity_limits(mhh_ctx* c, const mhh_smag_params* par, double* cfl_rate, double* dnmul)
{
    MHH_REQUIRE_BOUND(c);
    if (!par || !cfl_rate || !dnmul) return mhh::fail(MHH_EINVAL, "null argument");
    if (!c->f.evisc) return mhh::fail(MHH_ESTATE, "evisc field is not bound");
    if (par->surface_model) return mhh::fail(MHH_EINVAL, "the fused time-step limits cover the default boundary only");
    if (c->gd.igc < 3 || c->gd.jgc < 3) return mhh::fail(MHH_EINVAL, "the 2i5 CFL needs igc = jgc >= 3");
    int nb = 0;
    if (c->precision == MHH_FP64) MHH_CHECK(viscosity<double>(c, c->pd, *par, true, &nb));
    else MHH_CHECK(viscosity<float>(c, c->pf, *par, true, &nb));
    MHH_CHECK(mhh::reduce_max_partials_at(c, c->red, nb, cfl_rate));
    return mhh::reduce_max_partials_at(c, c->red + nb + 1, nb, dnmul);
}

int mhh_diff_smag2_exec(mhh_ctx* c, const mhh_smag_params* par)
{
    MHH_REQUIRE_BOUND(c);
    MHH_NOT_IN_BATCH(c, "mhh_diff_smag2_exec");
    MHH_CHECK(mhh::settle_tendencies(c));
    if (!par) return mhh::fail(MHH_EINVAL, "null smag params");
    if (!c->f.evisc) return mhh::fail(MHH_ESTATE, "evisc field is not bound");
    return c->precision == MHH_FP64 ? diffuse<double>(c, c->pd, *par) : diffuse<float>(c, c->pf, *par);
}

int mhh_diff_smag2_dnmul(mhh_ctx* c, double tPr, double* out)
{
    MHH_REQUIRE_BOUND(c);
    MHH_NOT_IN_BATCH(c, "mhh_diff_smag2_dnmul");
    if (!out) return mhh::fail(MHH_EINVAL, "null output");
    if (!c->f.evisc) return mhh::fail(MHH_ESTATE, "evisc field is not bound");
    return c->precision == MHH_FP64 ? dnmul<double>(c, c->pd, tPr, out) : dnmul<float>(c, c->pf, tPr, out);
}

int mhh_diff_2_exec(mhh_ctx* c, double visc, const double* svisc)
{
    MHH_REQUIRE_BOUND(c);
    MHH_NOT_IN_BATCH(c, "mhh_diff_2_exec");
    MHH_CHECK(mhh::settle_tendencies(c));
    return c->precision == MHH_FP64 ? diff_2<double>(c, c->pd, visc, svisc) : diff_2<float>(c, c->pf, visc, svisc);
}

} // extern "C"
