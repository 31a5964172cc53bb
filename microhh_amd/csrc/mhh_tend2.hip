// mhh_tend2.hip -- fused tendency of the 2nd-order operators: Advec_2::exec
// (src/advec_2.cxx:82-202) and Diff_2::exec (src/diff_2.cxx:39-85) of u, v, w
// and scalar 0 in one pass, each tendency taking the advection and then the
// diffusion, the order of the reference driver (src/model.cxx:388-414).  The
// expressions are those of the one-point kernels (advec_2_*_pt, diff_2_pt).
//
// Layout of the work, as in the fused 2i5 pass: a block owns a 64 x 4 column
// tile and marches up a chunk of levels; at level k the LDS holds
//     u, v at k-1 and k,  w at k and k+1,  s at k      (halo 1 in x and y)
// rotating as k advances, so every plane is read from HBM once per chunk;
// the own column's u, v, s at k+1 are loaded beside the planes of level k+1
// (the same cache lines), w and s at k-1 are carried from the level below.
#include <algorithm>

#include "mhh_batch.h"
#include "mhh_stencil.h"

namespace
{
    using namespace mhh;

    constexpr int TX = 64, TY = 4;
    constexpr int PW = TX + 2, PH = TY + 2, PN = PW*PH;
    constexpr int NQ = (PN + TX*TY - 1)/(TX*TY);

    template<typename TF>
    struct Tend2_args
    {
        TF dxi, dyi, dxidxi, dyidyi, visc, svisc;
        int nti, ntj, nkc, kchunk;
    };

    // A field at offsets from the point: the plane at k (dk = 0) or k-1
    // (dk = -1) in LDS, the own column at k+1 from a register.
    template<typename TF>
    struct Lacc
    {
        const TF* cur; const TF* below; TF up; int c;
        __device__ __forceinline__ TF operator()(int di, int dj, int dk) const
        {
            return dk == 0 ? cur[c + di + dj*PW] : dk < 0 ? below[c + di + dj*PW] : up;
        }
    };

    // w: the planes at k (dk = 0) and k+1 (dk = 1), the own column at k-1.
    template<typename TF>
    struct Wacc
    {
        const TF* cur; const TF* above; TF down; int c;
        __device__ __forceinline__ TF operator()(int di, int dj, int dk) const
        {
            return dk == 0 ? cur[c + di + dj*PW] : dk > 0 ? above[c + di + dj*PW] : down;
        }
    };

    // s: the plane at k, the own column at k-1 and k+1.
    template<typename TF>
    struct Sacc
    {
        const TF* cur; TF down, up; int c;
        __device__ __forceinline__ TF operator()(int di, int dj, int dk) const
        {
            return dk == 0 ? cur[c + di + dj*PW] : dk < 0 ? down : up;
        }
    };

    template<typename TF>
    __device__ __forceinline__ void plane_load(TF* __restrict__ dst, const TF* __restrict__ src, int k, const int (&o)[NQ],
                                               int tid, const Gd& g)
    {
        const TF* __restrict__ sk = src + static_cast<size_t>(k)*g.ijcells;
        #pragma unroll
        for (int q = 0; q < NQ; ++q)
        {
            const int idx = tid + q*TX*TY;
            if (idx < PN) dst[idx] = o[q] >= 0 ? sk[o[q]] : TF(0);
        }
    }

    template<typename TF>
    __device__ __forceinline__ TF ldo(const TF* __restrict__ base, uint32_t off)
    {
        return *reinterpret_cast<const TF*>(reinterpret_cast<const char*>(base) + off);
    }

    template<typename TF>
    __device__ __forceinline__ void plane_fetch(TF (&r)[NQ], const TF* __restrict__ src, int k, const uint32_t (&ob)[NQ],
                                                const Gd& g)
    {
        const TF* __restrict__ sk = src + static_cast<size_t>(k)*g.ijcells;
        #pragma unroll
        for (int q = 0; q < NQ; ++q) r[q] = ldo(sk, ob[q]);
    }

    template<typename TF>
    __device__ __forceinline__ void plane_store(TF* __restrict__ dst, const TF (&r)[NQ], int tid)
    {
        #pragma unroll
        for (int q = 0; q < NQ-1; ++q) dst[tid + q*TX*TY] = r[q];
        const int idx = tid + (NQ-1)*TX*TY;
        if (idx < PN) dst[idx] = r[NQ-1];
    }

    // NS: scalar 0 in the pass (0 or 1).
    template<typename TF, int NS>
    __device__ __forceinline__ void tend_2_g(TF* __restrict__ ut, TF* __restrict__ vt, TF* __restrict__ wt,
                                             TF* __restrict__ st, const TF* __restrict__ u, const TF* __restrict__ v,
                                             const TF* __restrict__ w, const TF* __restrict__ s,
                                             const Level<TF>* __restrict__ lev, Tend2_args<TF> a, Gd g,
                                             const Bid& bid_)
    {
        __shared__ __align__(16) TF lds[(6 + NS)*PN];
        const int ntiles = a.nti*a.ntj*a.nkc;
        const int tile = xcd_tile(bid_.x, bid_.nx);
        if (tile >= ntiles) return;
        const int ti = tile % a.nti, tj = (tile / a.nti) % a.ntj, kc = tile / (a.nti*a.ntj);
        const int tid = threadIdx.x + TX*threadIdx.y;
        const int i0 = g.istart + ti*TX, j0 = g.jstart + tj*TY;
        const int i = i0 + threadIdx.x, j = j0 + threadIdx.y;
        const bool active = i < g.iend && j < g.jend;
        const int kb = g.kstart + kc*a.kchunk, ke = min(kb + a.kchunk, g.kend);
        const size_t kk = g.ijcells;
        // threads outside the domain compute on the clamped column and store nothing
        const int ij = min(i, g.iend-1) + min(j, g.jend-1)*g.icells;
        const uint32_t oij = uint32_t(ij)*sizeof(TF);

        int o[NQ];
        uint32_t ob[NQ];
        #pragma unroll
        for (int q = 0; q < NQ; ++q)
        {
            const int idx = tid + q*TX*TY;
            const int pj = idx / PW, pi = idx - pj*PW;
            const int gi = i0 - 1 + pi, gj = j0 - 1 + pj;
            o[q] = (idx < PN && gi < g.icells && gj < g.jcells) ? gi + gj*g.icells : -1;
            ob[q] = o[q] >= 0 ? uint32_t(o[q])*sizeof(TF) : 0u;
        }
        TF* Up = lds;        TF* Uc = Up + PN;
        TF* Vp = Uc + PN;    TF* Vc = Vp + PN;
        TF* Wc = Vc + PN;    TF* Wn = Wc + PN;
        TF* Sc = Wn + PN;    // NS = 1 only
        plane_load(Up, u, kb-1, o, tid, g); plane_load(Uc, u, kb, o, tid, g);
        plane_load(Vp, v, kb-1, o, tid, g); plane_load(Vc, v, kb, o, tid, g);
        plane_load(Wc, w, kb, o, tid, g);   plane_load(Wn, w, kb+1, o, tid, g);
        if (NS) plane_load(Sc, s, kb, o, tid, g);
        // own column: w and s one level down
        TF wm = ldo(w + size_t(kb-1)*kk, oij);
        TF sm = NS ? ldo(s + size_t(kb-1)*kk, oij) : TF(0);
        const Level<TF> Lb = ld_const(lev, kb-1);
        TF rhom = Lb.rho, dzim = Lb.dzi;     // rhoref and dzi one level down
        const int c = (threadIdx.y + 1)*PW + (threadIdx.x + 1);
        TF ru[NQ], rv[NQ], rw[NQ], rs[NQ];
        __syncthreads();

        for (int k = kb; k < ke; ++k)
        {
            const size_t kofs = size_t(k)*kk;
            // the tendencies of this level, the own column one level up, then
            // the planes of the next level (in flight until its end)
            TF tu = ldo(ut + kofs, oij), tv = ldo(vt + kofs, oij), tw = ldo(wt + kofs, oij);
            TF ts = NS ? ldo(st + kofs, oij) : TF(0);
            const int k1 = min(k + 1, g.kcells - 1), k2 = min(k + 2, g.kcells - 1);
            const TF un = ldo(u + size_t(k1)*kk, oij), vn = ldo(v + size_t(k1)*kk, oij);
            const TF sn = NS ? ldo(s + size_t(k1)*kk, oij) : TF(0);
            __builtin_amdgcn_sched_barrier(0);
            plane_fetch(ru, u, k1, ob, g);
            plane_fetch(rv, v, k1, ob, g);
            plane_fetch(rw, w, k2, ob, g);
            if (NS) plane_fetch(rs, s, k1, ob, g);

            const Level<TF> L = ld_const(lev, k);
            const Lacc<TF> U{Uc, Up, un, c}, V{Vc, Vp, vn, c};
            const Wacc<TF> W{Wc, Wn, wm, c};
            // the u, v of w's stencil at k-1 and k are the planes below and at k
            tu += advec_2_u_pt(U, V, W, L.rho, L.rhoh, L.rhohp, a.dxi, a.dyi, L.dzi);
            tu += diff_2_pt(U, a.visc, a.dxidxi, a.dyidyi, L.dzi, L.dzhi, L.dzhip);
            tv += advec_2_v_pt(U, V, W, L.rho, L.rhoh, L.rhohp, a.dxi, a.dyi, L.dzi);
            tv += diff_2_pt(V, a.visc, a.dxidxi, a.dyidyi, L.dzi, L.dzhi, L.dzhip);
            if (k > g.kstart)
            {
                tw += advec_2_w_pt(U, V, W, rhom, L.rho, L.rhoh, a.dxi, a.dyi, L.dzhi);
                tw += diff_2_pt(W, a.visc, a.dxidxi, a.dyidyi, L.dzhi, dzim, L.dzi);
            }
            if (NS)
            {
                const Sacc<TF> S{Sc, sm, sn, c};
                ts += advec_2_s_pt(U, V, W, S, L.rho, L.rhoh, L.rhohp, a.dxi, a.dyi, L.dzi);
                ts += diff_2_pt(S, a.svisc, a.dxidxi, a.dyidyi, L.dzi, L.dzhi, L.dzhip);
            }
            if (active)
            {
                *reinterpret_cast<TF*>(reinterpret_cast<char*>(ut + kofs) + oij) = tu;
                *reinterpret_cast<TF*>(reinterpret_cast<char*>(vt + kofs) + oij) = tv;
                if (k > g.kstart) *reinterpret_cast<TF*>(reinterpret_cast<char*>(wt + kofs) + oij) = tw;
                if (NS) *reinterpret_cast<TF*>(reinterpret_cast<char*>(st + kofs) + oij) = ts;
            }
            wm = Wc[c];
            if (NS) sm = Sc[c];
            rhom = L.rho; dzim = L.dzi;
            __syncthreads();
            // rotate the ring and store the prefetched planes
            TF* x;
            x = Up; Up = Uc; Uc = x;
            x = Vp; Vp = Vc; Vc = x;
            x = Wc; Wc = Wn; Wn = x;
            plane_store(Uc, ru, tid);
            plane_store(Vc, rv, tid);
            plane_store(Wn, rw, tid);
            if (NS) plane_store(Sc, rs, tid);
            __syncthreads();
        }
    }

    template<typename TF, int NS>
    struct tend_2_k
    {
        static constexpr int NT = TX*TY, MINB = 0;
        TF* ut; TF* vt; TF* wt; TF* st; const TF* u; const TF* v; const TF* w; const TF* s;
        const Level<TF>* lev; Tend2_args<TF> a; Gd g;
        __device__ __forceinline__ void operator()(const Bid& bid_) const
        {
            tend_2_g<TF, NS>(ut, vt, wt, st, u, v, w, s, lev, a, g, bid_);
        }
    };

    template<typename TF>
    int tend2(mhh_ctx* c, const Prof<TF>& p, double visc, double svisc)
    {
        const Gd& g = c->gd;
        if (!p.lev)
            return fail(MHH_ESTATE, "the fused 2nd-order tendency needs the grid profiles");
        Tend2_args<TF> a{};
        a.dxi = TF(1.)/TF(g.dx); a.dyi = TF(1.)/TF(g.dy);
        a.dxidxi = TF(1/(g.dx*g.dx)); a.dyidyi = TF(1/(g.dy*g.dy));
        a.visc = TF(visc); a.svisc = TF(svisc);
        a.nti = (g.itot + TX - 1)/TX;
        a.ntj = (g.jtot + TY - 1)/TY;
        a.kchunk = c->tend_kchunk > 0 ? c->tend_kchunk : march_kchunk(c, a.nti*a.ntj, g.ktot, MARCH_LEAST_TEND);
        a.nkc = (g.ktot + a.kchunk - 1)/a.kchunk;
        const int nblocks = xcd_blocks(a.nti*a.ntj*a.nkc);
        const int ns = c->f.nscalars > 0 ? 1 : 0;
        TF* st = ns ? static_cast<TF*>(c->f.st[0]) : nullptr;
        const TF* s = ns ? static_cast<const TF*>(c->f.s[0]) : nullptr;
        {
            mhh::Timer _t(c, "tend_2");
            TF* ut = static_cast<TF*>(c->f.ut); TF* vt = static_cast<TF*>(c->f.vt); TF* wt = static_cast<TF*>(c->f.wt);
            const TF* u = static_cast<const TF*>(c->f.u); const TF* v = static_cast<const TF*>(c->f.v);
            const TF* w = static_cast<const TF*>(c->f.w);
            if (ns) launch(c, tend_2_k<TF, 1>{ut, vt, wt, st, u, v, w, s, p.lev, a, g}, nblocks, dim3(TX, TY));
            else    launch(c, tend_2_k<TF, 0>{ut, vt, wt, st, u, v, w, s, p.lev, a, g}, nblocks, dim3(TX, TY));
        }
        return check_launch("tend_2");
    }
}

extern "C" int mhh_tendency_2_2(mhh_ctx* c, double visc, const double* svisc)
{
    MHH_REQUIRE_BOUND(c);
    if (c->f.nscalars > 1) return mhh::fail(MHH_EINVAL, "mhh_tendency_2_2 covers u, v, w and scalar 0 only");
    MHH_CHECK(mhh::settle_tendencies(c));
    const double sv0 = svisc ? svisc[0] : visc;
    return c->precision == MHH_FP64 ? tend2<double>(c, c->pd, visc, sv0) : tend2<float>(c, c->pf, visc, sv0);
}
