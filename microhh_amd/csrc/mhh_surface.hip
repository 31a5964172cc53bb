// mhh_surface.hip -- the Monin-Obukhov surface layer of the "surface" boundary
// switch (Boundary_surface, src/boundary_surface.cxx:54-339, 703-990;
// include/boundary_surface_kernels.h; include/monin_obukhov.h) and the buffer
// sponge (Buffer, src/buffer.cxx:38-58, 101-185).
//
// The surface layer works on planes (icells x jcells): one thread per column,
// a few launches per substep (wind difference, stability, momentum and scalar
// fluxes, MO gradients).  The Obukhov length comes either from the lookup
// table of init_solver, searched from each column's previous crossing as the
// reference does, or from the Newton iteration of the iterative solver.
#include <algorithm>
#include <cmath>
#include <vector>

#include "mhh_batch.h"

struct mhh_surface_state
{
    mhh_surface_desc desc{};
    int nzl = 10000;                 // nzL_lut, include/boundary.h:56
    float* zl = nullptr;             // lookup table z/L and its evaluation function
    float* fl = nullptr;
    int* nobuk = nullptr;            // per column: the table index of the last crossing
    void* ustar = nullptr; void* obuk = nullptr; void* z0h = nullptr;
    void* dutot = nullptr; void* bflux = nullptr; void* b = nullptr; void* bbot = nullptr;
    double db_ref = 0.;
};

struct mhh_buffer_state
{
    mhh_buffer_desc desc{};
    int kb = 0, kbh = 0;             // first buffer level of the cell centres and of the faces
    int ndamped = 0;                 // u, v, w and the first ndamped-3 scalars
    double* prof = nullptr;          // (3 + MHH_MAX_SCALARS) x kcells reference profiles (FP64)
    double* part = nullptr;          // swupdate: partial plane sums of the damped fields
    void* sig_c = nullptr;           // kcells: sigma ((z - zstart)/(zsize - zstart))^beta, 0 below the buffer
    void* sig_h = nullptr;           // the same at the half levels (w)
};

namespace
{
    using namespace mhh;

    constexpr double kappa = 0.4;    // include/constants.h:28
    constexpr double grav = 9.81;    // include/constants.h:29
    constexpr double zL_max = 10., zL_min = -1.e4;
    constexpr double dsmall = 1.e-9, dbig = 1.e9, dhuge = 1.e30;

    // ------------------------------------------------ include/monin_obukhov.h
    // Wilson (2001) for unstable, IFS (Beljaars and Holtslag 1991) for stable
    // stratification.
    template<typename TF> __host__ __device__ TF phim_unstable(TF zeta)
    { return std::pow(TF(1.) + TF(3.6)*std::pow(std::fabs(zeta), TF(2./3.)), TF(-1./2.)); }
    template<typename TF> __host__ __device__ TF phih_unstable(TF zeta)
    { return std::pow(TF(1.) + TF(7.9)*std::pow(std::fabs(zeta), TF(2./3.)), TF(-1./2.)); }
    template<typename TF> __host__ __device__ TF phim(TF zeta)
    { return zeta <= TF(0.) ? phim_unstable(zeta) : TF(1) + TF(5)*zeta; }
    template<typename TF> __host__ __device__ TF phih(TF zeta)
    { const TF a = TF(1) + TF(4)*zeta; return zeta <= TF(0.) ? phih_unstable(zeta) : a*a; }
    template<typename TF> __host__ __device__ TF psim_unstable(TF zeta)
    { return TF(3.)*std::log((TF(1.) + TF(1.)/phim_unstable(zeta))/TF(2.)); }
    template<typename TF> __host__ __device__ TF psih_unstable(TF zeta)
    { return TF(3.)*std::log((TF(1.) + TF(1.)/phih_unstable(zeta))/TF(2.)); }
    template<typename TF> __host__ __device__ TF psim_stable(TF zeta)
    {
        const TF a = TF(1), b = TF(2)/TF(3), c = TF(5), d = TF(0.35);
        return -b*(zeta - (c/d))*std::exp(-d*zeta) - a*zeta - (b*c)/d;
    }
    template<typename TF> __host__ __device__ TF psih_stable(TF zeta)
    {
        const TF a = TF(1), b = TF(2)/TF(3), c = TF(5), d = TF(0.35);
        return -b*(zeta - (c/d))*std::exp(-d*zeta) - std::pow(TF(1) + b*a*zeta, TF(1.5)) - (b*c)/d + TF(1);
    }
    template<typename TF> __host__ __device__ TF most_fm(TF zsl, TF z0m, TF L)
    {
        return L <= TF(0.)
            ? TF(kappa) / (std::log(zsl/z0m) - psim_unstable(zsl/L) + psim_unstable(z0m/L))
            : TF(kappa) / (std::log(zsl/z0m) - psim_stable(zsl/L) + psim_stable(z0m/L));
    }
    template<typename TF> __host__ __device__ TF most_fh(TF zsl, TF z0h, TF L)
    {
        return L <= TF(0.)
            ? TF(kappa) / (std::log(zsl/z0h) - psih_unstable(zsl/L) + psih_unstable(z0h/L))
            : TF(kappa) / (std::log(zsl/z0h) - psih_stable(zsl/L) + psih_stable(z0h/L));
    }

    // Lookup table of init_solver (include/boundary_surface_kernels.h:80-132),
    // on the host in the element type, stored in single precision.
    template<typename TF>
    void prepare_lut(std::vector<float>& zl, std::vector<float>& fl, TF z0m, TF z0h, TF zsl, int nzl,
                     int mbcbot, int thermobc)
    {
        std::vector<TF> tmp(nzl);
        const TF zLrange_min = -5.;
        TF dzL = (TF(zL_max) - zLrange_min) / (9.*nzl/10. - 1.);
        tmp[0] = -TF(zL_max);
        for (int n = 1; n < 9*nzl/10; ++n) tmp[n] = tmp[n-1] + dzL;
        // the last tenth stretched geometrically down to the free-convection limit
        const TF zLend = -(TF(zL_min) - zLrange_min);
        TF r = 1.01, r0 = TF(dhuge);
        while (std::abs((r-r0)/r0) > 1.e-10)
        {
            r0 = r;
            r = std::pow(1. - (zLend/dzL)*(1.-r), (1./(nzl/10.)));
        }
        for (int n = 9*nzl/10; n < nzl; ++n) { tmp[n] = tmp[n-1] + dzL; dzL *= r; }
        zl.resize(nzl); fl.assign(nzl, 0.f);
        for (int n = 0; n < nzl; ++n) zl[n] = static_cast<float>(-tmp[nzl-n-1]);
        if (mbcbot == MHH_BC_DIRICHLET && thermobc == MHH_BC_FLUX)
            for (int n = 0; n < nzl; ++n)
                fl[n] = static_cast<float>(zl[n] * std::pow(most_fm<TF>(zsl, z0m, zsl/zl[n]), 3));
        else if (mbcbot == MHH_BC_DIRICHLET && thermobc == MHH_BC_DIRICHLET)
            for (int n = 0; n < nzl; ++n)
                fl[n] = static_cast<float>(zl[n] * std::pow(most_fm<TF>(zsl, z0m, zsl/zl[n]), 2)
                                           / most_fh<TF>(zsl, z0h, zsl/zl[n]));
    }

    // The table's crossing by Ri, searched from the column's previous one, and
    // the single-precision interpolation between the two entries
    // (include/boundary_surface_kernels.h:243-259).  The bound is tested
    // before the entry below is read.
    __device__ float find_zL(const float* __restrict__ zl, const float* __restrict__ fl, int& n, int nzl, float Ri)
    {
        #pragma clang fp contract(off)
        if ((fl[n] - Ri) > 0.f)
            while (n > 0 && (fl[n-1] - Ri) > 0.f) --n;
        else
            while ((fl[n] - Ri) < 0.f && n < nzl-1) ++n;
        if (n == 0 || n == nzl-1) return zl[n];
        return zl[n-1] + (Ri - fl[n-1]) / (fl[n] - fl[n-1]) * (zl[n] - zl[n-1]);
    }

    // Newton iterations of the iterative solvers
    // (include/boundary_surface_kernels.h:275-436).
    template<typename TF>
    __host__ __device__ TF obuk_flux_iterative(TF L, TF du, TF bfluxbot, TF zsl, TF z0m)
    {
        // the roundings of the reference's expressions (no fused multiply-adds):
        // the finite-difference Newton step magnifies every last-bit change
        #pragma clang fp contract(off)
        TF L0, Lstart, Lend, fx, fxdif;
        int m = 0, nlim = 10;
        const TF Lmax = 1.e16;
        const TF L_min_stable = zsl/TF(zL_max);
        bfluxbot = bfluxbot >= TF(0.) ? fmax(TF(dsmall), bfluxbot) : fmin(-TF(dsmall), bfluxbot);
        auto f = [&](TF l) { const TF x = du*most_fm<TF>(zsl, z0m, l); return zsl/l + TF(kappa)*zsl*bfluxbot/(x*x*x); };
        while (m <= 1)
        {
            if (m == 1 || L*bfluxbot >= TF(0.))
            {
                nlim = 200;
                L = bfluxbot >= TF(0.) ? -TF(dsmall) : L_min_stable;
            }
            L0 = bfluxbot >= TF(0.) ? -TF(dhuge) : TF(dhuge);
            int n = 0;
            while (fabs((L - L0)/L0) > TF(0.001) && n < nlim && fabs(L) < Lmax)
            {
                L0 = L;
                fx = f(L);
                Lstart = L - TF(0.001)*L;
                Lend = L + TF(0.001)*L;
                fxdif = (f(Lend) - f(Lstart)) / (Lend - Lstart);
                if (fabs(fxdif) < TF(1e-16)) break;
                L = L - fx/fxdif;
                if (L >= TF(0) && L < L_min_stable) L = L_min_stable;
                ++n;
            }
            if (n < nlim && fabs(L) < Lmax) break;
            ++m;
            nlim = 200;
        }
        if (m > 1)
            L = fabs(L) > Lmax ? -copysign(TF(1), bfluxbot)*Lmax : L_min_stable;
        return zsl/fmin(fmax(zsl/L, TF(zL_min)), TF(zL_max));
    }

    template<typename TF>
    __host__ __device__ TF obuk_dirichlet_iterative(TF L, TF du, TF db, TF zsl, TF z0m, TF z0h)
    {
        #pragma clang fp contract(off)
        TF L0, Lstart, Lend, fx, fxdif;
        int m = 0, nlim = 10;
        const TF Lmax = 1.e16;
        const TF L_min_stable = zsl/TF(zL_max);
        const TF Ri = TF(kappa)*db*zsl/(du*du);
        if (Ri > TF(0.13)) return L_min_stable;
        db = db >= TF(0.) ? fmax(TF(dsmall), db) : fmin(-TF(dsmall), db);
        auto f = [&](TF l) {
            const TF x = du*most_fm<TF>(zsl, z0m, l);
            return zsl/l - TF(kappa)*zsl*db*most_fh<TF>(zsl, z0h, l)/(x*x);
        };
        while (m <= 1)
        {
            if (m == 1 || L*db <= TF(0.))
            {
                nlim = 200;
                L = db >= TF(0.) ? L_min_stable : -TF(dsmall);
            }
            L0 = db >= TF(0.) ? TF(dhuge) : -TF(dhuge);
            int n = 0;
            while (fabs((L - L0)/L0) > TF(0.001) && n < nlim && fabs(L) < Lmax)
            {
                L0 = L;
                fx = f(L);
                Lstart = L - TF(0.001)*L;
                Lend = L + TF(0.001)*L;
                fxdif = (f(Lend) - f(Lstart)) / (Lend - Lstart);
                if (fabs(fxdif) < TF(1e-16)) break;
                L = L - fx/fxdif;
                if (L >= TF(0) && L < L_min_stable) L = L_min_stable;
                ++n;
            }
            if (n < nlim && fabs(L) < Lmax) break;
            ++m;
            nlim = 200;
        }
        if (m > 1)
            L = fabs(L) > Lmax ? copysign(TF(1), db)*Lmax : L_min_stable;
        return zsl/fmin(fmax(zsl/L, TF(zL_min)), TF(zL_max));
    }

    constexpr int PT = 256;   // threads per block of the plane kernels
    inline int pblocks(int n) { return (n + PT - 1)/PT; }

    // Periodic images of a plane: every ghost cell takes the interior cell
    // at its wrapped (i, j) (Boundary_cyclic::exec_2d, east-west then
    // north-south, corners included).
    template<typename TF>
    __device__ __forceinline__ void cyclic_2d_g(TF* __restrict__ a, TF* __restrict__ b, Gd g, const Bid& bid_)
    {
        const int ij = bid_.x*PT + threadIdx.x;
        if (ij >= g.ijcells) return;
        const int j = ij / g.icells, i = ij - j*g.icells;
        if (i >= g.istart && i < g.iend && j >= g.jstart && j < g.jend) return;
        const int is = g.istart + ((i - g.istart) % g.itot + g.itot) % g.itot;
        const int js = g.jstart + ((j - g.jstart) % g.jtot + g.jtot) % g.jtot;
        a[ij] = a[is + js*g.icells];
        if (b) b[ij] = b[is + js*g.icells];
    }

    template<typename TF>
    struct cyclic_2d_k
    {
        static constexpr int NT = PT, MINB = 0;
        TF* a; TF* b; Gd g;
        __device__ __forceinline__ void operator()(const Bid& bid_) const
        {
            cyclic_2d_g<TF>(a, b, g, bid_);
        }
    };

    // calc_dutot (include/boundary_surface_kernels.h:134-181), interior columns.
    template<typename TF>
    __device__ __forceinline__ void sfc_dutot_g(TF* __restrict__ dutot, const TF* __restrict__ u,
                                                const TF* __restrict__ v, const TF* __restrict__ ubot,
                                                const TF* __restrict__ vbot, Gd g, const Bid& bid_)
    {
        const int t = bid_.x*PT + threadIdx.x;
        if (t >= g.itot*g.jtot) return;
        const int j = t / g.itot + g.jstart, i = t % g.itot + g.istart;
        const int ii = 1, ii2 = 2, jj = g.icells, jj2 = 2*g.icells;
        const int ij = i + j*jj;
        const size_t ijk = ij + static_cast<size_t>(g.kstart)*g.ijcells;
        const TF h = TF(0.5);
        const TF uf = TF(1./9) *
            ( h*u[ijk-ii-jj] + u[ijk-jj] + u[ijk+ii-jj] + h*u[ijk+ii2-jj]
            + h*u[ijk-ii   ] + u[ijk   ] + u[ijk+ii   ] + h*u[ijk+ii2   ]
            + h*u[ijk-ii+jj] + u[ijk+jj] + u[ijk+ii+jj] + h*u[ijk+ii2+jj] );
        const TF vf = TF(1./9) *
            ( h*v[ijk-ii-jj] + v[ijk-ii] + v[ijk-ii+jj] + h*v[ijk-ii+jj2]
            + h*v[ijk   -jj] + v[ijk   ] + v[ijk   +jj] + h*v[ijk   +jj2]
            + h*v[ijk+ii-jj] + v[ijk+ii] + v[ijk+ii+jj] + h*v[ijk+ii+jj2] );
        const TF du = uf - h*(ubot[ij] + ubot[ij+ii]);
        const TF dv = vf - h*(vbot[ij] + vbot[ij+jj]);
        dutot[ij] = fmax(std::pow(du*du + dv*dv, TF(0.5)), TF(1.e-1));
    }

    template<typename TF>
    struct sfc_dutot_k
    {
        static constexpr int NT = PT, MINB = 0;
        TF* dutot; const TF* u; const TF* v; const TF* ubot; const TF* vbot; Gd g;
        __device__ __forceinline__ void operator()(const Bid& bid_) const
        {
            sfc_dutot_g<TF>(dutot, u, v, ubot, vbot, g, bid_);
        }
    };

    // Surface buoyancy of the dry thermodynamics (src/thermo_dry.cxx:131-160):
    // the buoyancy flux, and b at the first level and at the surface, all
    // columns.  gth, gthh: g/thref[kstart], g/threfh[kstart]; thref_rel,
    // threfh_rel: thref, threfh at kstart minus the storage offset of theta.
    template<typename TF>
    __device__ __forceinline__ void sfc_buoy_g(TF* __restrict__ bflux, TF* __restrict__ b, TF* __restrict__ bbot,
                                               const TF* __restrict__ thflux, const TF* __restrict__ th,
                                               const TF* __restrict__ thbot, TF gth, TF gthh,
                                               TF thref_rel, TF threfh_rel, Gd g, const Bid& bid_)
    {
        const int ij = bid_.x*PT + threadIdx.x;
        if (ij >= g.ijcells) return;
        bflux[ij] = gthh*thflux[ij];
        bbot[ij] = gthh*(thbot[ij] - threfh_rel);
        b[ij] = gth*(th[ij + static_cast<size_t>(g.kstart)*g.ijcells] - thref_rel);
    }

    template<typename TF>
    struct sfc_buoy_k
    {
        static constexpr int NT = PT, MINB = 0;
        TF* bflux; TF* b; TF* bbot; const TF* thflux; const TF* th; const TF* thbot; TF gth; TF gthh;
        TF thref_rel; TF threfh_rel; Gd g;
        __device__ __forceinline__ void operator()(const Bid& bid_) const
        {
            sfc_buoy_g<TF>(bflux, b, bbot, thflux, th, thbot, gth, gthh, thref_rel, threfh_rel, g, bid_);
        }
    };

    // Stability (src/boundary_surface.cxx:54-171): the Obukhov length and u*
    // per column.  MODE 0: fixed u*, flux condition; 1: no slip, flux
    // condition; 2: no slip, value condition; 3: neutral, fixed u*
    // (interior columns); 4: neutral, no slip.
    template<typename TF, int MODE, bool LUT>
    __device__ __forceinline__ void sfc_stability_g(TF* __restrict__ ustar, TF* __restrict__ obuk,
                                                    int* __restrict__ nobuk, const TF* __restrict__ bflux,
                                                    const TF* __restrict__ b, const TF* __restrict__ bbot,
                                                    const TF* __restrict__ dutot, const TF* __restrict__ z0m,
                                                    const TF* __restrict__ z0h, const float* __restrict__ zl,
                                                    const float* __restrict__ fl, int nzl, TF zsl, TF db_ref, Gd g, const Bid& bid_)
    {
        #pragma clang fp contract(off)
        const int ij = bid_.x*PT + threadIdx.x;
        if (ij >= g.ijcells) return;
        if (MODE == 0)
        {
            const TF us = ustar[ij];
            obuk[ij] = -(us*us*us) / (TF(kappa)*bflux[ij]);
        }
        else if (MODE == 1 || MODE == 2)
        {
            const TF du = dutot[ij];
            TF L;
            if (LUT)
            {
                int n = nobuk[ij];
                float Ri;
                if (MODE == 1) Ri = static_cast<float>(-TF(kappa) * bflux[ij] * zsl / (du*du*du));
                else           Ri = static_cast<float>(TF(kappa) * (b[ij] - bbot[ij] + db_ref) * zsl / (du*du));
                L = zsl/static_cast<TF>(find_zL(zl, fl, n, nzl, Ri));
                nobuk[ij] = n;
            }
            else if (MODE == 1)
                L = obuk_flux_iterative<TF>(obuk[ij], du, bflux[ij], zsl, z0m[ij]);
            else
                L = obuk_dirichlet_iterative<TF>(obuk[ij], du, b[ij] - bbot[ij] + db_ref, zsl, z0m[ij], z0h[ij]);
            obuk[ij] = L;
            ustar[ij] = du * most_fm<TF>(zsl, z0m[ij], L);
        }
        else if (MODE == 3)
        {
            const int j = ij / g.icells, i = ij - j*g.icells;
            if (i >= g.istart && i < g.iend && j >= g.jstart && j < g.jend) obuk[ij] = -TF(dbig);
        }
        else
        {
            obuk[ij] = -TF(dbig);
            ustar[ij] = dutot[ij] * most_fm<TF>(zsl, z0m[ij], -TF(dbig));
        }
    }

    template<typename TF, int MODE, bool LUT>
    struct sfc_stability_k
    {
        static constexpr int NT = PT, MINB = 0;
        TF* ustar; TF* obuk; int* nobuk; const TF* bflux; const TF* b; const TF* bbot; const TF* dutot;
        const TF* z0m; const TF* z0h; const float* zl; const float* fl; int nzl; TF zsl; TF db_ref; Gd g;
        __device__ __forceinline__ void operator()(const Bid& bid_) const
        {
            sfc_stability_g<TF, MODE, LUT>(ustar, obuk, nobuk, bflux, b, bbot, dutot, z0m, z0h, zl, fl, nzl,
                zsl, db_ref, g, bid_);
        }
    };

    // surfm (src/boundary_surface.cxx:173-286): momentum fluxes in the
    // interior (BC: MHH_BC_DIRICHLET or MHH_BC_USTAR), gradients everywhere.
    template<typename TF, int BC>
    __device__ __forceinline__ void sfc_surfm_g(TF* __restrict__ ufb, TF* __restrict__ vfb,
                                                TF* __restrict__ ugb, TF* __restrict__ vgb,
                                                const TF* __restrict__ ustar, const TF* __restrict__ obuk,
                                                const TF* __restrict__ u, const TF* __restrict__ ubot,
                                                const TF* __restrict__ v, const TF* __restrict__ vbot,
                                                const TF* __restrict__ z0m, TF zsl, Gd g, const Bid& bid_)
    {
        const int ij = bid_.x*PT + threadIdx.x;
        if (ij >= g.ijcells) return;
        const int j = ij / g.icells, i = ij - j*g.icells;
        const int ii = 1, jj = g.icells;
        const size_t ijk = ij + static_cast<size_t>(g.kstart)*g.ijcells;
        if (i >= g.istart && i < g.iend && j >= g.jstart && j < g.jend)
        {
            if (BC == MHH_BC_DIRICHLET)
            {
                const TF fc = ustar[ij]*most_fm<TF>(zsl, z0m[ij], obuk[ij]);
                ufb[ij] = -(u[ijk]-ubot[ij])*TF(0.5)*(ustar[ij-ii]*most_fm<TF>(zsl, z0m[ij-ii], obuk[ij-ii]) + fc);
                vfb[ij] = -(v[ijk]-vbot[ij])*TF(0.5)*(ustar[ij-jj]*most_fm<TF>(zsl, z0m[ij-jj], obuk[ij-jj]) + fc);
            }
            else
            {
                const TF minval = 1.e-2;
                auto sq = [](TF x) { return x*x; };
                const TF vonu2 = fmax(minval, TF(0.25)*(
                            sq(v[ijk-ii]-vbot[ij-ii]) + sq(v[ijk-ii+jj]-vbot[ij-ii+jj])
                          + sq(v[ijk   ]-vbot[ij   ]) + sq(v[ijk   +jj]-vbot[ij   +jj])) );
                const TF uonv2 = fmax(minval, TF(0.25)*(
                            sq(u[ijk-jj]-ubot[ij-jj]) + sq(u[ijk+ii-jj]-ubot[ij+ii-jj])
                          + sq(u[ijk   ]-ubot[ij   ]) + sq(u[ijk+ii   ]-ubot[ij+ii   ])) );
                const TF u2 = fmax(minval, sq(u[ijk]-ubot[ij]));
                const TF v2 = fmax(minval, sq(v[ijk]-vbot[ij]));
                const TF usu4 = TF(0.5)*(sq(sq(ustar[ij-ii])) + sq(sq(ustar[ij])));
                const TF usv4 = TF(0.5)*(sq(sq(ustar[ij-jj])) + sq(sq(ustar[ij])));
                ufb[ij] = -copysign(TF(1), u[ijk]-ubot[ij]) * std::pow(usu4 / (TF(1) + vonu2 / u2), TF(0.5));
                vfb[ij] = -copysign(TF(1), v[ijk]-vbot[ij]) * std::pow(usv4 / (TF(1) + uonv2 / v2), TF(0.5));
            }
        }
        ugb[ij] = (u[ijk]-ubot[ij])/zsl;
        vgb[ij] = (v[ijk]-vbot[ij])/zsl;
    }

    template<typename TF, int BC>
    struct sfc_surfm_k
    {
        static constexpr int NT = PT, MINB = 0;
        TF* ufb; TF* vfb; TF* ugb; TF* vgb; const TF* ustar; const TF* obuk; const TF* u; const TF* ubot;
        const TF* v; const TF* vbot; const TF* z0m; TF zsl; Gd g;
        __device__ __forceinline__ void operator()(const Bid& bid_) const
        {
            sfc_surfm_g<TF, BC>(ufb, vfb, ugb, vgb, ustar, obuk, u, ubot, v, vbot, z0m, zsl, g, bid_);
        }
    };

    // surfs (src/boundary_surface.cxx:288-339), all columns of one scalar.
    template<typename TF, int BC>
    __device__ __forceinline__ void sfc_surfs_g(TF* __restrict__ sbot, TF* __restrict__ sgrad,
                                                TF* __restrict__ sflux, const TF* __restrict__ ustar,
                                                const TF* __restrict__ obuk, const TF* __restrict__ s,
                                                const TF* __restrict__ z0h, TF zsl, Gd g, const Bid& bid_)
    {
        const int ij = bid_.x*PT + threadIdx.x;
        if (ij >= g.ijcells) return;
        const TF sk = s[ij + static_cast<size_t>(g.kstart)*g.ijcells];
        if (BC == MHH_BC_DIRICHLET)
            sflux[ij] = -(sk-sbot[ij])*ustar[ij]*most_fh<TF>(zsl, z0h[ij], obuk[ij]);
        else
            sbot[ij] = sflux[ij] / (ustar[ij]*most_fh<TF>(zsl, z0h[ij], obuk[ij])) + sk;
        sgrad[ij] = (sk-sbot[ij])/zsl;
    }

    template<typename TF, int BC>
    struct sfc_surfs_k
    {
        static constexpr int NT = PT, MINB = 0;
        TF* sbot; TF* sgrad; TF* sflux; const TF* ustar; const TF* obuk; const TF* s; const TF* z0h; TF zsl;
        Gd g;
        __device__ __forceinline__ void operator()(const Bid& bid_) const
        {
            sfc_surfs_g<TF, BC>(sbot, sgrad, sflux, ustar, obuk, s, z0h, zsl, g, bid_);
        }
    };

    // calc_duvdz_mo and calc_dbdz_mo (include/boundary_surface_kernels.h:183-241)
    // in the interior; the buoyancy flux from the scalar flux after surfs.
    template<typename TF, bool TH>
    __device__ __forceinline__ void sfc_gradients_g(TF* __restrict__ dudz, TF* __restrict__ dvdz,
                                                    TF* __restrict__ dbdz, const TF* __restrict__ u,
                                                    const TF* __restrict__ v, const TF* __restrict__ ubot,
                                                    const TF* __restrict__ vbot, const TF* __restrict__ ustar,
                                                    const TF* __restrict__ obuk, const TF* __restrict__ z0m,
                                                    const TF* __restrict__ thflux, TF gthh, TF zsl, Gd g, const Bid& bid_)
    {
        const int t = bid_.x*PT + threadIdx.x;
        if (t >= g.itot*g.jtot) return;
        const int j = t / g.itot + g.jstart, i = t % g.itot + g.istart;
        const int ii = 1, jj = g.icells;
        const int ij = i + j*jj;
        const size_t ijk = ij + static_cast<size_t>(g.kstart)*g.ijcells;
        const TF du_c = TF(0.5)*((u[ijk] - ubot[ij]) + (u[ijk+ii] - ubot[ij+ii]));
        const TF dv_c = TF(0.5)*((v[ijk] - vbot[ij]) + (v[ijk+jj] - vbot[ij+jj]));
        const TF us = ustar[ij], L = obuk[ij];
        const TF fm = most_fm<TF>(zsl, z0m[ij], L);
        const TF uf = -du_c * us * fm;
        const TF vf = -dv_c * us * fm;
        const TF pm = phim<TF>(zsl/L);
        dudz[ij] = -uf / (TF(kappa) * zsl * us) * pm;
        dvdz[ij] = -vf / (TF(kappa) * zsl * us) * pm;
        if (TH)
        {
            const TF bf = gthh*thflux[ij];
            dbdz[ij] = -bf / (TF(kappa) * zsl * us) * phih<TF>(zsl/L);
        }
    }

    template<typename TF, bool TH>
    struct sfc_gradients_k
    {
        static constexpr int NT = PT, MINB = 0;
        TF* dudz; TF* dvdz; TF* dbdz; const TF* u; const TF* v; const TF* ubot; const TF* vbot;
        const TF* ustar; const TF* obuk; const TF* z0m; const TF* thflux; TF gthh; TF zsl; Gd g;
        __device__ __forceinline__ void operator()(const Bid& bid_) const
        {
            sfc_gradients_g<TF, TH>(dudz, dvdz, dbdz, u, v, ubot, vbot, ustar, obuk, z0m, thflux, gthh, zsl,
                g, bid_);
        }
    };

    template<typename TF>
    int alloc_plane(mhh_ctx* c, void** p, TF fill)
    {
        const size_t n = static_cast<size_t>(c->gd.ijcells);
        MHH_CHECK(check_hip(hipMalloc(p, sizeof(TF)*n), "hipMalloc(surface plane)"));
        std::vector<TF> h(n, fill);
        return check_hip(hipMemcpy(*p, h.data(), sizeof(TF)*n, hipMemcpyHostToDevice), "hipMemcpy(surface plane)");
    }

    template<typename TF>
    int surface_init(mhh_ctx* c, const mhh_surface_desc& d)
    {
        const Gd& g = c->gd;
        auto* s = new mhh_surface_state();
        c->sfc = s;
        s->desc = d;
        MHH_CHECK(alloc_plane<TF>(c, &s->ustar, TF(d.mbcbot == MHH_BC_USTAR ? std::max(1e-4, d.ustar) : 1e-2)));
        MHH_CHECK(alloc_plane<TF>(c, &s->obuk, TF(dsmall)));
        MHH_CHECK(alloc_plane<TF>(c, &s->z0h, TF(d.z0h)));
        MHH_CHECK(alloc_plane<TF>(c, &s->dutot, TF(0)));
        MHH_CHECK(alloc_plane<TF>(c, &s->bflux, TF(0)));
        MHH_CHECK(alloc_plane<TF>(c, &s->b, TF(0)));
        MHH_CHECK(alloc_plane<TF>(c, &s->bbot, TF(0)));
        MHH_CHECK(check_hip(hipMalloc(&s->nobuk, sizeof(int)*g.ijcells), "hipMalloc(nobuk)"));
        MHH_CHECK(check_hip(hipMemset(s->nobuk, 0, sizeof(int)*g.ijcells), "hipMemset(nobuk)"));
        // z0m is the bound plane the viscosity's Mason length reads
        {
            std::vector<TF> h(g.ijcells, TF(d.z0m));
            MHH_CHECK(check_hip(hipMemcpy(c->f.z0m, h.data(), sizeof(TF)*g.ijcells, hipMemcpyHostToDevice),
                                "hipMemcpy(z0m)"));
        }
        if (d.thermo)
        {
            const int ks = g.kstart;
            s->db_ref = grav/c->h_thref[ks]*(c->h_thref[ks] - c->h_threfh[ks]);
        }
        if (d.constant_z0)
        {
            const int thermobc = d.thermo ? d.sbcbot[0] : MHH_BC_FLUX;
            std::vector<float> zl, fl;
            prepare_lut<TF>(zl, fl, TF(d.z0m), TF(d.z0h), TF(c->h_z[g.kstart]), s->nzl, d.mbcbot, thermobc);
            MHH_CHECK(check_hip(hipMalloc(&s->zl, sizeof(float)*s->nzl), "hipMalloc(lut)"));
            MHH_CHECK(check_hip(hipMalloc(&s->fl, sizeof(float)*s->nzl), "hipMalloc(lut)"));
            MHH_CHECK(check_hip(hipMemcpy(s->zl, zl.data(), sizeof(float)*s->nzl, hipMemcpyHostToDevice), "hipMemcpy(lut)"));
            MHH_CHECK(check_hip(hipMemcpy(s->fl, fl.data(), sizeof(float)*s->nzl, hipMemcpyHostToDevice), "hipMemcpy(lut)"));
        }
        return 0;
    }

    template<typename TF>
    int surface_exec(mhh_ctx* c)
    {
        mhh_surface_state& s = *c->sfc;
        const mhh_surface_desc& d = s.desc;
        const Gd& g = c->gd;
        const TF zsl = TF(c->h_z[g.kstart]);
        auto P = [](void* p) { return static_cast<TF*>(p); };
        const mhh_field_set& f = c->f;
        const int nb = pblocks(g.ijcells), nbi = pblocks(g.itot*g.jtot);
        mhh::Timer _t(c, "surface");

        launch(c, sfc_dutot_k<TF>{P(s.dutot), P(f.u), P(f.v), P(f.u_bot), P(f.v_bot), g}, nbi, PT);
        launch(c, cyclic_2d_k<TF>{P(s.dutot), nullptr, g}, nb, PT);

        const int ks = g.kstart;
        const TF gth = d.thermo ? TF(grav/c->h_thref[ks]) : TF(0);
        const TF gthh = d.thermo ? TF(grav/c->h_threfh[ks]) : TF(0);
        const float* zl = s.zl; const float* fl = s.fl;
        const bool lut = d.constant_z0 != 0;
        if (d.thermo)
        {
            launch(c, sfc_buoy_k<TF>{P(s.bflux), P(s.b), P(s.bbot), P(f.s_fluxbot[0]), P(f.s[0]),
                                                     P(f.s_bot[0]), gth, gthh, TF(c->h_thref[ks] - c->s_offset[0]),
                                                     TF(c->h_threfh[ks] - c->s_offset[0]), g}, nb, PT);
            const int bc = d.sbcbot[0];
#define MHH_STAB(M, L) launch(c, sfc_stability_k<TF, M, L>{P(s.ustar), P(s.obuk), s.nobuk, \
                P(s.bflux), P(s.b), P(s.bbot), P(s.dutot), P(f.z0m), P(s.z0h), zl, fl, s.nzl, zsl, TF(s.db_ref), g}, nb, PT)
            if (d.mbcbot == MHH_BC_USTAR) MHH_STAB(0, false);
            else if (bc == MHH_BC_FLUX) { if (lut) MHH_STAB(1, true); else MHH_STAB(1, false); }
            else { if (lut) MHH_STAB(2, true); else MHH_STAB(2, false); }
        }
        else
        {
            if (d.mbcbot == MHH_BC_USTAR) MHH_STAB(3, false);
            else MHH_STAB(4, false);
#undef MHH_STAB
        }

        if (d.mbcbot == MHH_BC_DIRICHLET)
            launch(c, sfc_surfm_k<TF, MHH_BC_DIRICHLET>{P(f.u_fluxbot), P(f.v_fluxbot),
                P(f.u_gradbot), P(f.v_gradbot), P(s.ustar), P(s.obuk), P(f.u), P(f.u_bot), P(f.v), P(f.v_bot),
                P(f.z0m), zsl, g}, nb, PT);
        else
            launch(c, sfc_surfm_k<TF, MHH_BC_USTAR>{P(f.u_fluxbot), P(f.v_fluxbot),
                P(f.u_gradbot), P(f.v_gradbot), P(s.ustar), P(s.obuk), P(f.u), P(f.u_bot), P(f.v), P(f.v_bot),
                P(f.z0m), zsl, g}, nb, PT);
        launch(c, cyclic_2d_k<TF>{P(f.u_fluxbot), P(f.v_fluxbot), g}, nb, PT);

        for (int n = 0; n < f.nscalars; ++n)
        {
            if (d.sbcbot[n] == MHH_BC_DIRICHLET)
                launch(c, sfc_surfs_k<TF, MHH_BC_DIRICHLET>{P(f.s_bot[n]), P(f.s_gradbot[n]),
                    P(f.s_fluxbot[n]), P(s.ustar), P(s.obuk), P(f.s[n]), P(s.z0h), zsl, g}, nb, PT);
            else
                launch(c, sfc_surfs_k<TF, MHH_BC_FLUX>{P(f.s_bot[n]), P(f.s_gradbot[n]),
                    P(f.s_fluxbot[n]), P(s.ustar), P(s.obuk), P(f.s[n]), P(s.z0h), zsl, g}, nb, PT);
        }

        if (d.thermo)
            launch(c, sfc_gradients_k<TF, true>{P(f.dudz), P(f.dvdz), P(f.dbdz), P(f.u), P(f.v),
                P(f.u_bot), P(f.v_bot), P(s.ustar), P(s.obuk), P(f.z0m), P(f.s_fluxbot[0]), gthh, zsl, g}, nbi, PT);
        else
            launch(c, sfc_gradients_k<TF, false>{P(f.dudz), P(f.dvdz), nullptr, P(f.u), P(f.v),
                P(f.u_bot), P(f.v_bot), P(s.ustar), P(s.obuk), P(f.z0m), nullptr, gthh, zsl, g}, nbi, PT);
        return check_launch("surface");
    }

    // ---------------------------------------------------------------- buffer
    template<typename TF>
    struct Buf_list
    {
        TF* at[3 + MHH_MAX_SCALARS];
        const TF* a[3 + MHH_MAX_SCALARS];
    };

    // calc_buffer (src/buffer.cxx:38-58) for u, v, w and the damped scalars:
    // blockIdx.z is the field (2: w, at the half levels), blockIdx.y the
    // level above the lowest buffer level.
    template<typename TF>
    __global__ void __launch_bounds__(BX*BY) buffer_g(Buf_list<TF> fl, const double* __restrict__ prof,
                                                      const TF* __restrict__ sig_c, const TF* __restrict__ sig_h,
                                                      int kfirst, int ntx, Gd g)
    {
        const int fi = blockIdx.z;
        const int k = kfirst + blockIdx.y;
        const int tx = blockIdx.x % ntx, ty = blockIdx.x / ntx;
        const int i = g.istart + tx*BX + threadIdx.x, j = g.jstart + ty*BY + threadIdx.y;
        if (i >= g.iend || j >= g.jend) return;
        const TF sig = (fi == 2 ? sig_h : sig_c)[k];
        if (sig == TF(0)) return;
        const size_t ijk = i + j*g.icells + static_cast<size_t>(k)*g.ijcells;
        fl.at[fi][ijk] -= sig*(fl.a[fi][ijk] - TF(prof[static_cast<size_t>(fi)*g.kcells + k]));
    }

    template<typename TF>
    int buffer_init(mhh_ctx* c, const mhh_buffer_desc& d, const double* up, const double* vp,
                    const double* const* sp, int ns)
    {
        const Gd& g = c->gd;
        auto* b = new mhh_buffer_state();
        c->buf = b;
        b->desc = d;
        b->ndamped = 3 + ns;
        // src/buffer.cxx:101-125
        b->kb = g.kstart; b->kbh = g.kstart;
        for (int k = g.kstart; k < g.kend; ++k)
        {
            if (c->h_z[k] < d.zstart) ++b->kb;
            if (c->h_zh[k] < d.zstart) ++b->kbh;
        }
        if (b->kbh == g.kend)
            return fail(MHH_EINVAL, "mhh_buffer_init: buffer is too close to the model top");
        const double zsize = c->h_zh[g.kend];
        std::vector<TF> sc(g.kcells, TF(0)), sh(g.kcells, TF(0));
        for (int k = b->kb; k < g.kend; ++k)
            sc[k] = TF(d.sigma*std::pow((c->h_z[k] - d.zstart)/(zsize - d.zstart), d.beta));
        for (int k = b->kbh; k < g.kend; ++k)
            sh[k] = TF(d.sigma*std::pow((c->h_zh[k] - d.zstart)/(zsize - d.zstart), d.beta));
        MHH_CHECK(check_hip(hipMalloc(&b->sig_c, sizeof(TF)*g.kcells), "hipMalloc(buffer)"));
        MHH_CHECK(check_hip(hipMalloc(&b->sig_h, sizeof(TF)*g.kcells), "hipMalloc(buffer)"));
        MHH_CHECK(check_hip(hipMemcpy(b->sig_c, sc.data(), sizeof(TF)*g.kcells, hipMemcpyHostToDevice), "hipMemcpy"));
        MHH_CHECK(check_hip(hipMemcpy(b->sig_h, sh.data(), sizeof(TF)*g.kcells, hipMemcpyHostToDevice), "hipMemcpy"));
        const size_t np = static_cast<size_t>(3 + MHH_MAX_SCALARS)*g.kcells;
        std::vector<double> prof(np, 0.);
        if (!d.swupdate)
        {
            // the initial profiles (w: zero), relative to the storage offsets
            for (int k = 0; k < g.kcells; ++k)
            {
                prof[0*g.kcells + k] = up[k];
                prof[1*g.kcells + k] = vp[k];
                for (int n = 0; n < ns; ++n)
                    prof[(3 + n)*g.kcells + k] = sp[n][k] - c->s_offset[n];
            }
        }
        MHH_CHECK(check_hip(hipMalloc(&b->prof, sizeof(double)*np), "hipMalloc(buffer)"));
        if (d.swupdate)
            MHH_CHECK(check_hip(hipMalloc(&b->part, sizeof(double)*np*plane_chunks(g)), "hipMalloc(buffer)"));
        return check_hip(hipMemcpy(b->prof, prof.data(), sizeof(double)*np, hipMemcpyHostToDevice), "hipMemcpy");
    }

    template<typename TF>
    int buffer_exec(mhh_ctx* c)
    {
        mhh_buffer_state& b = *c->buf;
        const Gd& g = c->gd;
        Buf_list<TF> fl{};
        const mhh_field_set& f = c->f;
        fl.at[0] = static_cast<TF*>(f.ut); fl.a[0] = static_cast<const TF*>(f.u);
        fl.at[1] = static_cast<TF*>(f.vt); fl.a[1] = static_cast<const TF*>(f.v);
        fl.at[2] = static_cast<TF*>(f.wt); fl.a[2] = static_cast<const TF*>(f.w);
        for (int n = 0; n < b.ndamped - 3; ++n)
        {
            fl.at[3 + n] = static_cast<TF*>(f.st[n]);
            fl.a[3 + n] = static_cast<const TF*>(f.s[n]);
        }
        if (b.desc.swupdate)
        {
            // all fields in one pass and one fold: with a pass per field a small
            // grid waits for launches (32^3 FP64, four fields: 32 us, now 12)
            Plane_fields<TF> pf{};
            std::copy(fl.a, fl.a + b.ndamped, pf.a);
            MHH_CHECK(mean_profiles<TF>(c, pf, b.ndamped, b.part, b.prof));
        }
        const int kfirst = std::min(b.kb, b.kbh);
        const int ntx = (g.itot + BX - 1)/BX, nty = (g.jtot + BY - 1)/BY;
        mhh::Timer _t(c, "buffer");
        buffer_g<TF><<<dim3(ntx*nty, g.kend - kfirst, b.ndamped), dim3(BX, BY), 0, c->stream>>>(
                fl, b.prof, static_cast<const TF*>(b.sig_c), static_cast<const TF*>(b.sig_h), kfirst, ntx, g);
        return check_launch("buffer");
    }
}

namespace mhh
{
    void surface_free(mhh_ctx* c)
    {
        if (c->sfc)
        {
            mhh_surface_state* s = c->sfc;
            for (void* p : {s->ustar, s->obuk, s->z0h, s->dutot, s->bflux, s->b, s->bbot})
                if (p) (void)hipFree(p);
            if (s->nobuk) (void)hipFree(s->nobuk);
            if (s->zl) (void)hipFree(s->zl);
            if (s->fl) (void)hipFree(s->fl);
            delete s;
            c->sfc = nullptr;
        }
        if (c->buf)
        {
            mhh_buffer_state* b = c->buf;
            if (b->prof) (void)hipFree(b->prof);
            if (b->part) (void)hipFree(b->part);
            if (b->sig_c) (void)hipFree(b->sig_c);
            if (b->sig_h) (void)hipFree(b->sig_h);
            delete b;
            c->buf = nullptr;
        }
    }
}

extern "C" {

int mhh_boundary_surface_init(mhh_ctx* c, const mhh_surface_desc* d)
{
    MHH_REQUIRE_BOUND(c);
    MHH_NOT_IN_BATCH(c, "mhh_boundary_surface_init");
    if (!d) return mhh::fail(MHH_EINVAL, "mhh_boundary_surface_init: null descriptor");
    if (d->mbcbot != MHH_BC_DIRICHLET && d->mbcbot != MHH_BC_USTAR)
        return mhh::fail(MHH_EINVAL, "the surface model takes a no-slip (Dirichlet) or fixed-u* momentum condition");
    for (int n = 0; n < c->f.nscalars; ++n)
    {
        if (d->sbcbot[n] != MHH_BC_FLUX && d->sbcbot[n] != MHH_BC_DIRICHLET)
            return mhh::fail(MHH_EINVAL, "the surface model takes flux or value conditions for the scalars");
        if (d->sbcbot[n] == MHH_BC_DIRICHLET && d->mbcbot == MHH_BC_USTAR)
            return mhh::fail(MHH_EINVAL, "a fixed u* with a value condition for a scalar is not supported");
    }
    if (d->thermo && c->f.nscalars < 1) return mhh::fail(MHH_ESTATE, "thermo needs scalar 0");
    if (d->thermo && !c->have_base_state) return mhh::fail(MHH_ESTATE, "thermo needs mhh_set_base_state()");
    if (!(d->z0m > 0.) || !(d->z0h > 0.)) return mhh::fail(MHH_EINVAL, "roughness lengths must be positive");
    if (d->z0m >= c->h_z[c->gd.kstart] || d->z0h >= c->h_z[c->gd.kstart])
        return mhh::fail(MHH_EINVAL, "roughness lengths must lie below the first level");
    const mhh_field_set& f = c->f;
    for (const void* p : {f.u_bot, f.v_bot, f.u_fluxbot, f.v_fluxbot, f.u_gradbot, f.v_gradbot, f.dudz, f.dvdz, f.z0m})
        if (!p) return mhh::fail(MHH_ESTATE, "the surface model needs the u, v bottom planes, dudz, dvdz and z0m bound");
    if (d->thermo && !f.dbdz) return mhh::fail(MHH_ESTATE, "the surface model with thermo needs dbdz bound");
    for (int n = 0; n < f.nscalars; ++n)
        if (!f.s_bot[n] || !f.s_gradbot[n] || !f.s_fluxbot[n])
            return mhh::fail(MHH_ESTATE, "the surface model needs every scalar's bottom planes bound");
    if (c->sfc)
    {
        // a second init replaces the state (the buffer is kept)
        mhh_buffer_state* keep = c->buf;
        c->buf = nullptr;
        mhh::surface_free(c);
        c->buf = keep;
    }
    const int rc = c->precision == MHH_FP64 ? surface_init<double>(c, *d) : surface_init<float>(c, *d);
    if (rc)
    {
        mhh_buffer_state* keep = c->buf;
        c->buf = nullptr;
        mhh::surface_free(c);
        c->buf = keep;
    }
    return rc;
}

int mhh_boundary_surface_exec(mhh_ctx* c)
{
    MHH_REQUIRE_BOUND(c);
    if (!c->sfc) return mhh::fail(MHH_ESTATE, "mhh_boundary_surface_exec: call mhh_boundary_surface_init first");
    return c->precision == MHH_FP64 ? surface_exec<double>(c) : surface_exec<float>(c);
}

int mhh_boundary_surface_set_roughness(mhh_ctx* c, const double* z0m, const double* z0h)
{
    MHH_REQUIRE_BOUND(c);
    MHH_NOT_IN_BATCH(c, "mhh_boundary_surface_set_roughness");
    if (!c->sfc) return mhh::fail(MHH_ESTATE, "call mhh_boundary_surface_init first");
    if (c->sfc->desc.constant_z0) return mhh::fail(MHH_ESTATE, "heterogeneous roughness needs the iterative solver (constant_z0 = 0)");
    if (!z0m || !z0h) return mhh::fail(MHH_EINVAL, "null argument");
    const int n = c->gd.ijcells;
    MHH_CHECK(mhh::check_hip(hipStreamSynchronize(c->stream), "hipStreamSynchronize"));
    auto put = [&](void* dst, const double* src) {
        if (c->precision == MHH_FP64)
            return mhh::check_hip(hipMemcpy(dst, src, sizeof(double)*n, hipMemcpyHostToDevice), "hipMemcpy");
        std::vector<float> h(src, src + n);
        return mhh::check_hip(hipMemcpy(dst, h.data(), sizeof(float)*n, hipMemcpyHostToDevice), "hipMemcpy");
    };
    MHH_CHECK(put(c->f.z0m, z0m));
    return put(c->sfc->z0h, z0h);
}

int mhh_boundary_surface_get(mhh_ctx* c, double* ustar, double* obuk)
{
    MHH_REQUIRE_BOUND(c);
    MHH_NOT_IN_BATCH(c, "mhh_boundary_surface_get");
    if (!c->sfc) return mhh::fail(MHH_ESTATE, "call mhh_boundary_surface_init first");
    const int n = c->gd.ijcells;
    MHH_CHECK(mhh::check_hip(hipStreamSynchronize(c->stream), "hipStreamSynchronize"));
    auto get = [&](double* dst, const void* src) {
        if (!dst) return 0;
        if (c->precision == MHH_FP64)
            return mhh::check_hip(hipMemcpy(dst, src, sizeof(double)*n, hipMemcpyDeviceToHost), "hipMemcpy");
        std::vector<float> h(n);
        MHH_CHECK(mhh::check_hip(hipMemcpy(h.data(), src, sizeof(float)*n, hipMemcpyDeviceToHost), "hipMemcpy"));
        std::copy(h.begin(), h.end(), dst);
        return 0;
    };
    MHH_CHECK(get(ustar, c->sfc->ustar));
    return get(obuk, c->sfc->obuk);
}

int mhh_boundary_surface_set(mhh_ctx* c, const double* ustar, const double* obuk)
{
    MHH_REQUIRE_BOUND(c);
    MHH_NOT_IN_BATCH(c, "mhh_boundary_surface_set");
    if (!c->sfc) return mhh::fail(MHH_ESTATE, "call mhh_boundary_surface_init first");
    const int n = c->gd.ijcells;
    MHH_CHECK(mhh::check_hip(hipStreamSynchronize(c->stream), "hipStreamSynchronize"));
    auto put = [&](void* dst, const double* src) {
        if (!src) return 0;
        if (c->precision == MHH_FP64)
            return mhh::check_hip(hipMemcpy(dst, src, sizeof(double)*n, hipMemcpyHostToDevice), "hipMemcpy");
        std::vector<float> h(src, src + n);
        return mhh::check_hip(hipMemcpy(dst, h.data(), sizeof(float)*n, hipMemcpyHostToDevice), "hipMemcpy");
    };
    MHH_CHECK(put(c->sfc->ustar, ustar));
    return put(c->sfc->obuk, obuk);
}

int mhh_buffer_init(mhh_ctx* c, const mhh_buffer_desc* d, const double* up, const double* vp,
                    const double* const* sp, int ns)
{
    MHH_REQUIRE_BOUND(c);
    MHH_NOT_IN_BATCH(c, "mhh_buffer_init");
    if (!d) return mhh::fail(MHH_EINVAL, "mhh_buffer_init: null descriptor");
    if (ns < 0 || ns > c->f.nscalars) return mhh::fail(MHH_EINVAL, "mhh_buffer_init: more scalars than bound");
    if (!d->swupdate && (!up || !vp || (ns > 0 && !sp)))
        return mhh::fail(MHH_EINVAL, "mhh_buffer_init: the reference profiles are required without swupdate");
    if (!d->swupdate)
        for (int n = 0; n < ns; ++n)
            if (!sp[n]) return mhh::fail(MHH_EINVAL, "mhh_buffer_init: a scalar profile is missing");
    const double zsize = c->h_zh[c->gd.kend];
    if (!(d->zstart < zsize)) return mhh::fail(MHH_EINVAL, "mhh_buffer_init: zstart must lie below the domain top");
    if (c->buf)
    {
        mhh_surface_state* keep = c->sfc;
        c->sfc = nullptr;
        mhh::surface_free(c);
        c->sfc = keep;
    }
    const int rc = c->precision == MHH_FP64 ? buffer_init<double>(c, *d, up, vp, sp, ns)
                                            : buffer_init<float>(c, *d, up, vp, sp, ns);
    if (rc)
    {
        mhh_surface_state* keep = c->sfc;
        c->sfc = nullptr;
        mhh::surface_free(c);
        c->sfc = keep;
    }
    return rc;
}

int mhh_buffer_exec(mhh_ctx* c)
{
    MHH_REQUIRE_BOUND(c);
    MHH_NOT_IN_BATCH(c, "mhh_buffer_exec");
    if (!c->buf) return mhh::fail(MHH_ESTATE, "mhh_buffer_exec: call mhh_buffer_init first");
    MHH_CHECK(mhh::settle_tendencies(c));
    return c->precision == MHH_FP64 ? buffer_exec<double>(c) : buffer_exec<float>(c);
}

} // extern "C"
