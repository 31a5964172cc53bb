// mhh_force.hip -- the large-scale pressure force of [force] swlspres = uflux
// (Force::exec with enforce_fixed_flux, src/force.cxx:65-75, 610-625): a
// uniform body force on ut that keeps the volume mean of u at uflux.
#include <vector>

#include "mhh_batch.h"

namespace
{
    using namespace mhh;

    // The dz-weighted volume means of u and ut (Field3d_operators::calc_mean,
    // src/field3d_operators.cxx:134-155) from their partial plane sums, and the
    // body force (uflux - u_mean - utrans)/dt - ut_mean, in FP64 by one block:
    // a thread takes every FT-th level, the block folds the shares.
    constexpr int FT = 256;

    __global__ void __launch_bounds__(FT) fixed_flux_force_g(const double* __restrict__ part, double* __restrict__ fbody,
                                                             const double* __restrict__ dz, int nchunk, int nk,
                                                             double npoints, double uflux, double utrans, double dti,
                                                             double zsize)
    {
        __shared__ double su[FT], st[FT];
        const int tid = threadIdx.x;
        double au = 0., at = 0.;
        for (int k = tid; k < nk; k += FT)
        {
            double pu = 0., pt = 0.;
            for (int q = 0; q < nchunk; ++q)
            {
                pu += part[static_cast<size_t>(k)*nchunk + q];
                pt += part[static_cast<size_t>(nk + k)*nchunk + q];
            }
            au += (pu/npoints)*dz[k];
            at += (pt/npoints)*dz[k];
        }
        su[tid] = au; st[tid] = at;
        __syncthreads();
        for (int w = FT/2; w > 0; w >>= 1)
        {
            if (tid < w) { su[tid] += su[tid + w]; st[tid] += st[tid + w]; }
            __syncthreads();
        }
        if (tid == 0)
            *fbody = (uflux - su[0]/zsize - utrans)*dti - st[0]/zsize;
    }

    template<typename TF>
    __global__ void __launch_bounds__(BX*BY) add_force_g(TF* __restrict__ ut, const double* __restrict__ fbody, Gd g)
    {
        const int i = blockIdx.x*BX + threadIdx.x + g.istart;
        const int j = blockIdx.y*BY + threadIdx.y + g.jstart;
        const int k = blockIdx.z + g.kstart;
        if (i >= g.iend || j >= g.jend) return;
        ut[i + j*g.icells + static_cast<size_t>(k)*g.ijcells] += TF(*fbody);
    }

    template<typename TF>
    int fixed_flux(mhh_ctx* c, double uflux, double utrans, double dt)
    {
        const Gd& g = c->gd;
        const int nchunk = plane_chunks(g);
        if (!c->force_buf)
        {
            MHH_CHECK(check_hip(hipMalloc(&c->force_buf, sizeof(double)*(1 + 2*static_cast<size_t>(g.ktot)*nchunk)),
                                "hipMalloc(force)"));
            MHH_CHECK(check_hip(hipMalloc(&c->force_dz, sizeof(double)*g.kcells), "hipMalloc(force)"));
            MHH_CHECK(check_hip(hipMemcpy(c->force_dz, c->h_dz.data(), sizeof(double)*g.kcells,
                                          hipMemcpyHostToDevice), "hipMemcpy(force)"));
        }
        mhh::Timer _t(c, "force");
        double* part = c->force_buf + 1;
        const Plane_fields<TF> uv{{static_cast<const TF*>(c->f.u), static_cast<const TF*>(c->f.ut)}};
        MHH_CHECK(plane_sums<TF>(c, uv, 2, g.kstart, g.ktot, part));
        fixed_flux_force_g<<<1, FT, 0, c->stream>>>(part, c->force_buf, c->force_dz + g.kstart, nchunk, g.ktot,
                                                    static_cast<double>(g.itot)*g.jtot, uflux, utrans, 1./dt,
                                                    c->h_zh[g.kend]);
        add_force_g<TF><<<grid3(g, g.kstart, g.kend), dim3(BX, BY), 0, c->stream>>>(
                static_cast<TF*>(c->f.ut), c->force_buf, g);
        return check_launch("force");
    }
}

extern "C" {

int mhh_force_fixed_flux(mhh_ctx* c, double uflux, double utrans, double dt)
{
    MHH_REQUIRE_BOUND(c);
    MHH_NOT_IN_BATCH(c, "mhh_force_fixed_flux");
    if (!(dt > 0.)) return mhh::fail(MHH_EINVAL, "mhh_force_fixed_flux: dt must be positive");
    MHH_CHECK(mhh::settle_tendencies(c));
    return c->precision == MHH_FP64 ? fixed_flux<double>(c, uflux, utrans, dt)
                                    : fixed_flux<float>(c, uflux, utrans, dt);
}

} // extern "C"
