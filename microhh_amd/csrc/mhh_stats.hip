// mhh_stats.hip -- horizontal means of the fields (Field3d_operators::
// calc_mean_profile, src/field3d_operators.cxx:46-66), used by the buffer
// with swupdate and by the diagnostics.
#include <algorithm>
#include <vector>

#include "mhh_batch.h"

namespace
{
    using namespace mhh;

    constexpr int MT = 256;

    // Partial plane sums in FP64: block (chunk, level, field) sums `rows` rows of
    // one level, a wave per row with four loads of a lane in flight, and
    // writes part[(field*nk + level)*nchunk + chunk].  A fixed order, so the
    // result is reproducible.  Reads are what bounds it, so the launch needs enough
    // blocks to fill the chip: at 768 x 384 x 256 FP64 one block per level took
    // 624 us per field (1.0 TB/s), the chunks 240 us for two (5.0 TB/s).
    template<typename TF>
    __global__ void __launch_bounds__(MT) plane_part_g(Plane_fields<TF> f, double* __restrict__ part, int k0, int rows, Gd g)
    {
        __shared__ double s[MT/64];
        const TF* __restrict__ fld = f.a[blockIdx.z];
        const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
        const TF* __restrict__ lev = fld + static_cast<size_t>(k0 + blockIdx.y)*g.ijcells + g.istart
                                   + static_cast<size_t>(g.jstart)*g.icells;
        const int j1 = min(static_cast<int>(blockIdx.x + 1)*rows, g.jtot);
        double acc[4] = {0., 0., 0., 0.};
        for (int j = blockIdx.x*rows + wv; j < j1; j += MT/64)
        {
            const TF* __restrict__ row = lev + static_cast<size_t>(j)*g.icells;
            for (int i = lane; i < g.itot; i += 256)
            {
                TF v[4];
                #pragma unroll
                for (int q = 0; q < 4; ++q) v[q] = row[min(i + 64*q, g.itot - 1)];
                #pragma unroll
                for (int q = 0; q < 4; ++q) acc[q] += i + 64*q < g.itot ? static_cast<double>(v[q]) : 0.;
            }
        }
        double sum = (acc[0] + acc[1]) + (acc[2] + acc[3]);
        #pragma unroll
        for (int o = 32; o > 0; o >>= 1) sum += __shfl_xor(sum, o);
        if (lane == 0) s[wv] = sum;
        __syncthreads();
        if (threadIdx.x == 0)
            part[(static_cast<size_t>(blockIdx.z)*gridDim.y + blockIdx.y)*gridDim.x + blockIdx.x]
                = (s[0] + s[1]) + (s[2] + s[3]);
    }

    // The means of the levels from their partial sums, one thread per level
    // of a field (nk: of all fields).
    __global__ void __launch_bounds__(64) plane_fold_g(const double* __restrict__ part, double* __restrict__ prof,
                                                       int nchunk, int nk, double npoints)
    {
        const int k = blockIdx.x*64 + threadIdx.x;
        if (k >= nk) return;
        double sum = 0.;
        for (int q = 0; q < nchunk; ++q) sum += part[static_cast<size_t>(k)*nchunk + q];
        prof[k] = sum/npoints;
    }
}

namespace
{
    // Per level of the interior, the sums over the level's points of the
    // three integrands of Fields::check_momentum/check_tke/check_mass
    // (src/fields.cxx:252-340): interp2 of u, v, w to the cell centre, the
    // same of their squares, and the first scalar.  FP64 accumulation; part
    // receives 3 values per level, the dz weighting is done by the caller.
    template<typename TF>
    __global__ void __launch_bounds__(MT) check_sums_g(const TF* __restrict__ u, const TF* __restrict__ v,
                                                       const TF* __restrict__ w, const TF* __restrict__ s,
                                                       Gd g, double* __restrict__ part)
    {
        __shared__ double sm[3][MT];
        const int k = g.kstart + blockIdx.x;
        const int jj = g.icells, kk = g.ijcells;
        const int n = g.itot*g.jtot;
        double am = 0., ae = 0., as = 0.;
        for (int t = threadIdx.x; t < n; t += MT)
        {
            const int j = t / g.itot, i = t - j*g.itot;
            const int ijk = (i + g.istart) + (j + g.jstart)*jj + k*kk;
            const double u0 = u[ijk], u1 = u[ijk+1], v0 = v[ijk], v1 = v[ijk+jj], w0 = w[ijk], w1 = w[ijk+kk];
            am += 0.5*(u0 + u1) + 0.5*(v0 + v1) + 0.5*(w0 + w1);
            ae += 0.5*(u0*u0 + u1*u1) + 0.5*(v0*v0 + v1*v1) + 0.5*(w0*w0 + w1*w1);
            if (s) as += static_cast<double>(s[ijk]);
        }
        sm[0][threadIdx.x] = am; sm[1][threadIdx.x] = ae; sm[2][threadIdx.x] = as;
        __syncthreads();
        for (int h = MT/2; h > 0; h >>= 1)
        {
            if (threadIdx.x < h)
                for (int q = 0; q < 3; ++q) sm[q][threadIdx.x] += sm[q][threadIdx.x + h];
            __syncthreads();
        }
        if (threadIdx.x < 3) part[3*blockIdx.x + threadIdx.x] = sm[threadIdx.x][0];
    }

    template<typename TF>
    int check_sums(mhh_ctx* c, double* mom, double* tke, double* mass)
    {
        const Gd& g = c->gd;
        MHH_CHECK(ensure_reduction(c, 3*g.ktot));
        const TF* s = c->f.nscalars > 0 ? static_cast<const TF*>(c->f.s[0]) : nullptr;
        {
            mhh::Timer _t(c, "check_sums");
            check_sums_g<TF><<<g.ktot, MT, 0, c->stream>>>(static_cast<const TF*>(c->f.u),
                    static_cast<const TF*>(c->f.v), static_cast<const TF*>(c->f.w), s, g, c->red);
        }
        MHH_CHECK(check_launch("check_sums"));
        std::vector<double> part(3*static_cast<size_t>(g.ktot));
        MHH_CHECK(check_hip(hipMemcpyAsync(part.data(), c->red, sizeof(double)*part.size(), hipMemcpyDeviceToHost,
                                           c->stream), "hipMemcpyAsync(check sums)"));
        MHH_CHECK(check_hip(hipStreamSynchronize(c->stream), "hipStreamSynchronize"));
        double sm = 0., se = 0., ss = 0., sdz = 0.;
        for (int k = 0; k < g.ktot; ++k)
        {
            const double dz = c->h_dz[g.kstart + k];
            sm += part[3*k]*dz; se += part[3*k+1]*dz; ss += part[3*k+2]*dz; sdz += dz;
        }
        // Fields::check_*: divided by itot*jtot*zsize (zsize = the sum of dz)
        const double vol = static_cast<double>(g.itot)*g.jtot*c->h_zh[g.kend];
        *mom = sm/vol;
        *tke = 0.5*se/vol;
        // a scalar held relative to an offset (mixed precision): the offset's share
        *mass = s ? ss/vol + c->s_offset[0]*(static_cast<double>(g.itot)*g.jtot*sdz)/vol : 0.;
        return 0;
    }
}

namespace mhh
{
    // Chunks of rows per level: about 2048 blocks for one field (8 per CU), at
    // least a wave's row each.
    int plane_chunks(const Gd& g)
    {
        const int want = std::max(1, 2048/g.kcells);
        const int rows = std::max(MT/64, (g.jtot + want - 1)/want);
        return (g.jtot + rows - 1)/rows;
    }

    template<typename TF>
    int plane_sums(mhh_ctx* c, const Plane_fields<TF>& f, int nf, int k0, int nk, double* part)
    {
        const Gd& g = c->gd;
        const int nchunk = plane_chunks(g), rows = (g.jtot + nchunk - 1)/nchunk;
        plane_part_g<TF><<<dim3(nchunk, nk, nf), MT, 0, c->stream>>>(f, part, k0, rows, g);
        return check_launch("plane_sums");
    }

    template<typename TF>
    int mean_profiles(mhh_ctx* c, const Plane_fields<TF>& f, int nf, double* part, double* prof)
    {
        const Gd& g = c->gd;
        mhh::Timer _t(c, "mean_profile");
        MHH_CHECK(plane_sums<TF>(c, f, nf, 0, g.kcells, part));
        plane_fold_g<<<(nf*g.kcells + 63)/64, 64, 0, c->stream>>>(part, prof, plane_chunks(g), nf*g.kcells,
                                                                  static_cast<double>(g.itot)*g.jtot);
        return check_launch("mean_profile");
    }

    template int plane_sums<double>(mhh_ctx*, const Plane_fields<double>&, int, int, int, double*);
    template int plane_sums<float>(mhh_ctx*, const Plane_fields<float>&, int, int, int, double*);
    template int mean_profiles<double>(mhh_ctx*, const Plane_fields<double>&, int, double*, double*);
    template int mean_profiles<float>(mhh_ctx*, const Plane_fields<float>&, int, double*, double*);
}

extern "C" int mhh_fields_check(mhh_ctx* c, double* mom, double* tke, double* mass)
{
    MHH_REQUIRE_BOUND(c);
    MHH_NOT_IN_BATCH(c, "mhh_fields_check");
    if (!mom || !tke || !mass) return mhh::fail(MHH_EINVAL, "mhh_fields_check: null output");
    return c->precision == MHH_FP64 ? check_sums<double>(c, mom, tke, mass) : check_sums<float>(c, mom, tke, mass);
}
