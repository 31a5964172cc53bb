// mhh_rowfft.hip -- the x and y transforms of the pressure projection for
// every length that has no kernel of its own (mhh_rowfft.h: lane groups,
// a few passes): the forward x transform with the right-hand side of
// Pres_2::input (src/pres_2.cxx:155-196) evaluated into its first pass, the y
// transforms in place on the spectrum's rows, and the inverse x transform into
// the ghosted p.  They replace FFTW's R2HC/HC2R and their per-slice order
// (src/fft.cxx:338-452), as the kernels for 128, 256 and 512 points do.
//
// What bounds them: the memory traffic of one pass over the fields (x, forward)
// or the spectrum, and on small grids the latency of the passes.  Measured, against
// the block-wide engine (a wave per row, block barriers between passes) that they
// replace:
//   768 x 384 x 256 FP64: forward x 956 us (7 passes over the fields, 4.5 TB/s;
//     1629), y 382 (416), inverse x 384 (764)
//   90 x 75 x 60 FP64: 14.3, 7.9, 8.9 us (15.9, 8.9, 13.1)
// and where that engine had only its ping-pong fallback (mhh_fft.h): the projection
// of 960 x 500 x 58 FP64 1.36 ms instead of 5.00.
#include <algorithm>

#include "mhh_batch.h"
#include "mhh_rowfft.h"

namespace
{
    using namespace mhh;

    // Waves per block: a wave transforms 64/L rows (pairs of real rows in x).
    // FP32 blocks of the x transforms take eight, so that a block writes and
    // reads 128-byte segments of C[k][kx][.] also with one pair per wave.
    constexpr int YWAVES = 4;
    template<typename TF> constexpr int xw() { return sizeof(TF) == 8 ? 4 : 8; }

    // The row group of block b of nb (nb a multiple of 8): XCD x = b mod 8 owns
    // the groups [x cpx, (x+1) cpx) and takes them level by level, so that the w
    // and wt planes of level k+1 are read again by the same XCD a little
    // later (its own L2).  With few groups the XCDs would be uneven:
    // linear then (cpx = 0), each XCD a contiguous range of (level, group).
    __device__ __forceinline__ bool row_group(int b, int nb, int nbj, int cpx, int nlev, int& bj, int& k)
    {
        if (cpx > 0)
        {
            const int li = b >> 3;
            k = li / cpx;
            bj = (b & 7)*cpx + li % cpx;
            return bj < nbj && k < nlev;
        }
        const int t = xcd_tile(b, nb);
        k = t / nbj;
        bj = t - k*nbj;
        return k < nlev;
    }

    struct Xgrid { int nbj, cpx, nb; };

    inline Xgrid xgrid(int rows, int per, int nlev)
    {
        Xgrid x;
        x.nbj = (rows + per - 1)/per;
        x.cpx = (x.nbj % 8 == 0 || x.nbj >= 64) ? (x.nbj + 7)/8 : 0;
        x.nb = x.cpx ? 8*x.cpx*nlev : xcd_blocks(x.nbj*nlev);
        return x;
    }

    // Right-hand side of Pres_2::input at the interior point (x, row) of the two
    // rows a pair packs; the expression of pres_in_g (mhh_pres.hip).
    template<typename TF>
    struct Row_rhs
    {
        const TF* __restrict__ u; const TF* __restrict__ v; const TF* __restrict__ w;
        const TF* __restrict__ ut; const TF* __restrict__ vt; const TF* __restrict__ wt;
        TF rk, rhk, rhkp, dzk, dxi, dyi, dti;
        int n, kk, a, b, an, bn;    // offsets of x = 0 in the rows a and b and in their north neighbours (halo rows)
        int atn, btn;               // the same wrapped into the interior, for the tendencies
        __device__ __forceinline__ cplx<TF> operator()(int x) const
        {
            const int xe = x + 1 == n ? 0 : x + 1;
            auto one = [&](int o, int on, int otn) {
                const int i = o + x;
                return rk * ( (ut[o+xe] + u[i+1] * dti) - (ut[i] + u[i] * dti) ) * dxi
                     + rk * ( (vt[otn+x] + v[on+x] * dti) - (vt[i] + v[i] * dti) ) * dyi
                     + ( rhkp * (wt[i+kk] + w[i+kk] * dti)
                       - rhk  * (wt[i   ] + w[i   ] * dti) ) * dzk;
            };
            cplx<TF> z;
            z.x = one(a, an, atn);
            z.y = one(b, bn, btn);
            return z;
        }
    };

    // The table of roots into LDS.
    template<typename TF>
    __device__ __forceinline__ void load_roots(cplx<TF>* tws, const double2* __restrict__ tw, int n, int tid, int nthr)
    {
        for (int t = tid; t < n; t += nthr) { cplx<TF> z; z.x = TF(tw[t].x); z.y = TF(tw[t].y); tws[lpad(t)] = z; }
    }

    // Forward x transform of the pairs of real rows (j, j+1) of level k packed
    // as a + i b; writes C[k][kx][j] for kx <= itot/2.  The rows are the right-hand
    // side evaluated here or (P, mixed mode) read from the dense array P minus the
    // plane mean pmean[k], whose mode the FP64 path solves (DENSE, a kernel of
    // its own: chosen at run time, it kept the right-hand side's loads from being
    // issued together, and the projection of 360 x 250 x 100 FP32 took 343 us
    // instead of 286).
    template<typename TF, int VALS, int ARITH, bool DENSE>
    __device__ __forceinline__ void row_x_fwd_g(cplx<TF>* __restrict__ C, const Row_plan& p, const double2* __restrict__ tw,
                                                const TF* __restrict__ P, const double* __restrict__ pmean,
                                                const TF* __restrict__ u, const TF* __restrict__ v, const TF* __restrict__ w,
                                                const TF* __restrict__ ut, const TF* __restrict__ vt, const TF* __restrict__ wt,
                                                const TF* __restrict__ dzi, const TF* __restrict__ rho,
                                                const TF* __restrict__ rhoh, TF dxi, TF dyi, TF dti, int nw, Xgrid xg, Gd g,
                                                const Bid& bid_)
    {
        using T = cplx<TF>;
        extern __shared__ unsigned char smem_raw[];
        T* tws = reinterpret_cast<T*>(smem_raw);
        const int n = p.n, nx = n/2 + 1, M = g.jtot, stride = row_stride(n);
        T* rows = tws + lpad(n - 1) + 1;
        int bj, k;
        if (!row_group(bid_.x, bid_.nx, xg.nbj, xg.cpx, g.ktot, bj, k)) return;
        const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
        const int L = 1 << p.lsh, l = lane & (L - 1), rpw = 64 >> p.lsh;
        const int rl = wv*rpw + (lane >> p.lsh);       // the group's row pair in the block
        const int RP = nw*rpw;
        const int j0 = bj*2*RP, ja = j0 + 2*rl;
        load_roots<TF>(tws, tw, n, tid, 64*nw);
        T* row = rows + rl*stride;

        const int kc = k + g.kgc, base = g.igc + g.jgc*g.icells + kc*g.ijcells;
        // rows past the last are read as the last (in bounds) and not stored; an
        // odd last row is packed with zero, so that it is rounded by itself
        const int jra = min(ja, M - 1), jrb = min(ja + 1, M - 1);
        const bool pair = ja + 1 < M;
        const Row_rhs<TF> rhs{u, v, w, ut, vt, wt, rho[kc], rhoh[kc], rhoh[kc+1], dzi[kc], dxi, dyi, dti, n, g.ijcells,
                        base + jra*g.icells, base + jrb*g.icells, base + (jra + 1)*g.icells, base + (jrb + 1)*g.icells,
                        base + (jra + 1 == M ? 0 : jra + 1)*g.icells, base + (jrb + 1 == M ? 0 : jrb + 1)*g.icells};
        // a lane's elements in steps of four, their loads in flight together
        constexpr int RU = 4;
        const double m = DENSE ? pmean[k] : 0.;
        const TF* __restrict__ Pa = P + (static_cast<size_t>(k)*M + jra)*n;
        const TF* __restrict__ Pb = P + (static_cast<size_t>(k)*M + jrb)*n;
        for (int x0 = l; x0 < n; x0 += RU*L)
        {
            T z[RU];
            if constexpr (DENSE)
            {
                #pragma unroll
                for (int q = 0; q < RU; ++q)
                {
                    const int x = min(x0 + q*L, n - 1);
                    z[q].x = Pa[x]; z[q].y = Pb[x];
                }
                #pragma unroll
                for (int q = 0; q < RU; ++q)
                {
                    z[q].x = TF(double(z[q].x) - m);
                    z[q].y = pair ? TF(double(z[q].y) - m) : TF(0);
                }
            }
            else
            {
                #pragma unroll
                for (int q = 0; q < RU; ++q)
                {
                    z[q] = rhs(min(x0 + q*L, n - 1));
                    if (!pair) z[q].y = TF(0);
                }
            }
            #pragma unroll
            for (int q = 0; q < RU; ++q)
                if (x0 + q*L < n) row[lpad(x0 + q*L)] = z[q];
        }
        __syncthreads();   // the roots
        row_fft<TF, VALS, ARITH, ROW_X_FWD>(row, tws, p, l);
        __syncthreads();
        // The half-spectra of the rows a, b from Z = FFT(a + i b): Xa =
        // (Z[k] + conj Z[-k])/2, Xb = (Z[k] - conj Z[-k])/(2i), into C[k][kx][j],
        // consecutive threads on consecutive pairs
        T* Ck = C + static_cast<size_t>(k)*nx*M;
        const int psh = 31 - __clz(RP);
        for (int idx = tid; idx < nx*RP; idx += 64*nw)
        {
            const int kx = idx >> psh, r = idx & (RP - 1), j = j0 + 2*r;
            const T* Sr = rows + r*stride;
            const T z = Sr[lpad(kx)], c = Sr[lpad(kx == 0 ? 0 : n - kx)];
            T xa, xb;
            xa.x = (z.x + c.x)*TF(0.5); xa.y = (z.y - c.y)*TF(0.5);
            xb.x = (z.y + c.y)*TF(0.5); xb.y = (c.x - z.x)*TF(0.5);
            T* __restrict__ d = Ck + static_cast<size_t>(kx)*M + j;
            if (j < M) d[0] = xa;
            if (j + 1 < M) d[1] = xb;
        }
    }

    template<typename TF, int VALS, int ARITH, bool DENSE>
    struct row_x_fwd_k
    {
        static constexpr int NT = 64*xw<TF>(), MINB = 0;
        cplx<TF>* C; Row_plan p; const double2* tw; const TF* P; const double* pmean; const TF* u; const TF* v; const TF* w; const TF* ut;
        const TF* vt; const TF* wt; const TF* dzi; const TF* rho; const TF* rhoh; TF dxi; TF dyi; TF dti; int nw; Xgrid xg;
        Gd g;
        __device__ __forceinline__ void operator()(const Bid& bid_) const
        {
            row_x_fwd_g<TF, VALS, ARITH, DENSE>(C, p, tw, P, pmean, u, v, w, ut, vt, wt, dzi, rho, rhoh, dxi, dyi, dti, nw, xg, g,
                                         bid_);
        }
    };

    // The same outside a batch, with the pointers as __restrict__ kernel
    // parameters: the right-hand side's loads of a lane are then issued together.
    template<typename TF, int VALS, int ARITH, bool DENSE>
    __global__ void __launch_bounds__(64*xw<TF>()) row_x_fwd_direct(
            cplx<TF>* __restrict__ C, Row_plan p, const double2* __restrict__ tw, const TF* __restrict__ P,
            const double* __restrict__ pmean,
            const TF* __restrict__ u, const TF* __restrict__ v, const TF* __restrict__ w,
            const TF* __restrict__ ut, const TF* __restrict__ vt, const TF* __restrict__ wt,
            const TF* __restrict__ dzi, const TF* __restrict__ rho, const TF* __restrict__ rhoh,
            TF dxi, TF dyi, TF dti, int nw, Xgrid xg, Gd g)
    {
        row_x_fwd_g<TF, VALS, ARITH, DENSE>(C, p, tw, P, pmean, u, v, w, ut, vt, wt, dzi, rho, rhoh, dxi, dyi, dti, nw, xg, g,
                              Bid{static_cast<int>(blockIdx.x), 0, 0, static_cast<int>(gridDim.x), 1, 1});
    }

    // y transform of nrows contiguous rows of C in place, a lane group per row;
    // waves walk the rows with a stride.  INV divides by jtot (src/fft.cxx:420).
    template<typename TF, int VALS, int ARITH, bool INV>
    __device__ __forceinline__ void row_y_g(cplx<TF>* __restrict__ C, const Row_plan& p, const double2* __restrict__ tw,
                                            int nrows, int nw, const Bid& bid_)
    {
        using T = cplx<TF>;
        extern __shared__ unsigned char smem_raw[];
        T* tws = reinterpret_cast<T*>(smem_raw);
        const int n = p.n;
        const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
        const int L = 1 << p.lsh, l = lane & (L - 1), rpw = 64 >> p.lsh, sub = lane >> p.lsh;
        load_roots<TF>(tws, tw, n, tid, 64*nw);
        __syncthreads();
        T* row = tws + lpad(n - 1) + 1 + (wv*rpw + sub)*row_stride(n);
        const TF ni = TF(1)/TF(n);   // exact for powers of two
        for (int r0 = (bid_.x*nw + wv)*rpw; r0 < nrows; r0 += bid_.nx*nw*rpw)
        {
            const int r = r0 + sub;
            const bool active = r < nrows;
            T* __restrict__ Cr = C + static_cast<size_t>(min(r, nrows - 1))*n;
            constexpr int YU = 8;    // loads of a lane in flight
            for (int x0 = l; x0 < n; x0 += YU*L)
            {
                T z[YU];
                #pragma unroll
                for (int q = 0; q < YU; ++q) z[q] = Cr[min(x0 + q*L, n - 1)];
                #pragma unroll
                for (int q = 0; q < YU; ++q)
                    if (x0 + q*L < n) row[lpad(x0 + q*L)] = z[q];
            }
            row_fft<TF, VALS, ARITH, INV ? ROW_Y_INV : ROW_Y_FWD>(row, tws, p, l);
            if (active)
                for (int x = l; x < n; x += L)
                {
                    T o = row[lpad(x)];
                    if (INV) { o.x *= ni; o.y *= ni; }
                    Cr[x] = o;
                }
            wave_lds_sync();
        }
    }

    template<typename TF, int VALS, int ARITH, bool INV>
    struct row_y_k
    {
        static constexpr int NT = 256, MINB = 0;
        cplx<TF>* C; Row_plan p; const double2* tw; int nrows; int nw;
        __device__ __forceinline__ void operator()(const Bid& bid_) const
        {
            row_y_g<TF, VALS, ARITH, INV>(C, p, tw, nrows, nw, bid_);
        }
    };

    // The bins kx and n - kx of the packed spectrum Z = Xa + i Xb of two real rows.
    template<typename T>
    __device__ __forceinline__ void put_bins(T* row, int kx, int n, T xa, T xb)
    {
        T z; z.x = xa.x - xb.y; z.y = xa.y + xb.x;
        row[lpad(kx)] = z;
        if (kx > 0 && 2*kx < n)
        {
            z.x = xa.x + xb.y; z.y = xb.x - xa.y;
            row[lpad(n - kx)] = z;
        }
    }

    // Inverse x transform (divides by itot, src/fft.cxx:446) of the row pairs of
    // C[k][kx][j] into the ghosted p: interior rows, their periodic images in the
    // y halo, the x halo columns and, at the lowest level, the ghost level
    // below (Pres_2::solve tail, src/pres_2.cxx:336-361).
    template<typename TF, int VALS, int ARITH>
    __device__ __forceinline__ void row_x_bwd_g(const cplx<TF>* __restrict__ C, TF* __restrict__ pf, const Row_plan& p,
                                                const double2* __restrict__ tw, int nw, Xgrid xg, Gd g, const Bid& bid_)
    {
        using T = cplx<TF>;
        extern __shared__ unsigned char smem_raw[];
        T* tws = reinterpret_cast<T*>(smem_raw);
        const int n = p.n, nx = n/2 + 1, M = g.jtot, stride = row_stride(n);
        T* rows = tws + lpad(n - 1) + 1;
        int bj, k;
        if (!row_group(bid_.x, bid_.nx, xg.nbj, xg.cpx, g.ktot, bj, k)) return;
        const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6, nthr = 64*nw;
        const int L = 1 << p.lsh, l = lane & (L - 1), rpw = 64 >> p.lsh;
        const int rl = wv*rpw + (lane >> p.lsh);
        const int RP = nw*rpw, psh = 31 - __clz(RP);
        const int j0 = bj*2*RP;
        // The packed spectrum Z = Xa + i Xb of a pair over all n bins from its two
        // half-spectra (Hermitian); consecutive
        // threads on consecutive pairs, several loads of a thread in flight
        const T* Ck = C + static_cast<size_t>(k)*nx*M;
        constexpr int SB = 4;
        for (int i0 = tid; i0 < nx*RP; i0 += SB*nthr)
        {
            T va[SB], vb[SB];
            #pragma unroll
            for (int q = 0; q < SB; ++q)
            {
                const int idx = min(i0 + q*nthr, nx*RP - 1);
                const int j = j0 + 2*(idx & (RP - 1));
                const T* Cj = Ck + static_cast<size_t>(idx >> psh)*M;
                va[q] = Cj[min(j, M - 1)]; vb[q] = Cj[min(j + 1, M - 1)];
            }
            #pragma unroll
            for (int q = 0; q < SB; ++q)
            {
                const int idx = i0 + q*nthr;
                if (idx < nx*RP)
                {
                    const int kx = idx >> psh;
                    T* Sr = rows + (idx & (RP - 1))*stride;
                    T xa = va[q], xb = vb[q];
                    if (kx == 0 || 2*kx == n) { xa.y = TF(0); xb.y = TF(0); }   // real bins of a real row
                    put_bins(Sr, kx, n, xa, xb);
                }
            }
        }
        if ((M & 1) && j0 + 2*RP > M)
        {
            // the block holds an odd last row, read above as its own partner: packed
            // with zero, so that it is rounded by itself (here and not in the loop
            // above, whose loads a condition holds up: 768 x 384 x 256 FP64 376 and 396 us)
            __syncthreads();
            T* Sr = rows + ((M - 1 - j0) >> 1)*stride;
            const T zero{TF(0), TF(0)};
            for (int kx = tid; kx < nx; kx += nthr)
            {
                T xa = Ck[static_cast<size_t>(kx)*M + M - 1];
                if (kx == 0 || 2*kx == n) xa.y = TF(0);
                put_bins(Sr, kx, n, xa, zero);
            }
        }
        load_roots<TF>(tws, tw, n, tid, nthr);
        __syncthreads();
        T* row = rows + rl*stride;
        row_fft<TF, VALS, ARITH, ROW_X_INV>(row, tws, p, l);
        const TF ni = TF(1)/TF(n);   // exact for powers of two
        TF* __restrict__ pk = pf + static_cast<size_t>(k + g.kgc)*g.ijcells;
        for (int h = 0; h < 2; ++h)
        {
            const int j = j0 + 2*rl + h;
            if (j >= M) continue;
            // the interior row and, within jgc of an edge, its periodic images
            int dst[3]; int nd = 0;
            dst[nd++] = j + g.jgc;
            if (j >= M - g.jgc) dst[nd++] = j - (M - g.jgc);
            if (j < g.jgc) dst[nd++] = g.jend + j;
            for (int x = l; x < g.icells; x += L)
            {
                // ghosted column x holds interior column x - igc, wrapped
                int xi = x - g.igc;
                xi = xi < 0 ? xi + n : xi >= n ? xi - n : xi;
                const T z = row[lpad(xi)];
                const TF val = (h ? z.y : z.x)*ni;
                for (int e = 0; e < nd; ++e)
                {
                    TF* __restrict__ pr = pk + x + static_cast<size_t>(dst[e])*g.icells;
                    *pr = val;
                    if (k == 0) pr[-g.ijcells] = val;
                }
            }
        }
    }

    template<typename TF, int VALS, int ARITH>
    struct row_x_bwd_k
    {
        static constexpr int NT = 64*xw<TF>(), MINB = 0;
        const cplx<TF>* C; TF* pf; Row_plan p; const double2* tw; int nw; Xgrid xg; Gd g;
        __device__ __forceinline__ void operator()(const Bid& bid_) const
        {
            row_x_bwd_g<TF, VALS, ARITH>(C, pf, p, tw, nw, xg, g, bid_);
        }
    };

    // Calls f with the plan's instance, (values per lane, arithmetic).
    template<typename TF, typename F>
    void with_instance(const Row_plan& p, F f)
    {
        auto arith = [&](auto v) {
            if (p.arith == ROW_DIRECT) return f(v, std::integral_constant<int, ROW_DIRECT>{});
            f(v, std::integral_constant<int, ROW_RADIX8>{});
        };
        if (p.vals == ROW_VALS) arith(std::integral_constant<int, ROW_VALS>{});
        else arith(std::integral_constant<int, ROW_VALS_WIDE>{});
    }

    template<typename TF>
    size_t row_lds(const Row_plan& p, int nw)
    {
        return (static_cast<size_t>(lpad(p.n - 1) + 1) + static_cast<size_t>(nw)*(64 >> p.lsh)*row_stride(p.n))
               *sizeof(cplx<TF>);
    }

    // Waves of a block: most, unless the rows of the launch need fewer or their LDS
    // would leave less than two blocks on a CU.
    template<typename TF>
    int row_waves(const Row_plan& p, int most, long long rows)
    {
        int nw = most;
        while (nw > 1 && (static_cast<long long>(nw/2)*(64 >> p.lsh) >= rows || row_lds<TF>(p, nw) > 80*1024)) nw /= 2;
        return nw;
    }
}

namespace mhh
{
    void row_plans_init(mhh_ctx* c)
    {
        const Gd& g = c->gd;
        make_row_plan(g.itot, static_cast<long long>(g.jtot + 1)/2*g.ktot, c->row_px);
        make_row_plan(g.jtot, static_cast<long long>(g.itot/2 + 1)*g.ktot, c->row_py);
    }

    template<typename TF, typename T>
    int row_x_fwd(mhh_ctx* c, const TF* P, T* C, const double* tw, const Prof<TF>& pr, TF dxi, TF dyi, TF dti)
    {
        const Gd& g = c->gd;
        const Row_plan& p = c->row_px;
        const int nw = row_waves<TF>(p, xw<TF>(), (g.jtot + 1)/2), rp = nw*(64 >> p.lsh);
        const Xgrid xg = xgrid(g.jtot, 2*rp, g.ktot);
        const size_t lds = row_lds<TF>(p, nw);
        const auto* t2 = reinterpret_cast<const double2*>(tw);
        const TF* u = static_cast<const TF*>(c->f.u); const TF* v = static_cast<const TF*>(c->f.v);
        const TF* w = static_cast<const TF*>(c->f.w); const TF* ut = static_cast<const TF*>(c->f.ut);
        const TF* vt = static_cast<const TF*>(c->f.vt); const TF* wt = static_cast<const TF*>(c->f.wt);
        {
            mhh::Timer _t(c, P ? "fft_x_fwd" : "pres_in_fft_x");
            with_instance<TF>(p, [&](auto vc, auto ac) {
                constexpr int V = decltype(vc)::value, A = decltype(ac)::value;
                auto go = [&](auto dc) {
                    constexpr bool D = decltype(dc)::value;
                    if (c->rec)
                        record(c, row_x_fwd_k<TF, V, A, D>{C, p, t2, P, c->pm_mean, u, v, w, ut, vt, wt, pr.dzi, pr.rhoref,
                                                           pr.rhorefh, dxi, dyi, dti, nw, xg, g}, xg.nb, 64*nw, lds);
                    else
                        row_x_fwd_direct<TF, V, A, D><<<xg.nb, 64*nw, lds, c->stream>>>(C, p, t2, P, c->pm_mean, u, v, w, ut,
                            vt, wt, pr.dzi, pr.rhoref, pr.rhorefh, dxi, dyi, dti, nw, xg, g);
                };
                if constexpr (sizeof(TF) == 4)
                    if (P) return go(std::true_type{});
                go(std::false_type{});
            });
        }
        return check_launch(P ? "fft_x_fwd" : "pres_in_fft_x");
    }

    template<typename TF, typename T>
    int row_y(mhh_ctx* c, T* C, const double* tw, int sign, int nrows, const char* name)
    {
        const Row_plan& p = c->row_py;
        const int nw = row_waves<TF>(p, YWAVES, nrows), rp = nw*(64 >> p.lsh);
        const size_t lds = row_lds<TF>(p, nw);
        // about as many blocks as run at once, each walking its rows
        const int nb = std::max(1, std::min((nrows + rp - 1)/rp, 8*256));
        const auto* t2 = reinterpret_cast<const double2*>(tw);
        {
            mhh::Timer _t(c, name);
            with_instance<TF>(p, [&](auto vc, auto ac) {
                constexpr int V = decltype(vc)::value, A = decltype(ac)::value;
                if (sign < 0) launch(c, row_y_k<TF, V, A, false>{C, p, t2, nrows, nw}, nb, 64*nw, lds);
                else launch(c, row_y_k<TF, V, A, true>{C, p, t2, nrows, nw}, nb, 64*nw, lds);
            });
        }
        return check_launch(name);
    }

    template<typename TF, typename T>
    int row_x_bwd(mhh_ctx* c, const T* C, TF* pf, const double* tw)
    {
        const Gd& g = c->gd;
        const Row_plan& p = c->row_px;
        const int nw = row_waves<TF>(p, xw<TF>(), (g.jtot + 1)/2), rp = nw*(64 >> p.lsh);
        const Xgrid xg = xgrid(g.jtot, 2*rp, g.ktot);
        const size_t lds = row_lds<TF>(p, nw);
        const auto* t2 = reinterpret_cast<const double2*>(tw);
        {
            mhh::Timer _t(c, "fft_x_bwd");
            with_instance<TF>(p, [&](auto vc, auto ac) {
                launch(c, row_x_bwd_k<TF, decltype(vc)::value, decltype(ac)::value>{C, pf, p, t2, nw, xg, g}, xg.nb, 64*nw,
                       lds);
            });
        }
        return check_launch("fft_x_bwd");
    }

    template int row_x_fwd<float, float2>(mhh_ctx*, const float*, float2*, const double*, const Prof<float>&, float, float,
                                              float);
    template int row_x_fwd<double, double2>(mhh_ctx*, const double*, double2*, const double*, const Prof<double>&, double,
                                                double, double);
    template int row_y<float, float2>(mhh_ctx*, float2*, const double*, int, int, const char*);
    template int row_y<double, double2>(mhh_ctx*, double2*, const double*, int, int, const char*);
    template int row_x_bwd<float, float2>(mhh_ctx*, const float2*, float*, const double*);
    template int row_x_bwd<double, double2>(mhh_ctx*, const double2*, double*, const double*);
}
