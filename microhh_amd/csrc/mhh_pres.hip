// mhh_pres.hip -- 2nd-order pressure projection (Pres_2, src/pres_2.cxx:64-422).
//
// Spectral layout.  The reference transforms with FFTW R2HC per k-slice along
// x then y (src/fft.cxx:338-394) and solves one tridiagonal system per
// halfcomplex entry.  Here the same eigen-decomposition is done with complex
// arithmetic: a real-to-complex transform in x (two real rows packed in one
// complex FFT), a complex transform in y, a Thomas solve per (kx, ky) mode
// with the reference's coefficients and boundary rows, and the inverse path.
// The solution p is the same up to rounding; only the intermediate
// representation differs.
//
// Memory layout of the spectrum (complex, in tmp1):
//     C[k][kx][j],  k < ktot, kx <= itot/2, j < jtot   (j contiguous)
// so that the y transforms read contiguous rows and the Thomas solve reads
// consecutive modes with consecutive threads.  The x transforms transpose
// through LDS to write/read 2*RB consecutive j values per kx.
//
// FFT: Stockham autosort with twiddles from a host-computed table: a wave per row
// for 128, 256 and 512 points (here), lane groups for the other lengths
// (mhh_rowfft.hip), DFT-as-GEMM for 1024 in the mixed mode (mhh_dft.hip), and the
// ping-pong engine of mhh_fft.h for the lengths that have no lane-group plan (55
// of the 105 from 1025 to 2048, none below 1050, all above).
#include <algorithm>
#include <cmath>
#include <type_traits>
#include <vector>

#include "mhh_batch.h"
#include "mhh_fft.h"
#include "mhh_stencil.h"

namespace
{
    using namespace mhh;

    // Pres_2::input (src/pres_2.cxx:155-196): divergence of u/dt + ut into the
    // dense [k][j][i] array P.  The periodic neighbours of ut and vt at the east
    // and north edges are read by index wrap instead of through their halos.
    // A thread takes its column through PIN_KCHUNK levels and carries the
    // vertical flux through the top face to the next level, so w and wt are
    // read once.
    constexpr int PIN_KCHUNK = 16;

    template<typename TF>
    __device__ __forceinline__ void pres_in_g(
            TF* __restrict__ P, const TF* __restrict__ u, const TF* __restrict__ v, const TF* __restrict__ w,
            const TF* __restrict__ ut, const TF* __restrict__ vt, const TF* __restrict__ wt,
            const TF* __restrict__ dzi, const TF* __restrict__ rho, const TF* __restrict__ rhoh,
            TF dxi, TF dyi, TF dti, Gd g, const Bid& bid_)
    {
        const int i = bid_.x*BX + threadIdx.x;
        const int j = bid_.y*BY + threadIdx.y;
        const int kb = bid_.z*PIN_KCHUNK, ke = min(kb + PIN_KCHUNK, g.ktot);
        if (i >= g.itot || j >= g.jtot) return;
        const int jj = g.icells, kk = g.ijcells;
        int ijk = i+g.igc + (j+g.jgc)*jj + (kb+g.kgc)*kk;
        const int de = (i+1 == g.itot) ? 1 - g.itot : 1;          // east neighbour of ut
        const int dn = (j+1 == g.jtot) ? jj - g.jtot*jj : jj;     // north neighbour of vt
        const size_t nplane = size_t(g.itot)*g.jtot;
        TF* __restrict__ Pk = P + i + size_t(j)*g.itot + kb*nplane;
        // the flux through the bottom face of the first level
        TF fb = rhoh[kb+g.kgc] * (wt[ijk] + w[ijk] * dti);
        for (int k = kb; k < ke; ++k)
        {
            const int kc = k + g.kgc;
            const TF ft = rhoh[kc+1] * (wt[ijk+kk] + w[ijk+kk] * dti);
            *Pk = rho[kc] * ( (ut[ijk+de] + u[ijk+1] * dti) - (ut[ijk] + u[ijk] * dti) ) * dxi
                + rho[kc] * ( (vt[ijk+dn] + v[ijk+jj] * dti) - (vt[ijk] + v[ijk] * dti) ) * dyi
                + ( ft - fb ) * dzi[kc];
            fb = ft;
            ijk += kk;
            Pk += nplane;
        }
    }

    template<typename TF>
    struct pres_in_k
    {
        static constexpr int NT = BX*BY, MINB = 0;
        TF* P; const TF* u; const TF* v; const TF* w; const TF* ut; const TF* vt; const TF* wt;
        const TF* dzi; const TF* rho; const TF* rhoh; TF dxi; TF dyi; TF dti; Gd g;
        __device__ __forceinline__ void operator()(const Bid& bid_) const
        {
            pres_in_g<TF>(P, u, v, w, ut, vt, wt, dzi, rho, rhoh, dxi, dyi, dti, g, bid_);
        }
    };

    // Inputs of Pres_2::input (src/pres_2.cxx:155-196) for the forward x
    // transform that evaluates the right-hand side while loading its rows.
    template<typename TF>
    struct Pin_args
    {
        const TF* __restrict__ u; const TF* __restrict__ v; const TF* __restrict__ w;
        const TF* __restrict__ ut; const TF* __restrict__ vt; const TF* __restrict__ wt;
        const TF* __restrict__ dzi; const TF* __restrict__ rho; const TF* __restrict__ rhoh;
        TF dxi, dyi, dti;
    };

    // P at interior point (i, j, k) (0-based), the expression of pres_in_g.
    template<typename TF>
    __device__ __forceinline__ TF pres_rhs(const Pin_args<TF>& a, int i, int j, int k, const Gd& g)
    {
        const int jj = g.icells, kk = g.ijcells;
        const int ijk = i+g.igc + (j+g.jgc)*jj + (k+g.kgc)*kk;
        const int ie = (i+1 == g.itot) ? ijk + 1 - g.itot : ijk + 1;
        const int jn = (j+1 == g.jtot) ? ijk + jj - g.jtot*jj : ijk + jj;
        const int kc = k + g.kgc;
        return a.rho[kc] * ( (a.ut[ie] + a.u[ijk+1] * a.dti) - (a.ut[ijk] + a.u[ijk] * a.dti) ) * a.dxi
             + a.rho[kc] * ( (a.vt[jn] + a.v[ijk+jj] * a.dti) - (a.vt[ijk] + a.v[ijk] * a.dti) ) * a.dyi
             + ( a.rhoh[kc+1] * (a.wt[ijk+kk] + a.w[ijk+kk] * a.dti)
               - a.rhoh[kc  ] * (a.wt[ijk   ] + a.w[ijk   ] * a.dti) ) * a.dzi[kc];
    }

    // Packed staging of the two half-spectra of a pair of real rows in n complex
    // slots: the DC (and, for even n, Nyquist) entries are real and share one
    // slot each as (row a, row b); every other kx holds (Xa, Xb) in two slots.
    __device__ __forceinline__ int stage_base(int kx, int n) { return (n & 1) ? 2*kx - 1 : 2*kx; }

    template<typename TF>
    __device__ __forceinline__ void unpack_pair(cplx<TF> z, cplx<TF> c, cplx<TF>& xa, cplx<TF>& xb)
    {
        // spectra of the real rows a, b from Z = FFT(a + i b): Xa = (Z[k] + conj(Z[-k]))/2,
        // Xb = (Z[k] - conj(Z[-k]))/(2i)
        xa.x = (z.x + c.x)*TF(0.5); xa.y = (z.y - c.y)*TF(0.5);
        xb.x = (z.y + c.y)*TF(0.5); xb.y = (c.x - z.x)*TF(0.5);
    }

    template<typename TF>
    __device__ __forceinline__ void stage_store(cplx<TF>* S, int kx, int n, cplx<TF> xa, cplx<TF> xb)
    {
        if (kx == 0) { cplx<TF> d; d.x = xa.x; d.y = xb.x; S[0] = d; }
        else if (2*kx == n) { cplx<TF> d; d.x = xa.x; d.y = xb.x; S[1] = d; }
        else { const int b = stage_base(kx, n); S[lpad(b)] = xa; S[lpad(b+1)] = xb; }
    }

    // The transforms of the lengths without a lane-group plan.
    // Forward x transform: RB complex rows per block, each packing two real
    // rows of P at level k; writes C[k][kx][j] for kx <= itot/2.
    template<typename TF>
    __device__ __forceinline__ void fft_x_fwd_g(const TF* __restrict__ P, cplx<TF>* __restrict__ C,
                                                const Plan& plan, const double2* __restrict__ tw, int RB, Gd g,
                                                const double* __restrict__ pmean, Pin_args<TF> pin, int fuse_in, const Bid& bid_)
    {
        using T = cplx<TF>;
        extern __shared__ unsigned char smem_raw[];
        const int n = plan.n, nx = n/2 + 1, M = g.jtot, re = row_elems(plan);
        T* rows = reinterpret_cast<T*>(smem_raw);
        const int row = threadIdx.y, lane = threadIdx.x;
        const int k = bid_.y;
        const int j0 = bid_.x*2*RB;              // first real row of the block
        const int ja = j0 + 2*row, jb = ja + 1;
        T* A = rows + row*re;
        const TF* Pk = P + static_cast<size_t>(k)*n*M;
        // mixed mode (pmean): the plane mean is solved separately in FP64
        const double m = !fuse_in && pmean ? pmean[k] : 0.;
        for (int x = lane; x < n; x += 64)
        {
            T z;
            if (fuse_in)
            {
                // the right-hand side evaluated here instead of in pres_in_g
                z.x = (ja < M) ? pres_rhs(pin, x, ja, k, g) : TF(0);
                z.y = (jb < M) ? pres_rhs(pin, x, jb, k, g) : TF(0);
            }
            else
            {
                z.x = (ja < M) ? TF(double(Pk[x + ja*n]) - m) : TF(0);
                z.y = (jb < M) ? TF(double(Pk[x + jb*n]) - m) : TF(0);
            }
            A[lpad(x)] = z;
        }
        __syncthreads();
        T* Z = fft_row_pingpong<TF>(A, A + row_half(n), plan, tw, -1, lane);
        // Stage the two half-spectra packed in n slots in the free buffer.
        const int soff = (Z == A) ? row_half(n) : 0;
        T* S = rows + row*re + soff;
        for (int kx = lane; kx < nx; kx += 64)
        {
            T xa, xb;
            unpack_pair<TF>(Z[lpad(kx)], Z[lpad((n - kx) % n)], xa, xb);
            stage_store<TF>(S, kx, n, xa, xb);
        }
        __syncthreads();
        // The block writes C[k][kx][j0 .. j0+2RB) with consecutive threads on consecutive j.
        const int nthr = 64*RB, tid = lane + 64*row;
        const int JB = 2*RB;
        T* Ck = C + static_cast<size_t>(k)*nx*M;
        for (int idx = tid; idx < nx*JB; idx += nthr)
        {
            const int kx = idx / JB, jl = idx % JB;
            const int r = jl >> 1, part = jl & 1;
            const int j = j0 + jl;
            if (j >= M) continue;
            const T* Sr = rows + r*re + soff;
            T val;
            if (kx == 0 || 2*kx == n)
            {
                const T d = Sr[kx == 0 ? 0 : 1];   // lpad(0) = 0, lpad(1) = 1
                val.x = part ? d.y : d.x; val.y = TF(0);
            }
            else
                val = Sr[lpad(stage_base(kx, n) + part)];
            Ck[static_cast<size_t>(kx)*M + j] = val;
        }
    }

    template<typename TF>
    struct fft_x_fwd_k
    {
        static constexpr int NT = 256, MINB = 0;
        const TF* P; cplx<TF>* C; Plan plan; const double2* tw; int RB; Gd g; const double* pmean;
        Pin_args<TF> pin; int fuse_in;
        __device__ __forceinline__ void operator()(const Bid& bid_) const
        {
            fft_x_fwd_g<TF>(P, C, plan, tw, RB, g, pmean, pin, fuse_in, bid_);
        }
    };

    // y transform (forward sign -1 or inverse +1) of RB contiguous rows of C;
    // the inverse divides by jtot as src/fft.cxx:420 does.
    template<typename TF>
    __device__ __forceinline__ void fft_y_g(cplx<TF>* __restrict__ C, const Plan& plan, const double2* __restrict__ tw,
                                            int sign, int nrows, int RB, const Bid& bid_)
    {
        using T = cplx<TF>;
        extern __shared__ unsigned char smem_raw[];
        const int n = plan.n, re = row_elems(plan);
        const int row = threadIdx.y, lane = threadIdx.x;
        const int r = bid_.x*RB + row;
        T* A = reinterpret_cast<T*>(smem_raw) + row*re;
        const bool active = r < nrows;
        T* Cr = C + static_cast<size_t>(active ? r : 0)*n;
        if (active)
            for (int x = lane; x < n; x += 64) A[lpad(x)] = Cr[x];
        __syncthreads();
        T* Z = fft_row_pingpong<TF>(A, A + row_half(n), plan, tw, sign, lane);
        if (!active) return;
        if (sign < 0)
            for (int x = lane; x < n; x += 64) Cr[x] = Z[lpad(x)];
        else
        {
            const TF ni = TF(1)/TF(n);   // exact for powers of two
            for (int x = lane; x < n; x += 64) { T z = Z[lpad(x)]; z.x *= ni; z.y *= ni; Cr[x] = z; }
        }
    }

    template<typename TF>
    struct fft_y_k
    {
        static constexpr int NT = 256, MINB = 0;
        cplx<TF>* C; Plan plan; const double2* tw; int sign; int nrows; int RB;
        __device__ __forceinline__ void operator()(const Bid& bid_) const
        {
            fft_y_g<TF>(C, plan, tw, sign, nrows, RB, bid_);
        }
    };

    // LDS ordering between the lanes of one wave: LDS operations of a wave
    // execute in issue order, so a wave exchanging data through its own LDS
    // rows needs no block barrier, only a point the compiler may not move
    // memory operations across.
    __device__ __forceinline__ void wave_lds_sync()
    {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    }

    // Number of radix-R passes of a row of n = 64 R (R = 2, 4, 8: n = 128,
    // 256, 512) and the padded row length in LDS.
    template<int R> constexpr int wave_passes() { return R == 8 ? 3 : R == 4 ? 4 : 7; }
    template<int R> constexpr int wave_row_elems() { return ((64*R - 1) + ((64*R - 1) >> 3) + 1) | 1; }

    // LDS rows of the wave x transforms.  The FFT passes use the lpad slots
    // 0 .. lpad(n-1); after the transform the staged half-spectra of the
    // wave's two real rows sit as Xa(kx) in slot kx and Xb(kx) in slot
    // XH + kx, the DC pair (a, b) in slot 0 and the Nyquist pair in slot XH.
    // XH = 32 R + 2 and a row stride of 4 mod 32 slots spread the transposed
    // copies between C and the rows (lanes over kx, the rows and the two
    // parts) over distinct LDS banks for 8- and 16-byte slots.
    template<int R> constexpr int xhalf() { return 32*R + 2; }
    template<int R> constexpr int xrow_base() { return wave_row_elems<R>() > 2*xhalf<R>() ? wave_row_elems<R>() : 2*xhalf<R>(); }
    template<int R> constexpr int xrow_elems() { return xrow_base<R>() + ((4 - xrow_base<R>() % 32) + 32) % 32; }

    template<typename TF, int R>
    __device__ __forceinline__ void xstage_store(cplx<TF>* S, int kx, cplx<TF> xa, cplx<TF> xb)
    {
        constexpr int n = 64*R, XH = xhalf<R>();
        if (kx == 0) { cplx<TF> d; d.x = xa.x; d.y = xb.x; S[0] = d; }
        else if (2*kx == n) { cplx<TF> d; d.x = xa.x; d.y = xb.x; S[XH] = d; }
        else { S[kx] = xa; S[XH + kx] = xb; }
    }

    // Per-lane twiddles of passes 1 .. P-1 of the wave FFT of length n = 64 R:
    // pass p (Ns = R^p) multiplies input q of butterfly `lane` by
    // tw[q (lane mod Ns) n/(Ns R)], conjugated for the inverse (S = +1).
    template<typename TF, int R, int S>
    __device__ __forceinline__ void wave_twiddles(cplx<TF> (&wt)[wave_passes<R>()-1][R-1],
                                                  const double2* __restrict__ tw, int lane)
    {
        constexpr int n = 64*R, P = wave_passes<R>();
        int Ns = R;
        #pragma unroll
        for (int p = 1; p < P; ++p)
        {
            const int k = lane & (Ns - 1), ts = n/(Ns*R);
            #pragma unroll
            for (int q = 1; q < R; ++q)
            {
                const double2 x = tw[q*k*ts];
                wt[p-1][q-1].x = TF(x.x); wt[p-1][q-1].y = TF(S < 0 ? x.y : -x.y);
            }
            Ns *= R;
        }
    }

    // Unnormalised FFT of one row of n = 64 R by one wave.  With a uniform
    // radix R every Stockham pass has exactly 64 butterflies, one per lane:
    // the first pass works on the row as the lanes hold it (v[q] = x[lane +
    // 64 q]), the last pass leaves the transform in the same order, and only
    // the passes between go through the wave's LDS row A (padded indices).
    template<typename TF, int R, int S>
    __device__ __forceinline__ void wave_fft(cplx<TF> (&v)[R], cplx<TF>* A,
                                             const cplx<TF> (&wt)[wave_passes<R>()-1][R-1], int lane)
    {
        constexpr int P = wave_passes<R>();
        // pass 0 (Ns = 1, no twiddles): butterfly lane, outputs lane*R + q
        dft<TF, R>(v, S);
        #pragma unroll
        for (int q = 0; q < R; ++q) A[lpad(lane*R + q)] = v[q];
        wave_lds_sync();
        int Ns = R;
        #pragma unroll
        for (int p = 1; p < P-1; ++p)
        {
            #pragma unroll
            for (int q = 0; q < R; ++q) v[q] = A[lpad(lane + 64*q)];
            #pragma unroll
            for (int q = 1; q < R; ++q) v[q] = cmul(v[q], wt[p-1][q-1]);
            dft<TF, R>(v, S);
            wave_lds_sync();
            const int d = (lane/Ns)*Ns*R + (lane & (Ns - 1));
            #pragma unroll
            for (int q = 0; q < R; ++q) A[lpad(d + q*Ns)] = v[q];
            wave_lds_sync();
            Ns *= R;
        }
        // last pass (Ns = 64): outputs lane + 64 q
        #pragma unroll
        for (int q = 0; q < R; ++q) v[q] = A[lpad(lane + 64*q)];
        wave_lds_sync();
        #pragma unroll
        for (int q = 1; q < R; ++q) v[q] = cmul(v[q], wt[P-2][q-1]);
        dft<TF, R>(v, S);
    }

    // wave_fft with the twiddles of each pass loaded at that pass (tw is a
    // few KB and cache-resident) instead of held in registers for the whole
    // transform: for kernels that transform one row per wave.
    template<typename TF, int R, int S>
    __device__ __forceinline__ void wave_fft_tw(cplx<TF> (&v)[R], cplx<TF>* A, const double2* __restrict__ tw, int lane)
    {
        constexpr int n = 64*R, P = wave_passes<R>();
        auto load_tw = [&](cplx<TF> (&w)[R-1], int Ns)
        {
            const int k = lane & (Ns - 1), ts = n/(Ns*R);
            #pragma unroll
            for (int q = 1; q < R; ++q)
            {
                const double2 x = tw[q*k*ts];
                w[q-1].x = TF(x.x); w[q-1].y = TF(S < 0 ? x.y : -x.y);
            }
        };
        dft<TF, R>(v, S);
        #pragma unroll
        for (int q = 0; q < R; ++q) A[lpad(lane*R + q)] = v[q];
        wave_lds_sync();
        int Ns = R;
        #pragma unroll
        for (int p = 1; p < P-1; ++p)
        {
            cplx<TF> w[R-1];
            load_tw(w, Ns);
            #pragma unroll
            for (int q = 0; q < R; ++q) v[q] = A[lpad(lane + 64*q)];
            #pragma unroll
            for (int q = 1; q < R; ++q) v[q] = cmul(v[q], w[q-1]);
            dft<TF, R>(v, S);
            wave_lds_sync();
            const int d = (lane/Ns)*Ns*R + (lane & (Ns - 1));
            #pragma unroll
            for (int q = 0; q < R; ++q) A[lpad(d + q*Ns)] = v[q];
            wave_lds_sync();
            Ns *= R;
        }
        cplx<TF> w[R-1];
        load_tw(w, Ns);
        #pragma unroll
        for (int q = 0; q < R; ++q) v[q] = A[lpad(lane + 64*q)];
        wave_lds_sync();
        #pragma unroll
        for (int q = 1; q < R; ++q) v[q] = cmul(v[q], w[q-1]);
        dft<TF, R>(v, S);
    }

    // y transform of contiguous rows of length n = 64 R, one wave per row
    // (no block barriers).  Waves walk the rows with a stride and load the next
    // row while transforming the current one.  S = -1 forward, +1 inverse
    // (which divides by n, as src/fft.cxx:420 does).
    template<typename TF, int R, int S>
    __device__ __forceinline__ void fft_y_wave_g(cplx<TF>* __restrict__ C, const double2* __restrict__ tw,
                                                 int nrows, const Bid& bid_)
    {
        using T = cplx<TF>;
        constexpr int n = 64*R, P = wave_passes<R>();
        __shared__ T rows[4][wave_row_elems<R>()];
        const int lane = threadIdx.x, wv = threadIdx.y;
        T* A = rows[wv];
        const int nw = bid_.nx*4;
        int r = bid_.x*4 + wv;
        if (r >= nrows) return;    // per wave; the kernel has no block barrier

        T wt[P-1][R-1];
        wave_twiddles<TF, R, S>(wt, tw, lane);
        T cur[R];
        #pragma unroll
        for (int q = 0; q < R; ++q) cur[q] = C[static_cast<size_t>(r)*n + lane + 64*q];
        for (; r < nrows; r += nw)
        {
            T nxt[R];
            const size_t rn = static_cast<size_t>(min(r + nw, nrows - 1));
            #pragma unroll
            for (int q = 0; q < R; ++q) nxt[q] = C[rn*n + lane + 64*q];
            // FP32 forward: the row minus its FP64 mean, bin 0 set to the FP64
            // sum afterwards (only bin 0 changes; the rest rounds against the
            // fluctuations, not the mean)
            constexpr bool demean = S < 0 && sizeof(TF) == 4;
            double sx = 0., sy = 0.;
            if (demean)
            {
                #pragma unroll
                for (int q = 0; q < R; ++q) { sx += double(cur[q].x); sy += double(cur[q].y); }
                #pragma unroll
                for (int o = 32; o > 0; o >>= 1) { sx += __shfl_xor(sx, o); sy += __shfl_xor(sy, o); }
                const TF mx = TF(sx/n), my = TF(sy/n);
                #pragma unroll
                for (int q = 0; q < R; ++q) { cur[q].x -= mx; cur[q].y -= my; }
            }
            wave_fft<TF, R, S>(cur, A, wt, lane);
            if (demean && lane == 0) { cur[0].x = TF(sx); cur[0].y = TF(sy); }
            T* __restrict__ Cr = C + static_cast<size_t>(r)*n;
            #pragma unroll
            for (int q = 0; q < R; ++q)
            {
                T z = cur[q];
                if (S > 0) { z.x *= TF(1)/TF(n); z.y *= TF(1)/TF(n); }
                Cr[lane + 64*q] = z;
            }
            #pragma unroll
            for (int q = 0; q < R; ++q) cur[q] = nxt[q];
        }
    }

    template<typename TF, int R, int S>
    struct fft_y_wave_k
    {
        static constexpr int NT = 256, MINB = 0;
        cplx<TF>* C; const double2* tw; int nrows;
        __device__ __forceinline__ void operator()(const Bid& bid_) const
        {
            fft_y_wave_g<TF, R, S>(C, tw, nrows, bid_);
        }
    };

    // Forward x transform of n = 64 R points: block (blockIdx.x, k) covers the
    // 8 real rows j0 .. j0+7 of level k (jtot a multiple of 8), one wave per
    // pair of rows packed as a + i b.  MODE 0: P as stored; 1: P minus the
    // plane mean pmean[k] (mixed mode); 2: the right-hand side of pres_in_g
    // evaluated from u, v, w and their tendencies; 3: as 2, and the block's
    // FP64 sum of the right-hand side into part[k*gridDim.x + blockIdx.x]
    // (mixed mode: the plane means, whose mode the FP64 path solves).
    // Writes C[k][kx][j].
    // Waves per block of the x wave kernels: each wave owns two rows, so a
    // block writes (reads) 2*XW consecutive j of every kx in C, a 128-byte
    // line in either precision.
    template<typename TF> constexpr int xwaves() { return sizeof(TF) == 8 ? 4 : 8; }

    template<typename TF, int R, int MODE>
    __device__ __forceinline__ void fft_x_fwd_wave_g(
            const TF* __restrict__ P, cplx<TF>* __restrict__ C, const double2* __restrict__ tw, Gd g,
            const double* __restrict__ pmean, double* __restrict__ part,
            const TF* __restrict__ u, const TF* __restrict__ v, const TF* __restrict__ w,
            const TF* __restrict__ ut, const TF* __restrict__ vt, const TF* __restrict__ wt,
            const TF* __restrict__ dzi, const TF* __restrict__ rho, const TF* __restrict__ rhoh,
            TF dxi, TF dyi, TF dti, int cpx, int packed, const Bid& bid_)
    {
        using T = cplx<TF>;
        constexpr int XW = xwaves<TF>(), NT = 64*XW;
        constexpr int n = 64*R, nx = n/2 + 1, JB = 2*XW, P_ = wave_passes<R>(), XH = xhalf<R>();
        constexpr int NQ = (nx + 63)/64;
        __shared__ T rows[XW][xrow_elems<R>()];
        __shared__ double wsum[XW];
        const int lane = threadIdx.x, wv = threadIdx.y, tid = lane + 64*wv;
        const int M = g.jtot, nbj = M/JB;
        // cpx > 0: a 1-D grid in which XCD x (blocks b = x mod 8) owns the
        // cpx row groups [x cpx, (x+1) cpx) and takes them level by level,
        // so the w and wt planes of level k+1 and the v, vt rows of the next
        // group are read again by a block that runs shortly after on the
        // same XCD (its own L2); else blockIdx = (group, level).
        int k, bj;
        if (cpx > 0)
        {
            const int li = bid_.x >> 3;
            k = li / cpx;
            bj = (bid_.x & 7)*cpx + li % cpx;
        }
        else { k = bid_.y; bj = bid_.x; }
        const int j0 = bj*JB, ja = j0 + 2*wv, jb = ja + 1;
        T* A = rows[wv];

        T z[R];
        if (MODE >= 2)
        {
            // pres_in_g's expression; the east and north tendency neighbours
            // wrap periodically, u, v, w have periodic halos already
            const int jj = g.icells, kk = g.ijcells, kc = k + g.kgc;
            const TF rk = rho[kc], rhk = rhoh[kc], rhkp = rhoh[kc+1], dzk = dzi[kc];
            #pragma unroll
            for (int h = 0; h < 2; ++h)
            {
                const int j = h ? jb : ja;
                const int row = g.igc + (j + g.jgc)*jj + kc*kk;
                const int dn = (j + 1 == g.jtot) ? jj - g.jtot*jj : jj;
                #pragma unroll
                for (int q = 0; q < R; ++q)
                {
                    const int x = lane + 64*q;
                    const int ijk = row + x;
                    const int de = (x + 1 == n) ? 1 - n : 1;
                    const TF val = rk * ( (ut[ijk+de] + u[ijk+1] * dti) - (ut[ijk] + u[ijk] * dti) ) * dxi
                                 + rk * ( (vt[ijk+dn] + v[ijk+jj] * dti) - (vt[ijk] + v[ijk] * dti) ) * dyi
                                 + ( rhkp * (wt[ijk+kk] + w[ijk+kk] * dti)
                                   - rhk  * (wt[ijk   ] + w[ijk   ] * dti) ) * dzk;
                    if (h) z[q].y = val; else z[q].x = val;
                }
            }
        }
        else
        {
            const TF* Pk = P + static_cast<size_t>(k)*n*M;
            const double m = MODE == 1 ? pmean[k] : 0.;
            #pragma unroll
            for (int q = 0; q < R; ++q)
            {
                const int x = lane + 64*q;
                if (MODE == 1) { z[q].x = TF(double(Pk[x + ja*n]) - m); z[q].y = TF(double(Pk[x + jb*n]) - m); }
                else           { z[q].x = Pk[x + ja*n]; z[q].y = Pk[x + jb*n]; }
            }
        }
        double sa = 0., sb = 0.;
        if (MODE == 3)
        {
            // FP64 sums of the wave's two rows in a fixed order (lane sums,
            // then a butterfly), so the result is reproducible.  The rows go
            // into the FP32 transform minus their means, which leaves every
            // bin but kx = 0 unchanged and rounds the others against the
            // fluctuations instead of the mean; bin 0 is set to the FP64 sum.
            #pragma unroll
            for (int q = 0; q < R; ++q) { sa += double(z[q].x); sb += double(z[q].y); }
            #pragma unroll
            for (int o = 32; o > 0; o >>= 1) { sa += __shfl_xor(sa, o); sb += __shfl_xor(sb, o); }
            if (lane == 0) wsum[wv] = sa + sb;
            const TF ma = TF(sa/n), mb = TF(sb/n);
            #pragma unroll
            for (int q = 0; q < R; ++q) { z[q].x -= ma; z[q].y -= mb; }
        }
        wave_fft_tw<TF, R, -1>(z, A, tw, lane);
        if (MODE == 3 && lane == 0) { z[0].x = TF(sa); z[0].y = TF(sb); }   // x = 0 is lane 0, q = 0

        // the two half-spectra: Z[kx] and Z[n-kx] come from other lanes
        #pragma unroll
        for (int q = 0; q < R; ++q) A[lpad(lane + 64*q)] = z[q];
        wave_lds_sync();
        T xs[NQ][2];
        #pragma unroll
        for (int q = 0; q < NQ; ++q)
        {
            const int kx = lane + 64*q;
            if (kx < nx) unpack_pair<TF>(A[lpad(kx)], A[lpad((n - kx) % n)], xs[q][0], xs[q][1]);
        }
        wave_lds_sync();
        #pragma unroll
        for (int q = 0; q < NQ; ++q)
        {
            const int kx = lane + 64*q;
            if (kx < nx) xstage_store<TF, R>(A, kx, xs[q][0], xs[q][1]);
        }
        __syncthreads();
        if (MODE == 3 && tid == 0)
        {
            double sm = 0.;
            #pragma unroll
            for (int q = 0; q < XW; ++q) sm += wsum[q];
            part[static_cast<size_t>(k)*nbj + bj] = sm;
        }
        // C[k][kx][j0 .. j0+JB): consecutive threads on consecutive j.  The
        // real bins kx = 0 and n/2 go to C[k][0][j] as one complex value when
        // packed (the layout of the paired y/tridiagonal kernels), else each
        // to its own row with a zero imaginary part.
        T* Ck = C + static_cast<size_t>(k)*nx*M;
        const int nkx = packed ? nx - 1 : nx;
        for (int idx = tid; idx < nkx*JB; idx += NT)
        {
            const int kx = idx / JB, jl = idx % JB;
            const int r = jl >> 1, part = jl & 1;
            const T* Sr = rows[r];
            T val;
            if (kx == 0 && packed)
            {
                const T d0 = Sr[0], dn = Sr[XH];
                val.x = part ? d0.y : d0.x; val.y = part ? dn.y : dn.x;
            }
            else if (kx == 0 || 2*kx == n)
            {
                const T d = Sr[kx == 0 ? 0 : XH];
                val.x = part ? d.y : d.x; val.y = TF(0);
            }
            else
                val = Sr[part*XH + kx];
            Ck[static_cast<size_t>(kx)*M + j0 + jl] = val;
        }
    }

    template<typename TF, int R, int MODE>
    struct fft_x_fwd_wave_k
    {
        static constexpr int NT = 64*xwaves<TF>(), MINB = 0;
        const TF* P; cplx<TF>* C; const double2* tw; Gd g; const double* pmean; double* part; const TF* u;
        const TF* v; const TF* w; const TF* ut; const TF* vt; const TF* wt; const TF* dzi; const TF* rho;
        const TF* rhoh; TF dxi; TF dyi; TF dti; int cpx; int packed;
        __device__ __forceinline__ void operator()(const Bid& bid_) const
        {
            fft_x_fwd_wave_g<TF, R, MODE>(P, C, tw, g, pmean, part, u, v, w, ut, vt, wt, dzi, rho, rhoh,
                dxi, dyi, dti, cpx, packed, bid_);
        }
    };

    // The same as a kernel of its own, for launches outside a batch: with the
    // pointers as __restrict__ kernel parameters the compiler issues the
    // right-hand side's loads of a row together (28 before the first use
    // instead of 3 through the functor's members), which FP32 needs to hide
    // their latency.
    template<typename TF, int R, int MODE>
    __global__ void __launch_bounds__(64*xwaves<TF>()) fft_x_fwd_wave_direct(
            const TF* __restrict__ P, cplx<TF>* __restrict__ C, const double2* __restrict__ tw, Gd g,
            const double* __restrict__ pmean, double* __restrict__ part,
            const TF* __restrict__ u, const TF* __restrict__ v, const TF* __restrict__ w,
            const TF* __restrict__ ut, const TF* __restrict__ vt, const TF* __restrict__ wt,
            const TF* __restrict__ dzi, const TF* __restrict__ rho, const TF* __restrict__ rhoh,
            TF dxi, TF dyi, TF dti, int cpx, int packed)
    {
        fft_x_fwd_wave_g<TF, R, MODE>(P, C, tw, g, pmean, part, u, v, w, ut, vt, wt, dzi, rho, rhoh,
            dxi, dyi, dti, cpx, packed,
            Bid{static_cast<int>(blockIdx.x), static_cast<int>(blockIdx.y), static_cast<int>(blockIdx.z),
                static_cast<int>(gridDim.x), static_cast<int>(gridDim.y), static_cast<int>(gridDim.z)});
    }

    // Inverse x transform of n = 64 R points (divides by n, src/fft.cxx:446)
    // into the ghosted p: interior rows, their periodic images in the y halo,
    // the x halo columns and, at the lowest level, the ghost level below.
    template<typename TF, int R>
    __device__ __forceinline__ void fft_x_bwd_wave_g(const cplx<TF>* __restrict__ C,
                                                     TF* __restrict__ p,
                                                     const double2* __restrict__ tw, Gd g,
                                                     int packed, const Bid& bid_)
    {
        using T = cplx<TF>;
        constexpr int XW = xwaves<TF>(), NT = 64*XW;
        constexpr int n = 64*R, nx = n/2 + 1, JB = 2*XW, P_ = wave_passes<R>(), XH = xhalf<R>();
        __shared__ T rows[XW][xrow_elems<R>()];
        const int lane = threadIdx.x, wv = threadIdx.y, tid = lane + 64*wv;
        const int M = g.jtot, k = bid_.y;
        const int j0 = bid_.x*JB;
        T* A = rows[wv];
        T wtw[P_-1][R-1];
        wave_twiddles<TF, R, +1>(wtw, tw, lane);

        // stage the block's spectra packed as in the forward kernel (packed:
        // bins 0 and n/2 both in C[k][0][j])
        const T* Ck = C + static_cast<size_t>(k)*nx*M;
        const int nkx = packed ? nx - 1 : nx;
        // every load of the thread in flight before the first LDS store
        constexpr int NLD = (nx*JB + NT - 1)/NT;
        T vals[NLD];
        #pragma unroll
        for (int u = 0; u < NLD; ++u)
        {
            const int idx = tid + u*NT;
            if (idx < nkx*JB)
                vals[u] = Ck[static_cast<size_t>(idx / JB)*M + j0 + idx % JB];
        }
        #pragma unroll
        for (int u = 0; u < NLD; ++u)
        {
            const int idx = tid + u*NT;
            if (idx >= nkx*JB) break;
            const int kx = idx / JB, jl = idx % JB;
            const int r = jl >> 1, part = jl & 1;
            const T val = vals[u];
            T* Sr = rows[r];
            if (kx == 0 && packed)
            {
                reinterpret_cast<TF*>(&Sr[0])[part] = val.x;
                reinterpret_cast<TF*>(&Sr[XH])[part] = val.y;
            }
            else if (kx == 0 || 2*kx == n)
            {
                TF* d = reinterpret_cast<TF*>(&Sr[kx == 0 ? 0 : XH]);
                d[part] = val.x;
            }
            else
                Sr[part*XH + kx] = val;
        }
        __syncthreads();
        // Hermitian extension of both spectra and packing Z = Xa + i Xb
        T z[R];
        #pragma unroll
        for (int q = 0; q < R; ++q)
        {
            const int x = lane + 64*q;
            const int kx = (x <= n/2) ? x : n - x;
            T xa, xb;
            if (kx == 0 || 2*kx == n)
            {
                const T d = A[kx == 0 ? 0 : XH];
                xa.x = d.x; xa.y = TF(0); xb.x = d.y; xb.y = TF(0);
            }
            else
            {
                xa = A[kx]; xb = A[XH + kx];
                if (x > n/2) { xa.y = -xa.y; xb.y = -xb.y; }
            }
            z[q].x = xa.x - xb.y; z[q].y = xa.y + xb.x;
        }
        wave_lds_sync();
        wave_fft<TF, R, +1>(z, A, wtw, lane);

        const TF ni = TF(1)/TF(n);   // exact for powers of two
        const int jj = g.icells, kk = g.ijcells, kc = k + g.kgc;
        const int ja = j0 + 2*wv;
        // x halo columns: ghosted x < igc and x >= iend wrap to n - igc + x and x - iend
        #pragma unroll
        for (int q = 0; q < R; ++q) A[lpad(lane + 64*q)] = z[q];
        wave_lds_sync();
        T zh; zh.x = TF(0); zh.y = TF(0);
        int xh = -1;
        if (lane < 2*g.igc)
        {
            xh = lane < g.igc ? lane : g.iend + (lane - g.igc);
            const int xi = lane < g.igc ? n - g.igc + lane : lane - g.igc;
            zh = A[lpad(xi)];
        }
        #pragma unroll
        for (int h = 0; h < 2; ++h)
        {
            const int j = ja + h;
            // the interior row and, within jgc of an edge, its periodic image
            int dst[2]; int nd = 0;
            dst[nd++] = j + g.jgc;
            if (j >= M - g.jgc) dst[nd++] = j - (M - g.jgc);
            else if (j < g.jgc) dst[nd++] = g.jend + j;
            for (int e = 0; e < nd; ++e)
            {
                TF* __restrict__ pr = p + static_cast<size_t>(kc)*kk + static_cast<size_t>(dst[e])*jj;
                #pragma unroll
                for (int q = 0; q < R; ++q)
                {
                    const TF val = (h ? z[q].y : z[q].x)*ni;
                    pr[g.igc + lane + 64*q] = val;
                    if (k == 0) pr[g.igc + lane + 64*q - kk] = val;
                }
                if (xh >= 0)
                {
                    const TF val = (h ? zh.y : zh.x)*ni;
                    pr[xh] = val;
                    if (k == 0) pr[xh - kk] = val;
                }
            }
        }
    }

    template<typename TF, int R>
    struct fft_x_bwd_wave_k
    {
        static constexpr int NT = 64*xwaves<TF>(), MINB = 0;
        const cplx<TF>* C; TF* p; const double2* tw; Gd g; int packed;
        __device__ __forceinline__ void operator()(const Bid& bid_) const
        {
            fft_x_bwd_wave_g<TF, R>(C, p, tw, g, packed, bid_);
        }
    };

    // Tridiagonal solve per (kx, ky) mode (Pres_2::solve + tdma,
    // src/pres_2.cxx:266-324, 200-263).  The matrix is real, so the two
    // components of a mode are two real systems: lane l of a wave owns
    // component l % 2 of mode l / 2, which are consecutive words of every level
    // of the spectrum.  The elimination (reciprocal pivots, gamma) depends on
    // the mode only through lambda and is precomputed per system
    // (Pres_tables::tri_*): no division in the sweeps.  TF is the element type
    // of the spectrum, TC the arithmetic type of the sweep (double in the mixed
    // mode).
    //
    // What bounds it: on large grids the bytes (768 x 384 x 256 FP64: 0.52 ms, 5.3
    // TB/s of the spectrum twice in and out and the two tables; 0.55 ms with the
    // blocks of 32 modes dealt to the XCDs in turn), on small ones the chain
    // over the levels, a multiply-add each if a level's values have arrived.
    // The loads of TRI_G levels are in flight while the TRI_G before them are
    // eliminated: 32^3 FP32 7.8 us, 90 x 75 x 60 FP64 14.8, 256 x 192 x 96 mixed
    // 25, 240 x 180 x 120 FP64 43 (15.5, 35.5, 58 and 112 with one level per trip
    // to memory).  That form, 64 modes per wave, was faster on two of 16 sizes, both 513 x 320
    // modes in FP64 (96 levels 188 us, 210 now; 320 levels 695 and 758).  LDSB: the eliminated
    // right-hand side stays in the wave's LDS column (K x 64 words) for the
    // back substitution, so the spectrum is read and written once.  Only for
    // columns of at most TRI_LDS bytes, five waves
    // on a CU: with longer ones too few waves are in flight (1024 x 1024 x 192
    // mixed, 48 KB: 36.5 against 35.0 ms per step; 768 x 384 x 256 FP64, 128 KB:
    // 24.3 against 22.0), with shorter ones the saved trip shows (256 x 192 x 96
    // mixed: 0.94 against 0.96 ms per step).
    constexpr int TRI_G = 16;
    constexpr int TRI_XCD = 512;
    constexpr size_t TRI_LDS = 32*1024;

    template<typename TF, typename TC, bool LDSB>
    __device__ __forceinline__ void tdma_g(TF* __restrict__ C,
                                           const TC* __restrict__ wi, const TC* __restrict__ gam,
                                           const TC* __restrict__ a, const TC* __restrict__ dz2,
                                           int nx, int nsys, Gd g, bool skip_mean, const Bid& bid_)
    {
        extern __shared__ unsigned char smem_raw[];
        TF* col = reinterpret_cast<TF*>(smem_raw) + threadIdx.x;    // LDSB: level k at col[64 k]
        const int M = g.jtot, K = g.ktot;
        const int nmodes = nx*M;
        // with two blocks per CU or more every XCD takes a contiguous range of modes: a
        // level of its share is then one run of memory, and the tables of modes ky
        // and M - ky meet in one L2.  Fewer are dealt to the XCDs in turn (24 x 24 x 300
        // FP32, 10 blocks: projection 83.0 us, 86.2 in ranges; 128 x 160 x 64 FP64, 325:
        // 79.0 and 80.3; but 240 x 180 x 120 FP64, 681: 287.7 and 282.1)
        const int tile = bid_.nx < TRI_XCD ? bid_.x : xcd_tile(bid_.x, bid_.nx);
        if (64*tile >= 2*nmodes) return;
        const int r0 = 64*tile + static_cast<int>(threadIdx.x);
        const bool active = r0 < 2*nmodes;
        const int r = active ? r0 : 2*nmodes - 1;
        const int mode = r >> 1;
        const int kx = mode / M, ky = mode - kx*M;
        const int l = kx*(M/2 + 1) + (ky <= M/2 ? ky : M - ky);
        // the mixed mode solves the horizontal mean in FP64 (mean_mode_g)
        const bool zero = skip_mean && mode == 0;
        const size_t ks = 2*static_cast<size_t>(nmodes), ls = static_cast<size_t>(nsys);
        TF* __restrict__ Cr = C + r;
        const TC* __restrict__ wr = wi + l;
        const TC* __restrict__ gr = gam + l;

        TF q[TRI_G], qn[TRI_G];
        TC w[TRI_G], wn[TRI_G];
        auto load = [&](TF (&qd)[TRI_G], TC (&wd)[TRI_G], int k0) {
            #pragma unroll
            for (int m = 0; m < TRI_G; ++m)
            {
                const size_t k = static_cast<size_t>(min(k0 + m, K-1));
                qd[m] = Cr[k*ks];
                wd[m] = wr[k*ls];
            }
        };
        // forward elimination (src/pres_2.cxx:200-252); the product with a is
        // rounded on its own
        load(q, w, 0);
        TC pr = TC(0);
        for (int k0 = 0; k0 < K; k0 += TRI_G)
        {
            load(qn, wn, k0 + TRI_G);
            #pragma unroll
            for (int m = 0; m < TRI_G; ++m)
            {
                const int k = k0 + m;
                if (k < K)
                {
                    const TC d = ld_const(dz2, k);
                    const TC x = (k > 0 ? fma(d, TC(q[m]), -mul_rn(ld_const(a, k), pr)) : d*TC(q[m]))*w[m];
                    if (LDSB) col[64*k] = TF(x);
                    else if (active) Cr[k*ks] = TF(x);
                    pr = x;
                }
            }
            #pragma unroll
            for (int m = 0; m < TRI_G; ++m) { q[m] = qn[m]; w[m] = wn[m]; }
        }
        // back substitution (src/pres_2.cxx:254-262) from the top; w[m] holds
        // gamma of the level above
        auto loadb = [&](TF (&qd)[TRI_G], TC (&wd)[TRI_G], int kt) {
            #pragma unroll
            for (int m = 0; m < TRI_G; ++m)
            {
                const int k = max(kt - m, 0);
                qd[m] = LDSB ? col[64*k] : Cr[k*ks];
                wd[m] = gr[static_cast<size_t>(min(k + 1, K-1))*ls];
            }
        };
        loadb(q, w, K-1);
        for (int k0 = K-1; k0 >= 0; k0 -= TRI_G)
        {
            // the levels of the next group are written only in their own group
            loadb(qn, wn, k0 - TRI_G);
            #pragma unroll
            for (int m = 0; m < TRI_G; ++m)
            {
                const int k = k0 - m;
                if (k >= 0)
                {
                    const TC x = k == K-1 ? pr : fma(-w[m], pr, TC(q[m]));
                    if (active) Cr[k*ks] = zero ? TF(0) : TF(x);
                    pr = x;
                }
            }
            #pragma unroll
            for (int m = 0; m < TRI_G; ++m) { q[m] = qn[m]; w[m] = wn[m]; }
        }
    }

    template<typename TF, typename TC, bool LDSB>
    struct tdma_k
    {
        static constexpr int NT = 64, MINB = 0;
        TF* C; const TC* wi; const TC* gam; const TC* a; const TC* dz2; int nx; int nsys; Gd g;
        bool skip_mean;
        __device__ __forceinline__ void operator()(const Bid& bid_) const
        {
            tdma_g<TF, TC, LDSB>(C, wi, gam, a, dz2, nx, nsys, g, skip_mean, bid_);
        }
    };

    // Paired modes.  The x spectrum at kx = 0 and at the last mode kxN =
    // itot/2 is real, and the wave x transforms can store the two packed as
    // Z = X0 + i XN in row kx = 0; block 0 of the fused y/tridiagonal kernels
    // then takes both (nx - 1 blocks instead of nx, which would leave one
    // block to run after all the others on a 256-CU device), transforming Z
    // as one complex row.  Both y spectra are Hermitian, as are the solutions
    // (the systems depend on ky only through bmatj[ky] = bmatj[jtot-ky]), so
    // their independent halves fill one row of jtot slots, the layout row
    // kx = 0 holds between the two kernels:
    //   slot 0, jtot/2    the real pair (mode (0, ky), mode (kxN, ky)) = Z[ky]
    //   0 < ky < jtot/2   mode (0, ky)         = (Z[ky] + conj Z[-ky])/2
    //   jtot/2 < ky       mode (kxN, jtot-ky)  = (Z[-ky] - conj Z[ky])/(2i)
    // Every thread solves one complex system; only the two real pairs have
    // different pivots for their two components.  Returns the elimination
    // table indices of the thread's x and y components.
    __device__ __forceinline__ void pair_systems(bool pair, int kx, int kxN, int ky, int n, int& lx, int& ly)
    {
        const int h = n/2 + 1;
        if (!pair) { lx = ly = kx*h + (ky <= n/2 ? ky : n - ky); return; }
        lx = ky <= n/2 ? ky : kxN*h + (n - ky);
        ly = (ky == 0 || 2*ky == n) ? kxN*h + ky : lx;
    }

    // y transform and tridiagonal sweep fused, for jtot = 64 R.  A block of R
    // waves owns one kx (block 0: the paired kx = 0 and kxN when paired) and
    // runs through the levels in groups of R: each wave transforms one level's
    // y row (the wave FFT) into its LDS row, then each thread, one per ky,
    // takes the group's R levels of its mode through the forward elimination
    // (precomputed per system, see tdma_g) and stores them.  The spectrum is
    // read and written once instead of twice.
    // Reciprocal pivots of the elimination of one system, level by level, as
    // setup_tables computes them (the same roundings: the products are not
    // fused into the subtractions, the division is IEEE), so they equal its
    // tri_wi entries: the forward sweep needs no table.
    template<typename TC>
    struct Pivots
    {
        TC lam, w;
        bool mean;
        __device__ __forceinline__ void first(const TC* __restrict__ av, const TC* __restrict__ acv,
                                              const TC* __restrict__ dz2rho, const TC* __restrict__ cv, int K)
        {
            TC b = mul_rn(dz2rho[0], lam) - acv[0];
            b += av[0];
            if (K == 1) { if (mean) b -= cv[0]; else b += cv[0]; }
            w = TC(1)/b;
        }
        __device__ __forceinline__ void next(const TC* __restrict__ av, const TC* __restrict__ acv,
                                             const TC* __restrict__ dz2rho, const TC* __restrict__ cv, int k, int K)
        {
            const TC gk = cv[k-1]*w;
            TC b = mul_rn(dz2rho[k], lam) - acv[k];
            if (k == K-1) { if (mean) b -= cv[K-1]; else b += cv[K-1]; }
            w = TC(1)/(b - mul_rn(av[k], gk));
        }
    };

    template<typename TF, typename TC, int R>
    __device__ __forceinline__ void ytri_fwd_g(cplx<TF>* __restrict__ C, const double2* __restrict__ tw,
                                               const TC* __restrict__ bmati, const TC* __restrict__ bmatj,
                                               const TC* __restrict__ a, const TC* __restrict__ cv,
                                               const TC* __restrict__ acv, const TC* __restrict__ dz2rho,
                                               const TC* __restrict__ dz2, int nx, Gd g,
                                               bool skip_mean, bool paired, const Bid& bid_)
    {
        using T = cplx<TF>;
        constexpr int n = 64*R, P_ = wave_passes<R>();
        __shared__ T rows[R][wave_row_elems<R>()];
        const int lane = threadIdx.x, wv = threadIdx.y, ky = lane + 64*wv;
        const int kx = bid_.x, K = g.ktot, kxN = nx - 1;
        const bool pair = paired && kx == 0;
        const size_t ks = static_cast<size_t>(nx)*n;
        int lx, ly;
        pair_systems(pair, kx, kxN, ky, n, lx, ly);
        // mixed mode: the mean is solved in FP64 (the x component of thread 0
        // is mode (0, 0) also when paired)
        const bool zero_mode = skip_mean && kx == 0 && ky == 0;
        // the thread's systems: lambda = bmati[kx] + bmatj[ky] of the mode
        // behind table index l = kx (n/2 + 1) + ky, the mean mode l = 0 with
        // its Dirichlet top row; only waves 0 and R/2 of a paired block hold
        // a second (real) system in the y component
        const bool two = pair && (wv == 0 || 2*wv == R);
        Pivots<TC> px_, py_;
        px_.lam = bmati[lx / (n/2 + 1)] + bmatj[lx % (n/2 + 1)]; px_.mean = lx == 0;
        py_.lam = bmati[ly / (n/2 + 1)] + bmatj[ly % (n/2 + 1)]; py_.mean = ly == 0;
        T* A = rows[wv];
        T* __restrict__ Ck = C + static_cast<size_t>(kx)*n;      // C[k][kx][.] = Ck[k*ks + .]
        T wtw[P_-1][R-1];
        wave_twiddles<TF, R, -1>(wtw, tw, lane);
        auto load_row = [&](T (&d)[R], size_t kr) {
            #pragma unroll
            for (int q = 0; q < R; ++q) d[q] = Ck[kr*ks + lane + 64*q];
        };

        T cur[R];
        load_row(cur, min(wv, K-1));
        TC px = TC(0), py = TC(0);
        for (int k0 = 0; k0 < K; k0 += R)
        {
            // the next group's row loads while this group is solved
            T nxt[R];
            const size_t kn = static_cast<size_t>(min(k0 + R + wv, K-1));
            load_row(nxt, kn);
            // the y transform of level k0 + wv (every wave transforms; rows
            // past the top are clamped copies, never used).  FP32: the row
            // minus its FP64 mean, bin 0 set to the FP64 sum afterwards, as in
            // fft_y_wave_g.
            constexpr bool demean = sizeof(TF) == 4;
            double sx = 0., sy = 0.;
            if (demean)
            {
                #pragma unroll
                for (int q = 0; q < R; ++q) { sx += double(cur[q].x); sy += double(cur[q].y); }
                #pragma unroll
                for (int o = 32; o > 0; o >>= 1) { sx += __shfl_xor(sx, o); sy += __shfl_xor(sy, o); }
                const TF mx = TF(sx/n), my = TF(sy/n);
                #pragma unroll
                for (int q = 0; q < R; ++q) { cur[q].x -= mx; cur[q].y -= my; }
            }
            wave_fft<TF, R, -1>(cur, A, wtw, lane);
            if (demean && lane == 0) { cur[0].x = TF(sx); cur[0].y = TF(sy); }
            #pragma unroll
            for (int q = 0; q < R; ++q) A[lpad(lane + 64*q)] = cur[q];
            __syncthreads();
            // forward elimination of mode (kx, ky) over the group (src/pres_2.cxx:200-252)
            #pragma unroll
            for (int m = 0; m < R; ++m)
            {
                const int k = k0 + m;
                if (k >= K) break;
                const T q = rows[m][lpad(ky)];
                TC zx = TC(q.x), zy = TC(q.y);
                if (pair && ky != 0 && 2*ky != n)
                {
                    // the thread's half-spectrum value from Z[ky] and Z[-ky]
                    const T r = rows[m][lpad(n - ky)];
                    if (2*ky < n) { zx = TC(0.5)*(zx + TC(r.x)); zy = TC(0.5)*(zy - TC(r.y)); }
                    else { const TC dx = TC(r.x) - zx, dy = TC(r.y) + zy; zx = TC(0.5)*dy; zy = TC(-0.5)*dx; }
                }
                if (k == 0) { px_.first(a, acv, dz2rho, cv, K); if (two) py_.first(a, acv, dz2rho, cv, K); }
                else { px_.next(a, acv, dz2rho, cv, k, K); if (two) py_.next(a, acv, dz2rho, cv, k, K); }
                const TC wx = px_.w, wy = two ? py_.w : px_.w;
                TC qx = dz2[k]*zx, qy = dz2[k]*zy;
                if (k > 0) { qx -= a[k]*px; qy -= a[k]*py; }
                qx *= wx; qy *= wy;
                if (zero_mode) { qx = TC(0); if (!pair) qy = TC(0); }
                Ck[k*ks + ky] = T{TF(qx), TF(qy)};
                px = qx; py = qy;
            }
            __syncthreads();
            #pragma unroll
            for (int q = 0; q < R; ++q) cur[q] = nxt[q];
        }
    }

    template<typename TF, typename TC, int R>
    struct ytri_fwd_k
    {
        static constexpr int NT = 64*R, MINB = 0;
        cplx<TF>* C; const double2* tw; const TC* bmati; const TC* bmatj; const TC* a; const TC* cv;
        const TC* acv; const TC* dz2rho; const TC* dz2; int nx; Gd g; bool skip_mean; bool paired;
        __device__ __forceinline__ void operator()(const Bid& bid_) const
        {
            ytri_fwd_g<TF, TC, R>(C, tw, bmati, bmatj, a, cv, acv, dz2rho, dz2, nx, g, skip_mean, paired,
                bid_);
        }
    };

    // Back substitution and inverse y transform fused (the counterpart of
    // ytri_fwd_g): from the top down in groups of R levels, each thread takes
    // its mode through the group's back substitution into the LDS rows, then
    // each wave inverse-transforms one level's row (dividing by jtot as
    // src/fft.cxx:420 does) and stores it.
    template<typename TF, typename TC, int R>
    __device__ __forceinline__ void ytri_bwd_g(cplx<TF>* __restrict__ C, const double2* __restrict__ tw,
                                               const TC* __restrict__ gam, int nx, int nsys, Gd g,
                                               bool paired, const Bid& bid_)
    {
        using T = cplx<TF>;
        constexpr int n = 64*R, P_ = wave_passes<R>();
        __shared__ T rows[R][wave_row_elems<R>()];
        const int lane = threadIdx.x, wv = threadIdx.y, ky = lane + 64*wv;
        const int kx = bid_.x, K = g.ktot, kxN = nx - 1;
        const bool pair = paired && kx == 0;
        const size_t ks = static_cast<size_t>(nx)*n, ls = static_cast<size_t>(nsys);
        int lx, ly;
        pair_systems(pair, kx, kxN, ky, n, lx, ly);
        T* A = rows[wv];
        T* __restrict__ Ck = C + static_cast<size_t>(kx)*n;
        T wtw[P_-1][R-1];
        wave_twiddles<TF, R, +1>(wtw, tw, lane);

        // the forward sweep's value at the top level is the solution there
        TC px = TC(0), py = TC(0);
        T qv[R]; TC gv[R], gvy[R];
        auto load_group = [&](T (&qd)[R], TC (&gd)[R], TC (&gdy)[R], int kt) {
            #pragma unroll
            for (int m = 0; m < R; ++m)
            {
                const int k = max(kt - m, 0);
                qd[m] = Ck[k*ks + ky];
                gd[m] = gam[min(k + 1, K-1)*ls + lx];
                gdy[m] = gam[min(k + 1, K-1)*ls + ly];
            }
        };
        load_group(qv, gv, gvy, K-1);
        for (int k0 = K-1; k0 >= 0; k0 -= R)
        {
            // the next group's values load while this one is solved: the
            // levels below k0 - R + 1 are not written before their group
            T qn[R]; TC gn[R], gny[R];
            load_group(qn, gn, gny, k0 - R);
            // back substitution (src/pres_2.cxx:254-262) of levels k0, k0-1, ...
            #pragma unroll
            for (int m = 0; m < R; ++m)
            {
                const int k = k0 - m;
                if (k < 0) break;
                TC qx = TC(qv[m].x), qy = TC(qv[m].y);
                if (k < K-1) { qx -= gv[m]*px; qy -= gvy[m]*py; }
                rows[m][lpad(ky)] = T{TF(qx), TF(qy)};
                px = qx; py = qy;
            }
            __syncthreads();
            const int k = k0 - wv;
            T v[R];
            if (pair)
            {
                // W = P0 + i PN over all ky from the row's half spectra S:
                // W[0], W[n/2] = S; 0 < ky < n/2: S[ky] + i S[-ky];
                // n/2 < ky: conj S[-ky] + i conj S[ky]
                #pragma unroll
                for (int q = 0; q < R; ++q)
                {
                    const int x = lane + 64*q;
                    const T sp = A[lpad(x)];
                    if (x == 0 || 2*x == n) v[q] = sp;
                    else
                    {
                        const T sm = A[lpad(n - x)];
                        v[q] = 2*x < n ? T{sp.x - sm.y, sp.y + sm.x} : T{sm.x + sp.y, sp.x - sm.y};
                    }
                }
            }
            else
            {
                #pragma unroll
                for (int q = 0; q < R; ++q) v[q] = A[lpad(lane + 64*q)];
            }
            wave_lds_sync();
            wave_fft<TF, R, +1>(v, A, wtw, lane);
            if (k >= 0)
            {
                #pragma unroll
                for (int q = 0; q < R; ++q)
                {
                    // paired: p0 + i pN, the two real x bins packed in row 0
                    T z = v[q];
                    z.x *= TF(1)/TF(n); z.y *= TF(1)/TF(n);
                    Ck[static_cast<size_t>(k)*ks + lane + 64*q] = z;
                }
            }
            __syncthreads();
            #pragma unroll
            for (int m = 0; m < R; ++m) { qv[m] = qn[m]; gv[m] = gn[m]; gvy[m] = gny[m]; }
        }
    }

    template<typename TF, typename TC, int R>
    struct ytri_bwd_k
    {
        static constexpr int NT = 64*R, MINB = 0;
        cplx<TF>* C; const double2* tw; const TC* gam; int nx; int nsys; Gd g; bool paired;
        __device__ __forceinline__ void operator()(const Bid& bid_) const
        {
            ytri_bwd_g<TF, TC, R>(C, tw, gam, nx, nsys, g, paired, bid_);
        }
    };

    // Inverse x transform and scatter into the ghosted p (Pres_2::solve tail,
    // src/pres_2.cxx:336-361): interior, the periodic halos of the rows the
    // block owns, and the bottom ghost level p[kstart-1] = p[kstart].
    template<typename TF>
    __device__ __forceinline__ void fft_x_bwd_g(const cplx<TF>* __restrict__ C, TF* __restrict__ p,
                                                const Plan& plan, const double2* __restrict__ tw, int RB, Gd g, const Bid& bid_)
    {
        using T = cplx<TF>;
        extern __shared__ unsigned char smem_raw[];
        const int n = plan.n, nx = n/2 + 1, M = g.jtot, re = row_elems(plan);
        T* rows = reinterpret_cast<T*>(smem_raw);
        const int row = threadIdx.y, lane = threadIdx.x;
        const int k = bid_.y;
        const int j0 = bid_.x*2*RB;
        const int nthr = 64*RB, tid = lane + 64*row;
        const int JB = 2*RB;
        const T* Ck = C + static_cast<size_t>(k)*nx*M;
        // Stage the block's spectra packed as in the forward kernel, in the
        // row's second buffer; the DC and Nyquist entries of a real row are real.
        const int soff = row_half(n);
        for (int idx = tid; idx < nx*JB; idx += nthr)
        {
            const int kx = idx / JB, jl = idx % JB;
            const int r = jl >> 1, part = jl & 1;
            const int j = j0 + jl;
            T val; val.x = TF(0); val.y = TF(0);
            if (j < M) val = Ck[static_cast<size_t>(kx)*M + j];
            T* Sr = rows + r*re + soff;
            if (kx == 0 || 2*kx == n)
            {
                TF* d = reinterpret_cast<TF*>(&Sr[kx == 0 ? 0 : 1]);
                d[part] = val.x;
            }
            else
                Sr[lpad(stage_base(kx, n) + part)] = val;
        }
        __syncthreads();
        T* A = rows + row*re;
        const T* B = A + soff;
        // Hermitian extension of both spectra and packing Z = Xa + i Xb.
        for (int x = lane; x < n; x += 64)
        {
            T xa, xb;
            const int kx = (x <= n/2) ? x : n - x;
            if (kx == 0 || 2*kx == n)
            {
                const T d = B[kx == 0 ? 0 : 1];
                xa.x = d.x; xa.y = TF(0); xb.x = d.y; xb.y = TF(0);
            }
            else
            {
                const int b = stage_base(kx, n);
                xa = B[lpad(b)]; xb = B[lpad(b+1)];
                if (x > n/2) { xa.y = -xa.y; xb.y = -xb.y; }
            }
            T z; z.x = xa.x - xb.y; z.y = xa.y + xb.x;
            A[lpad(x)] = z;
        }
        __syncthreads();
        T* Z = fft_row_pingpong<TF>(A, A + soff, plan, tw, +1, lane);
        const int ja = j0 + 2*row, jb = ja + 1;
        const int jj = g.icells, kk = g.ijcells;
        const TF ni = TF(1)/TF(n);   // the /itot of src/fft.cxx:446, exact for powers of two
        const int kc = k + g.kgc;
        for (int pr = 0; pr < 2; ++pr)
        {
            const int j = pr ? jb : ja;
            if (j >= M) continue;
            // destination rows: the interior row and, within jgc of an edge, its periodic image
            int rows_[3]; int nrow = 0;
            rows_[nrow++] = j + g.jgc;
            if (j >= M - g.jgc) rows_[nrow++] = j - (M - g.jgc);
            if (j < g.jgc) rows_[nrow++] = g.jend + j;
            for (int x = lane; x < g.icells; x += 64)
            {
                // ghosted column x maps to interior column x - igc, wrapped
                int xi = x - g.igc;
                xi = (xi < 0) ? xi + n : (xi >= n ? xi - n : xi);
                const T z = Z[lpad(xi)];
                const TF val = (pr ? z.y : z.x) * ni;
                for (int q = 0; q < nrow; ++q)
                {
                    const int ij = x + rows_[q]*jj;
                    p[ij + kc*kk] = val;
                    if (k == 0) p[ij + (kc-1)*kk] = val;
                }
            }
        }
    }

    template<typename TF>
    struct fft_x_bwd_k
    {
        static constexpr int NT = 256, MINB = 0;
        const cplx<TF>* C; TF* p; Plan plan; const double2* tw; int RB; Gd g;
        __device__ __forceinline__ void operator()(const Bid& bid_) const
        {
            fft_x_bwd_g<TF>(C, p, plan, tw, RB, g, bid_);
        }
    };

    // Mixed mode: partial plane sums of the RHS P in FP64, PM_CHUNKS per level
    // (a fixed summation order, so the result is reproducible).
    template<typename TF>
    __device__ __forceinline__ void plane_sum_g(const TF* __restrict__ P, double* __restrict__ part, int nplane, const Bid& bid_)
    {
        __shared__ double sm[256];
        const int k = bid_.y, chunk = bid_.x, tid = threadIdx.x;
        const int len = (nplane + PM_CHUNKS - 1)/PM_CHUNKS;
        const int b = chunk*len, e = min(b + len, nplane);
        const TF* Pk = P + static_cast<size_t>(k)*nplane;
        double s = 0.;
        for (int x = b + tid; x < e; x += 256) s += double(Pk[x]);
        sm[tid] = s;
        __syncthreads();
        for (int w = 128; w > 0; w >>= 1)
        {
            if (tid < w) sm[tid] += sm[tid + w];
            __syncthreads();
        }
        if (tid == 0) part[k*PM_CHUNKS + chunk] = sm[0];
    }

    template<typename TF>
    struct plane_sum_k
    {
        static constexpr int NT = 256, MINB = 0;
        const TF* P; double* part; int nplane;
        __device__ __forceinline__ void operator()(const Bid& bid_) const
        {
            plane_sum_g<TF>(P, part, nplane, bid_);
        }
    };

    // Mixed mode: the horizontal-mean mode of the projection in FP64.  The
    // plane means of P are its (0,0) Fourier coefficient divided by
    // itot*jtot, so the same tridiagonal system (lambda = 0, Neumann bottom,
    // p = 0 at the top face, src/pres_2.cxx:306-324) with the means as RHS gives
    // the mean pressure directly.  Its elimination depends on the grid only:
    // coef holds the reciprocal pivots (ktot) and gamma (ktot), so the sweep is
    // a chain of multiply-adds.  One workgroup: the partial sums (nparts per
    // level) are folded in parallel, thread 0 sweeps an LDS copy, the results
    // go out in parallel.  Dynamic LDS: ktot doubles.
    __device__ __forceinline__ void mean_mode_g(const double* __restrict__ part, int nparts,
                                                double* __restrict__ pmean,
                                                double* __restrict__ pbar, float* __restrict__ dpbar,
                                                const double* __restrict__ a, const double* __restrict__ dz2,
                                                const double* __restrict__ coef, double inv_nplane, Gd g, const Bid& bid_)
    {
        extern __shared__ double sp[];   // the sweep's right-hand side, then its solution
        const int K = g.ktot;
        const double* __restrict__ wi = coef;
        const double* __restrict__ gam = coef + K;
        for (int k = threadIdx.x; k < K; k += blockDim.x)
        {
            double s = 0.;
            for (int q = 0; q < nparts; ++q) s += part[static_cast<size_t>(k)*nparts + q];
            const double m = s*inv_nplane;
            pmean[k] = m;
            sp[k] = dz2[k]*m;
        }
        __syncthreads();
        if (threadIdx.x == 0)
        {
            double pk = sp[0]*wi[0];
            sp[0] = pk;
            for (int k = 1; k < K; ++k)
            {
                pk = (sp[k] - a[k]*pk)*wi[k];
                sp[k] = pk;
            }
            for (int k = K-2; k >= 0; --k)
            {
                pk = sp[k] - gam[k+1]*pk;
                sp[k] = pk;
            }
        }
        __syncthreads();
        for (int k = threadIdx.x; k < K; k += blockDim.x)
        {
            pbar[g.kstart + k] = sp[k];
            dpbar[g.kstart + k] = k == 0 ? 0.f : float(sp[k] - sp[k-1]);
        }
        if (threadIdx.x == 0) pbar[g.kstart-1] = sp[0];
    }

    struct mean_mode_k
    {
        static constexpr int NT = 256, MINB = 0;
        const double* part; int nparts; double* pmean; double* pbar; float* dpbar; const double* a;
        const double* dz2; const double* coef; double inv_nplane; Gd g;
        __device__ __forceinline__ void operator()(const Bid& bid_) const
        {
            mean_mode_g(part, nparts, pmean, pbar, dpbar, a, dz2, coef, inv_nplane, g, bid_);
        }
    };

    // Pres_2::output (src/pres_2.cxx:364-387).
    template<typename TF>
    __device__ __forceinline__ void pres_out_g(TF* __restrict__ ut, TF* __restrict__ vt, TF* __restrict__ wt,
                                               const TF* __restrict__ p, const TF* __restrict__ dzhi,
                                               TF dxi, TF dyi, Gd g, const TF* __restrict__ dpbar, const Bid& bid_)
    {
        const int i = bid_.x*BX + threadIdx.x + g.istart;
        const int j = bid_.y*BY + threadIdx.y + g.jstart;
        const int k = bid_.z + g.kstart;
        if (i >= g.iend || j >= g.jend) return;
        const int ijk = i + j*g.icells + k*g.ijcells;
        const TF pc = p[ijk];
        TF dpz = pc - p[ijk-g.ijcells];
        if (dpbar) dpz += dpbar[k];   // mixed mode: the FP64 mean's part
        ut[ijk] -= (pc - p[ijk-1]) * dxi;
        vt[ijk] -= (pc - p[ijk-g.icells]) * dyi;
        wt[ijk] -= dpz * dzhi[k];
    }

    template<typename TF>
    struct pres_out_k
    {
        static constexpr int NT = BX*BY, MINB = 0;
        TF* ut; TF* vt; TF* wt; const TF* p; const TF* dzhi; TF dxi; TF dyi; Gd g; const TF* dpbar;
        __device__ __forceinline__ void operator()(const Bid& bid_) const
        {
            pres_out_g<TF>(ut, vt, wt, p, dzhi, dxi, dyi, g, dpbar, bid_);
        }
    };

    // Pres_2::output (src/pres_2.cxx:364-387) followed by the RK3 update of
    // u, v, w (src/timeloop.cxx:251-286) and, with NS = 1, of scalar s (whose
    // update needs no pressure), one point per thread on the plane-ordered
    // grid: a pure streaming pass.  DEFER: the tendencies are left as they
    // came in (before the gradient and the cA scaling); the next fused
    // tendency pass, or settle_g, completes them.
    template<typename TF, int NS, bool DEFER>
    __device__ __forceinline__ void pres_out_rk3_g(
            TF* __restrict__ u, TF* __restrict__ v, TF* __restrict__ w,
            TF* __restrict__ ut, TF* __restrict__ vt, TF* __restrict__ wt,
            TF* __restrict__ s, TF* __restrict__ st,
            const TF* __restrict__ p, const TF* __restrict__ dzhi, const TF* __restrict__ dpbar,
            TF dxi, TF dyi, TF cBdt, TF cAn, int zero, Gd g, int nbx, int nby, const Bid& bid_)
    {
        // 1-D grid in XCD-contiguous order: the p rows and plane a tile reads
        // from its neighbours sit in the same L2
        const int tile = xcd_tile(bid_.x, bid_.nx);
        if (tile >= nbx*nby*g.ktot) return;
        const int i = (tile % nbx)*BX + threadIdx.x + g.istart;
        const int j = ((tile / nbx) % nby)*BY + threadIdx.y + g.jstart;
        const int k = tile/(nbx*nby) + g.kstart;
        if (i >= g.iend || j >= g.jend) return;
        const int ijk = i + j*g.icells + k*g.ijcells;
        const TF pc = p[ijk];
        TF dpz = pc - p[ijk-g.ijcells];
        if (dpbar) dpz += dpbar[k];   // mixed mode: the FP64 mean's part
        // one rounding per gradient term, written out as the deferred update
        // of the tendency pass writes it
        const TF tu = fma(p[ijk-1] - pc, dxi, ut[ijk]);
        const TF tv = fma(p[ijk-g.icells] - pc, dyi, vt[ijk]);
        const TF tw = fma(-dpz, dzhi[k], wt[ijk]);
        u[ijk] += cBdt*tu; v[ijk] += cBdt*tv; w[ijk] += cBdt*tw;
        if (!DEFER)
        {
            ut[ijk] = zero ? TF(0) : tu*cAn;
            vt[ijk] = zero ? TF(0) : tv*cAn;
            wt[ijk] = zero ? TF(0) : tw*cAn;
        }
        if (NS)
        {
            const TF ts = st[ijk];
            s[ijk] += cBdt*ts;
            if (!DEFER) st[ijk] = zero ? TF(0) : ts*cAn;
        }
    }

    template<typename TF, int NS, bool DEFER>
    struct pres_out_rk3_k
    {
        static constexpr int NT = BX*BY, MINB = 0;
        TF* u; TF* v; TF* w; TF* ut; TF* vt; TF* wt; TF* s; TF* st; const TF* p; const TF* dzhi;
        const TF* dpbar; TF dxi; TF dyi; TF cBdt; TF cAn; int zero; Gd g; int nbx; int nby;
        __device__ __forceinline__ void operator()(const Bid& bid_) const
        {
            pres_out_rk3_g<TF, NS, DEFER>(u, v, w, ut, vt, wt, s, st, p, dzhi, dpbar, dxi, dyi, cBdt, cAn,
                zero, g, nbx, nby, bid_);
        }
    };

    // Completes a deferred RK3 update of the tendencies: at = cA (at - grad p)
    // for u, v, w (the gradient of the p the update used, as in
    // pres_out_rk3_g) and at = cA at for scalar 0 (NS = 1); cA = 0 writes
    // zeros, as the reference's first substep does.
    template<typename TF, int NS>
    __device__ __forceinline__ void settle_g(
            TF* __restrict__ ut, TF* __restrict__ vt, TF* __restrict__ wt, TF* __restrict__ st,
            const TF* __restrict__ p, const TF* __restrict__ dzhi, const TF* __restrict__ dpbar,
            TF dxi, TF dyi, TF cA, int zero, Gd g, int nbx, int nby, const Bid& bid_)
    {
        const int tile = xcd_tile(bid_.x, bid_.nx);
        if (tile >= nbx*nby*g.ktot) return;
        const int i = (tile % nbx)*BX + threadIdx.x + g.istart;
        const int j = ((tile / nbx) % nby)*BY + threadIdx.y + g.jstart;
        const int k = tile/(nbx*nby) + g.kstart;
        if (i >= g.iend || j >= g.jend) return;
        const int ijk = i + j*g.icells + k*g.ijcells;
        if (zero)
        {
            ut[ijk] = TF(0); vt[ijk] = TF(0); wt[ijk] = TF(0);
            if (NS) st[ijk] = TF(0);
            return;
        }
        const TF pc = p[ijk];
        TF dpz = pc - p[ijk-g.ijcells];
        if (dpbar) dpz += dpbar[k];
        const TF tu = fma(p[ijk-1] - pc, dxi, ut[ijk]);
        const TF tv = fma(p[ijk-g.icells] - pc, dyi, vt[ijk]);
        const TF tw = fma(-dpz, dzhi[k], wt[ijk]);
        ut[ijk] = tu*cA; vt[ijk] = tv*cA; wt[ijk] = tw*cA;
        if (NS) st[ijk] *= cA;
    }

    template<typename TF, int NS>
    struct settle_k
    {
        static constexpr int NT = BX*BY, MINB = 0;
        TF* ut; TF* vt; TF* wt; TF* st; const TF* p; const TF* dzhi; const TF* dpbar; TF dxi; TF dyi; TF cA;
        int zero; Gd g; int nbx; int nby;
        __device__ __forceinline__ void operator()(const Bid& bid_) const
        {
            settle_g<TF, NS>(ut, vt, wt, st, p, dzhi, dpbar, dxi, dyi, cA, zero, g, nbx, nby, bid_);
        }
    };

    // Pres_2::calc_divergence (src/pres_2.cxx:389-422), per-block maxima.  TC
    // is the arithmetic type (double in the mixed mode: the FP64 residual of
    // the FP32 fields).
    template<typename TF, typename TC>
    __global__ void __launch_bounds__(BX*BY) divergence_g(const TF* __restrict__ u, const TF* __restrict__ v,
                                                          const TF* __restrict__ w, const TC* __restrict__ dzi,
                                                          const TC* __restrict__ rho, const TC* __restrict__ rhoh,
                                                          TC dxi, TC dyi, Gd g, double* __restrict__ red)
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
                const int jj = g.icells, kk = g.ijcells;
                const int ijk = i + j*jj + k*kk;
                const TC div = rho[k]*((TC(u[ijk+1])-TC(u[ijk]))*dxi + (TC(v[ijk+jj])-TC(v[ijk]))*dyi)
                             + (rhoh[k+1]*TC(w[ijk+kk])-rhoh[k]*TC(w[ijk]))*dzi[k];
                m = fmax(m, static_cast<double>(fabs(div)));
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

    // Rows per block so that the row buffers fit in 64 KiB.
    int rows_per_block(const Plan& p, size_t elem)
    {
        return std::max(1, std::min(4, static_cast<int>(65536/elem/static_cast<size_t>(row_elems(p)))));
    }

    size_t lds_bytes(const Plan& p, int RB, size_t elem)
    {
        return static_cast<size_t>(RB)*row_elems(p)*elem;
    }

    template<typename TF>
    int setup_tables(mhh_ctx* c, Pres_tables<TF>& t)
    {
        const Gd& g = c->gd;
        const int N = g.itot, M = g.jtot, K = g.ktot;
        // Pres_2::set_values (src/pres_2.cxx:124-153) in the element type.
        std::vector<TF> bi(N), bj(M), av(K), cv(K), acv(K), dz2v(K), dz2rhov(K);
        const TF dxidxi = TF(1.)/(TF(g.dx)*TF(g.dx));
        const TF dyidyi = TF(1.)/(TF(g.dy)*TF(g.dy));
        const TF pi = std::acos(TF(-1.));
        for (int j = 0; j < M/2+1; ++j) bj[j] = TF(2.) * (std::cos(TF(2.)*pi*TF(j)/TF(M)) - TF(1.)) * dyidyi;
        for (int j = M/2+1; j < M; ++j) bj[j] = bj[M-j];
        for (int i = 0; i < N/2+1; ++i) bi[i] = TF(2.) * (std::cos(TF(2.)*pi*TF(i)/TF(N)) - TF(1.)) * dxidxi;
        for (int i = N/2+1; i < N; ++i) bi[i] = bi[N-i];
        for (int k = 0; k < K; ++k)
        {
            av[k] = TF(c->h_dz[k+g.kgc]) * TF(c->h_rhorefh[k+g.kgc  ])*TF(c->h_dzhi[k+g.kgc  ]);
            cv[k] = TF(c->h_dz[k+g.kgc]) * TF(c->h_rhorefh[k+g.kgc+1])*TF(c->h_dzhi[k+g.kgc+1]);
            // the factors of b in the order of src/pres_2.cxx:311-312
            acv[k] = av[k] + cv[k];
            dz2v[k] = TF(c->h_dz[k+g.kgc])*TF(c->h_dz[k+g.kgc]);
            dz2rhov[k] = dz2v[k]*TF(c->h_rhoref[k+g.kgc]);
        }
        auto up = [](TF** d, const std::vector<TF>& h) -> int {
            MHH_CHECK(check_hip(hipMalloc(d, sizeof(TF)*h.size()), "hipMalloc(pres table)"));
            return check_hip(hipMemcpy(*d, h.data(), sizeof(TF)*h.size(), hipMemcpyHostToDevice), "hipMemcpy(pres table)");
        };
        MHH_CHECK(up(&t.bmati, bi));
        MHH_CHECK(up(&t.bmatj, bj));
        MHH_CHECK(up(&t.a, av));
        MHH_CHECK(up(&t.c, cv));
        MHH_CHECK(up(&t.ac, acv));
        MHH_CHECK(up(&t.dz2, dz2v));
        MHH_CHECK(up(&t.dz2rho, dz2rhov));
        // Elimination of every distinct system (src/pres_2.cxx:200-252, 306-324):
        // b = dz*dz*rho*lambda - (a + c), the bottom Neumann row, the top row
        // Dirichlet for the mean mode (l = 0) and Neumann otherwise.
        {
            const int NY = M/2 + 1;
            t.nsys = (N/2 + 1)*NY;
            const size_t ns = static_cast<size_t>(t.nsys);
            std::vector<TF> twi(ns*K), tgam(ns*K, TF(0));
            for (int kx = 0; kx <= N/2; ++kx)
                for (int ky = 0; ky < NY; ++ky)
                {
                    const size_t l = static_cast<size_t>(kx)*NY + ky;
                    const TF lam = bi[kx] + bj[ky];
                    const bool mean_mode = kx == 0 && ky == 0;
                    auto bcoef = [&](int k) -> TF {
                        TF b = dz2rhov[k]*lam - acv[k];
                        if (k == 0) b += av[0];
                        if (k == K-1) { if (mean_mode) b -= cv[K-1]; else b += cv[K-1]; }
                        return b;
                    };
                    TF w = TF(1)/bcoef(0);
                    twi[l] = w;
                    for (int k = 1; k < K; ++k)
                    {
                        const TF gk = cv[k-1]*w;
                        tgam[k*ns + l] = gk;
                        w = TF(1)/(bcoef(k) - av[k]*gk);
                        twi[k*ns + l] = w;
                    }
                }
            MHH_CHECK(up(&t.tri_wi, twi));
            MHH_CHECK(up(&t.tri_gam, tgam));
        }
        // Twiddles exp(-2 pi i t/n) in long double, rounded once.
        auto roots = [](double** d, int n) -> int {
            std::vector<double> h(2*static_cast<size_t>(n));
            const long double pil = 3.141592653589793238462643383279502884L;
            for (int t = 0; t < n; ++t)
            {
                const long double ang = 2.0L*pil*static_cast<long double>(t)/static_cast<long double>(n);
                h[2*t] = static_cast<double>(cosl(ang));
                h[2*t+1] = static_cast<double>(-sinl(ang));
            }
            MHH_CHECK(check_hip(hipMalloc(d, sizeof(double)*h.size()), "hipMalloc(twiddles)"));
            return check_hip(hipMemcpy(*d, h.data(), sizeof(double)*h.size(), hipMemcpyHostToDevice), "hipMemcpy(twiddles)");
        };
        MHH_CHECK(roots(&t.twx, N));
        MHH_CHECK(roots(&t.twy, M));
        return 0;
    }

    template<typename TF>
    void free_tables(Pres_tables<TF>& t)
    {
        if (t.bmati) (void)hipFree(t.bmati);
        if (t.bmatj) (void)hipFree(t.bmatj);
        if (t.a) (void)hipFree(t.a);
        if (t.c) (void)hipFree(t.c);
        if (t.ac) (void)hipFree(t.ac);
        if (t.dz2) (void)hipFree(t.dz2);
        if (t.dz2rho) (void)hipFree(t.dz2rho);
        if (t.twx) (void)hipFree(t.twx);
        if (t.twy) (void)hipFree(t.twy);
        if (t.tri_wi) (void)hipFree(t.tri_wi);
        if (t.tri_gam) (void)hipFree(t.tri_gam);
        t = Pres_tables<TF>();
    }

    // y transform of nrows contiguous rows: the wave-per-row kernel for n = 128,
    // 256 and 512, lane groups where there is a plan, the ping-pong engine
    // otherwise.
    template<typename TF, int R>
    void launch_fft_y_wave(mhh_ctx* c, cplx<TF>* C, const double* tw, int sign, int nrows)
    {
        // enough waves to fill the chip a few times over; each walks its rows
        const int nblocks = std::max(1, std::min((nrows + 3)/4, 4*256));
        const double2* t2 = reinterpret_cast<const double2*>(tw);
        if (sign < 0) launch(c, fft_y_wave_k<TF, R, -1>{C, t2, nrows}, nblocks, dim3(64, 4));
        else          launch(c, fft_y_wave_k<TF, R, +1>{C, t2, nrows}, nblocks, dim3(64, 4));
    }

    template<typename TF>
    int fft_y(mhh_ctx* c, cplx<TF>* C, const Plan& py, const double* tw, int sign, int nrows, const char* name)
    {
        if ((c->fft_generic || (py.n != 128 && py.n != 256 && py.n != 512)) && c->row_py.n)
            return row_y<TF, cplx<TF>>(c, C, tw, sign, nrows, name);
        {
            mhh::Timer _t(c, name);
            if (!c->fft_generic && py.n == 512)      launch_fft_y_wave<TF, 8>(c, C, tw, sign, nrows);
            else if (!c->fft_generic && py.n == 256) launch_fft_y_wave<TF, 4>(c, C, tw, sign, nrows);
            else if (!c->fft_generic && py.n == 128) launch_fft_y_wave<TF, 2>(c, C, tw, sign, nrows);
            else
            {
                const int RBy = rows_per_block(py, sizeof(cplx<TF>));
                const size_t ldsy = lds_bytes(py, RBy, sizeof(cplx<TF>));
                const auto* t2 = reinterpret_cast<const double2*>(tw);
                const dim3 grd((nrows + RBy - 1)/RBy), blk(64, RBy);
                launch(c, fft_y_k<TF>{C, py, t2, sign, nrows, RBy}, grd, blk, ldsy);
            }
        }
        return check_launch(name);
    }

    // Tridiagonal sweep of every mode, one wave per 32 modes.
    template<typename TF, typename TC>
    int tdma(mhh_ctx* c, cplx<TF>* C, const Pres_tables<TC>& t, int nx, bool skip_mean)
    {
        const Gd& g = c->gd;
        const int tiles = (2*nx*g.jtot + 63)/64, nb = tiles < TRI_XCD ? tiles : xcd_blocks(tiles);
        const size_t lds = sizeof(TF)*64*static_cast<size_t>(g.ktot);
        {
            mhh::Timer _t(c, "tdma");
            TF* Cr = reinterpret_cast<TF*>(C);
            if (lds <= TRI_LDS)
                launch(c, tdma_k<TF, TC, true>{Cr, t.tri_wi, t.tri_gam, t.a, t.dz2, nx, t.nsys, g, skip_mean}, nb, 64, lds);
            else
                launch(c, tdma_k<TF, TC, false>{Cr, t.tri_wi, t.tri_gam, t.a, t.dz2, nx, t.nsys, g, skip_mean}, nb, 64);
        }
        return check_launch("tdma");
    }

    // Fused y transforms and tridiagonal sweep (jtot = 64 R, R = 2, 4, 8).
    template<typename TF, typename TC, int R>
    void launch_ytri(mhh_ctx* c, cplx<TF>* C, const double2* twy, const Pres_tables<TC>& d, int nx, bool skip_mean,
                     bool paired)
    {
        const dim3 blk(64, R);
        // paired (the x transform stored bins 0 and itot/2 packed in row 0):
        // block 0 takes both
        const int nb = paired ? nx - 1 : nx;
        { mhh::Timer _t(c, "ytri_fwd"); launch(c, ytri_fwd_k<TF, TC, R>{C, twy, d.bmati, d.bmatj,
                d.a, d.c, d.ac, d.dz2rho, d.dz2, nx, c->gd, skip_mean, paired}, nb, blk); }
        { mhh::Timer _t(c, "ytri_bwd"); launch(c, ytri_bwd_k<TF, TC, R>{C, twy, d.tri_gam,
                nx, d.nsys, c->gd, paired}, nb, blk); }
    }

    template<typename TF, typename TC>
    int ytri(mhh_ctx* c, cplx<TF>* C, const double2* twy, const Pres_tables<TC>& d, int nx, bool skip_mean,
             bool paired)
    {
        switch (c->gd.jtot)
        {
            case 512: launch_ytri<TF, TC, 8>(c, C, twy, d, nx, skip_mean, paired); break;
            case 256: launch_ytri<TF, TC, 4>(c, C, twy, d, nx, skip_mean, paired); break;
            default:  launch_ytri<TF, TC, 2>(c, C, twy, d, nx, skip_mean, paired); break;
        }
        return check_launch("ytri");
    }

    // Forward and inverse x transforms through the wave kernels (itot = 64 R,
    // R = 2, 4, 8; jtot a multiple of 8).
    template<typename TF, int R>
    void launch_fft_x_fwd_wave(mhh_ctx* c, const TF* P, cplx<TF>* C, const double2* tw, int mode,
                               const Prof<TF>& p, TF dxi, TF dyi, TF dti, int packed)
    {
        const Gd& g = c->gd;
        const int nbj = g.jtot/(2*xwaves<TF>());
        const int cpx = nbj % 8 == 0 ? nbj/8 : 0;
        const dim3 grd = cpx ? dim3(nbj*g.ktot) : dim3(nbj, g.ktot), blk(64, xwaves<TF>());
        const TF* u = static_cast<const TF*>(c->f.u); const TF* v = static_cast<const TF*>(c->f.v);
        const TF* w = static_cast<const TF*>(c->f.w); const TF* ut = static_cast<const TF*>(c->f.ut);
        const TF* vt = static_cast<const TF*>(c->f.vt); const TF* wt = static_cast<const TF*>(c->f.wt);
#define MHH_XF(MODE) do { if (c->rec) record(c, fft_x_fwd_wave_k<TF, R, MODE>{P, C, tw, g, c->pm_mean, c->pm_part, \
                u, v, w, ut, vt, wt, p.dzi, p.rhoref, p.rhorefh, dxi, dyi, dti, cpx, packed}, grd, blk); \
            else fft_x_fwd_wave_direct<TF, R, MODE><<<grd, blk, 0, c->stream>>>(P, C, tw, g, c->pm_mean, c->pm_part, \
                u, v, w, ut, vt, wt, p.dzi, p.rhoref, p.rhorefh, dxi, dyi, dti, cpx, packed); } while (0)
        if (mode == 3) MHH_XF(3);
        else if (mode == 2) MHH_XF(2);
        else if (mode == 1) MHH_XF(1);
        else MHH_XF(0);
#undef MHH_XF
    }

    template<typename TF>
    int fft_x_fwd_wave(mhh_ctx* c, const TF* P, cplx<TF>* C, const double* tw, int mode,
                       const Prof<TF>& p, TF dxi, TF dyi, TF dti, const char* name, int packed)
    {
        const double2* t2 = reinterpret_cast<const double2*>(tw);
        {
            mhh::Timer _t(c, name);
            switch (c->gd.itot)
            {
                case 512: launch_fft_x_fwd_wave<TF, 8>(c, P, C, t2, mode, p, dxi, dyi, dti, packed); break;
                case 256: launch_fft_x_fwd_wave<TF, 4>(c, P, C, t2, mode, p, dxi, dyi, dti, packed); break;
                default:  launch_fft_x_fwd_wave<TF, 2>(c, P, C, t2, mode, p, dxi, dyi, dti, packed); break;
            }
        }
        return check_launch(name);
    }

    template<typename TF>
    int fft_x_bwd_wave(mhh_ctx* c, const cplx<TF>* C, TF* P, const double* tw, int packed)
    {
        const Gd& g = c->gd;
        const double2* t2 = reinterpret_cast<const double2*>(tw);
        const dim3 grd(g.jtot/(2*xwaves<TF>()), g.ktot), blk(64, xwaves<TF>());
        {
            mhh::Timer _t(c, "fft_x_bwd");
            switch (g.itot)
            {
                case 512: launch(c, fft_x_bwd_wave_k<TF, 8>{C, P, t2, g, packed}, grd, blk); break;
                case 256: launch(c, fft_x_bwd_wave_k<TF, 4>{C, P, t2, g, packed}, grd, blk); break;
                default:  launch(c, fft_x_bwd_wave_k<TF, 2>{C, P, t2, g, packed}, grd, blk); break;
            }
        }
        return check_launch("fft_x_bwd");
    }

    // rk3 >= 0: apply the gradient together with the RK3 update of substep
    // rk3 (time step rkdt) instead of Pres_2::output alone.
    // Forward x transform of a length without a lane-group plan (the right-hand
    // side evaluated in the kernel when fuse_in, else read from P).
    template<typename TF>
    int fft_x_fwd_general(mhh_ctx* c, const TF* P, cplx<TF>* C, const Plan& px, const Pres_tables<TF>& t,
                          const Pin_args<TF>& pin, int fuse_in)
    {
        const Gd& g = c->gd;
        const int M = g.jtot, K = g.ktot;
        const int RB = rows_per_block(px, sizeof(cplx<TF>));
        const dim3 grd((M + 2*RB - 1)/(2*RB), K);
        const size_t lds = lds_bytes(px, RB, sizeof(cplx<TF>));
        { mhh::Timer _t(c, fuse_in ? "pres_in_fft_x" : "fft_x_fwd");
          const auto* t2 = reinterpret_cast<const double2*>(t.twx);
          const double* pm = c->mixed ? c->pm_mean : nullptr;
          const dim3 blk(64, RB);
          launch(c, fft_x_fwd_k<TF>{P, C, px, t2, RB, g, pm, pin, fuse_in}, grd, blk, lds); }
        return check_launch("fft_x_fwd");
    }

    template<typename TF>
    int exec(mhh_ctx* c, const Prof<TF>& p, const Pres_tables<TF>& t, double dt, int rk3 = -1, double rkdt = 0.,
             bool with_scalars = false, bool defer = false)
    {
        using T = cplx<TF>;
        // a deferred update needs the p it used: complete it before the solve
        MHH_CHECK(settle_tendencies(c));
        if (defer && (!with_scalars || c->f.nscalars < 1))
            return fail(MHH_EINVAL, "pres_2: a deferred tendency update needs scalar 0 in the same call");
        const Gd& g = c->gd;
        if (!c->f.p || !c->f.tmp1 || !c->f.tmp2)
            return fail(MHH_ESTATE, "pres_2 needs p, tmp1 and tmp2 bound");
        const int N = g.itot, M = g.jtot, K = g.ktot, nx = N/2 + 1;
        Plan px, py;
        if (!make_plan(N, px) || !make_plan(M, py))
            return fail(MHH_EINVAL, "pres_2: itot and jtot must factor into primes <= 13");

        TF* P = static_cast<TF*>(c->f.p);
        T* C = static_cast<T*>(c->f.tmp1);
        const TF dxi = TF(1.)/TF(g.dx), dyi = TF(1.)/TF(g.dy), dti = TF(1.)/TF(dt);

        // 1. divergence into the dense array P (stored in p); without the mixed
        // mode's plane means the forward x transform evaluates it itself
        Pin_args<TF> pin{static_cast<const TF*>(c->f.u), static_cast<const TF*>(c->f.v), static_cast<const TF*>(c->f.w),
                         static_cast<const TF*>(c->f.ut), static_cast<const TF*>(c->f.vt), static_cast<const TF*>(c->f.wt),
                         p.dzi, p.rhoref, p.rhorefh, dxi, dyi, dti};
        const bool xwave = !c->fft_generic && (N == 128 || N == 256 || N == 512) && M % (2*xwaves<TF>()) == 0
                        && g.igc <= 32;
        const bool xdft = !xwave && dft_applies(c, N);
        const bool xrow = !xwave && !xdft && c->row_px.n;
        // The wave x transforms evaluate the right-hand side themselves (and, in
        // the mixed mode, the FP64 plane sums); the others do so except in the
        // mixed mode, whose plane means come first.
        const int fuse_in = (xwave || !c->mixed) ? 1 : 0;
        const Pres_tables<double>& d = c->td;
        const size_t mm_lds = sizeof(double)*K;
        if (!fuse_in)
        {
            const dim3 grd((N + BX - 1)/BX, (M + BY - 1)/BY, (K + PIN_KCHUNK - 1)/PIN_KCHUNK);
            { mhh::Timer _t(c, "pres_in"); launch(c, pres_in_k<TF>{P,
                    static_cast<const TF*>(c->f.u), static_cast<const TF*>(c->f.v), static_cast<const TF*>(c->f.w),
                    static_cast<const TF*>(c->f.ut), static_cast<const TF*>(c->f.vt), static_cast<const TF*>(c->f.wt),
                    p.dzi, p.rhoref, p.rhorefh, dxi, dyi, dti, g}, grd, dim3(BX, BY)); }
            MHH_CHECK(check_launch("pres_in"));
            { mhh::Timer _t(c, "pres_mean"); launch(c, plane_sum_k<TF>{P, c->pm_part, N*M}, dim3(PM_CHUNKS, K), 256); }
            MHH_CHECK(check_launch("plane_sum"));
            { mhh::Timer _t(c, "pres_mean"); launch(c, mean_mode_k{c->pm_part, PM_CHUNKS, c->pm_mean,
                    c->pbar, c->dpbar, d.a, d.dz2, c->pm_coef, 1./(double(N)*double(M)), g}, 1, 256, mm_lds); }
            MHH_CHECK(check_launch("mean_mode"));
        }
        // y transforms and tridiagonal sweep fused for jtot = 128, 256, 512;
        // with the wave x transforms as well, the real x bins 0 and itot/2
        // travel packed in row kx = 0 and share a block there
        const bool ywave = !c->fft_generic && !c->ytri_split && (M == 128 || M == 256 || M == 512);
        const int packed = xwave && ywave ? 1 : 0;
        // 2. forward x transform
        if (xwave)
        {
            const int mode = c->mixed ? 3 : 2;
            MHH_CHECK(fft_x_fwd_wave<TF>(c, P, C, t.twx, mode, p, dxi, dyi, dti, "pres_in_fft_x", packed));
            if (c->mixed)
            {
                { mhh::Timer _t(c, "pres_mean"); launch(c, mean_mode_k{c->pm_part, M/(2*xwaves<TF>()), c->pm_mean,
                        c->pbar, c->dpbar, d.a, d.dz2, c->pm_coef, 1./(double(N)*double(M)), g}, 1, 256, mm_lds); }
                MHH_CHECK(check_launch("mean_mode"));
            }
        }
        else
        {
            if constexpr (std::is_same<TF, float>::value)
                if (xdft) MHH_CHECK(dft_x_fwd(c, P, C, c->pm_mean));
            if (xrow) MHH_CHECK((row_x_fwd<TF, T>(c, fuse_in ? nullptr : P, C, t.twx, p, dxi, dyi, dti)));
            else if (!xdft) MHH_CHECK(fft_x_fwd_general<TF>(c, P, C, px, t, pin, fuse_in));
        }
        const int nrows = nx*K;
        if (ywave)
        {
            // 3-5. y transform, tridiagonal sweep, inverse y transform: two
            // fused passes
            const double2* twy = reinterpret_cast<const double2*>(t.twy);
            if (c->mixed)
            {
                const Pres_tables<double>& d = c->td;
                MHH_CHECK((ytri<TF, double>(c, C, twy, d, nx, true, packed)));
            }
            else
                MHH_CHECK((ytri<TF, TF>(c, C, twy, t, nx, false, packed)));
        }
        else
        {
        const bool ydft = dft_applies(c, M);
        // 3. forward y transform
        if constexpr (std::is_same<TF, float>::value)
        {
            if (ydft) MHH_CHECK(dft_y(c, C, nrows, -1));
            else MHH_CHECK(fft_y<TF>(c, C, py, t.twy, -1, nrows, "fft_y_fwd"));
        }
        else
            MHH_CHECK(fft_y<TF>(c, C, py, t.twy, -1, nrows, "fft_y_fwd"));
        // 4. tridiagonal per mode
        if constexpr (std::is_same<TF, float>::value)
        {
            if (c->mixed) MHH_CHECK((tdma<TF, double>(c, C, c->td, nx, true)));
            else MHH_CHECK((tdma<TF, TF>(c, C, t, nx, false)));
        }
        else
            MHH_CHECK((tdma<TF, TF>(c, C, t, nx, false)));
        // 5. inverse y transform (divides by jtot)
        if constexpr (std::is_same<TF, float>::value)
        {
            if (ydft) MHH_CHECK(dft_y(c, C, nrows, +1));
            else MHH_CHECK(fft_y<TF>(c, C, py, t.twy, +1, nrows, "fft_y_bwd"));
        }
        else
            MHH_CHECK(fft_y<TF>(c, C, py, t.twy, +1, nrows, "fft_y_bwd"));
        }
        // 6. inverse x transform (divides by itot) into the ghosted p with halos
        if (xwave)
            MHH_CHECK(fft_x_bwd_wave<TF>(c, C, P, t.twx, packed));
        else
        {
            if constexpr (std::is_same<TF, float>::value)
                if (xdft) MHH_CHECK(dft_x_bwd(c, C, P));
            if (xrow)
                MHH_CHECK((row_x_bwd<TF, T>(c, C, P, t.twx)));
            else if (!xdft)
            {
                const int RB = rows_per_block(px, sizeof(T));
                const dim3 grd((M + 2*RB - 1)/(2*RB), K);
                const size_t lds = lds_bytes(px, RB, sizeof(T));
                const auto* t2 = reinterpret_cast<const double2*>(t.twx);
                mhh::Timer _t(c, "fft_x_bwd");
                const dim3 blk(64, RB);
                launch(c, fft_x_bwd_k<TF>{C, P, px, t2, RB, g}, grd, blk, lds);
                MHH_CHECK(check_launch("fft_x_bwd"));
            }
        }
        // 7. pressure gradient on the tendencies (with the FP64 mean's part in the
        // mixed mode, whose fields are float)
        const TF* dpb = c->mixed ? reinterpret_cast<const TF*>(c->dpbar) : nullptr;
        if (rk3 < 0)
        {
            { mhh::Timer _t(c, "pres_out"); launch(c, pres_out_k<TF>{
                    static_cast<TF*>(c->f.ut), static_cast<TF*>(c->f.vt), static_cast<TF*>(c->f.wt),
                    P, p.dzhi, dxi, dyi, g, dpb}, grid3(g, g.kstart, g.kend), dim3(BX, BY)); }
            return check_launch("pres_out");
        }
        // Williamson low-storage coefficients (src/timeloop.cxx:255-256).
        const TF cA[] = {TF(0.), TF(-5./9.), TF(-153./128.)};
        const TF cB[] = {TF(1./3.), TF(15./16.), TF(8./15.)};
        const int substepn = (rk3 + 1) % 3;
        const TF cBdt = cB[rk3]*TF(rkdt);
        // scalar 0 rides along with the momentum update; further scalars get
        // their own pass
        const int ns = with_scalars ? c->f.nscalars : 0;
        {
            TF* s0 = ns > 0 ? static_cast<TF*>(c->f.s[0]) : nullptr;
            TF* st0 = ns > 0 ? static_cast<TF*>(c->f.st[0]) : nullptr;
            mhh::Timer _t(c, "pres_out_rk3");
            const int nbx = (g.itot + BX - 1)/BX, nby = (g.jtot + BY - 1)/BY;
            const int nb = xcd_blocks(nbx*nby*g.ktot);
#define MHH_PO(NS, D) launch(c, pres_out_rk3_k<TF, NS, D>{ \
                static_cast<TF*>(c->f.u), static_cast<TF*>(c->f.v), static_cast<TF*>(c->f.w), \
                static_cast<TF*>(c->f.ut), static_cast<TF*>(c->f.vt), static_cast<TF*>(c->f.wt), s0, st0, \
                P, p.dzhi, dpb, dxi, dyi, cBdt, cA[substepn], substepn == 0, g, nbx, nby}, nb, dim3(BX, BY))
            if (defer) MHH_PO(1, true);
            else if (ns > 0) MHH_PO(1, false);
            else MHH_PO(0, false);
#undef MHH_PO
        }
        MHH_CHECK(check_launch("pres_out_rk3"));
        if (defer)
        {
            c->defer_pending = true;
            c->defer_cA = double(cA[substepn]);
        }
        for (int n = 1; n < ns; ++n)
            MHH_CHECK(rk3_field<TF>(c, static_cast<TF*>(c->f.s[n]), static_cast<TF*>(c->f.st[n]),
                                    cBdt, cA[substepn], substepn == 0));
        if (substepn == 0)
        {
            TF* tl[4] = {static_cast<TF*>(c->f.ut), static_cast<TF*>(c->f.vt), static_cast<TF*>(c->f.wt),
                         ns > 0 ? static_cast<TF*>(c->f.st[0]) : nullptr};
            MHH_CHECK(zero_tendency_ghosts<TF>(c, tl, ns > 0 ? 4 : 3));
        }
        return 0;
    }

    template<typename TF>
    int settle(mhh_ctx* c, const Prof<TF>& p)
    {
        const Gd& g = c->gd;
        const TF dxi = TF(1.)/TF(g.dx), dyi = TF(1.)/TF(g.dy);
        const TF* dpb = c->mixed ? reinterpret_cast<const TF*>(c->dpbar) : nullptr;
        const int nbx = (g.itot + BX - 1)/BX, nby = (g.jtot + BY - 1)/BY;
        const int nb = xcd_blocks(nbx*nby*g.ktot);
        const double cA = c->defer_cA;
        { mhh::Timer _t(c, "settle");
          launch(c, settle_k<TF, 1>{
                static_cast<TF*>(c->f.ut), static_cast<TF*>(c->f.vt), static_cast<TF*>(c->f.wt),
                static_cast<TF*>(c->f.st[0]), static_cast<const TF*>(c->f.p), p.dzhi, dpb, dxi, dyi,
                TF(cA), cA == 0., g, nbx, nby}, nb, dim3(BX, BY)); }
        return check_launch("settle");
    }

    // The per-block maxima of the divergence into red[1..nb] (nb = the blocks of grid_red).
    template<typename TF>
    int divergence_partials(mhh_ctx* c, const Prof<TF>& p, double* red)
    {
        const Gd& g = c->gd;
        const dim3 grd = grid_red(g);
        if (c->mixed)
        {
            const Prof<double>& d = c->pd;
            mhh::Timer _t(c, "divergence");
            divergence_g<TF, double><<<grd, dim3(BX, BY), 0, c->stream>>>(
                    static_cast<const TF*>(c->f.u), static_cast<const TF*>(c->f.v), static_cast<const TF*>(c->f.w),
                    d.dzi, d.rhoref, d.rhorefh, 1./g.dx, 1./g.dy, g, red);
        }
        else
        {
            mhh::Timer _t(c, "divergence");
            divergence_g<TF, TF><<<grd, dim3(BX, BY), 0, c->stream>>>(
                    static_cast<const TF*>(c->f.u), static_cast<const TF*>(c->f.v), static_cast<const TF*>(c->f.w),
                    p.dzi, p.rhoref, p.rhorefh, TF(1.)/TF(g.dx), TF(1.)/TF(g.dy), g, red);
        }
        return check_launch("divergence");
    }

    template<typename TF>
    int divergence(mhh_ctx* c, const Prof<TF>& p, double* out)
    {
        const dim3 grd = grid_red(c->gd);
        const int nb = static_cast<int>(grd.x*grd.y*grd.z);
        MHH_CHECK(ensure_reduction(c, nb));
        MHH_CHECK(divergence_partials<TF>(c, p, c->red));
        return reduce_max_partials(c, nb, out);
    }

    // The same maximum with the partials in this device's static scratch array
    // and the result left in device memory: no allocation, no host copy.
    template<typename TF>
    int divergence_noalloc(mhh_ctx* c, const Prof<TF>& p, double* out_dev)
    {
        const dim3 grd = grid_red(c->gd);
        const long long nb = static_cast<long long>(grd.x)*grd.y*grd.z;
        constexpr long long cap = MHH_NOALLOC_SCRATCH_BYTES/sizeof(double);
        if (nb + 1 > cap)
            return fail(MHH_EINVAL, "mhh_pres_2_divergence_noalloc: this grid needs " + std::to_string(nb) +
                                    " partial maxima (one per 64 x 4 columns x 32 levels); the static scratch "
                                    "holds " + std::to_string(cap - 1));
        double* scr = static_scratch(c->device);
        if (!scr)
            return fail(MHH_ESTATE, "mhh_pres_2_divergence_noalloc: no static scratch address for this device");
        MHH_CHECK(divergence_partials<TF>(c, p, scr));
        return fold_max_to_device(c, scr + 1, static_cast<int>(nb), out_dev);
    }
}

namespace mhh
{
    int pres_init(mhh_ctx* c)
    {
        Plan px, py;
        if (!make_plan(c->gd.itot, px) || !make_plan(c->gd.jtot, py))
            return fail(MHH_EINVAL, "itot and jtot must factor into primes <= 13 (FFT radices)");
        // FP64 tables for FP64 fields and for the FP64 tridiagonal of the mixed mode.
        if (c->precision == MHH_FP64 || c->mixed) MHH_CHECK(setup_tables<double>(c, c->td));
        if (c->precision == MHH_FP32) MHH_CHECK(setup_tables<float>(c, c->tf));
        MHH_CHECK(dft_init(c));
        row_plans_init(c);
        if (c->mixed)
        {
            const size_t K = c->gd.ktot, nk = c->gd.kcells;
            // partial plane sums: PM_CHUNKS per level (plane_sum_g) or one per
            // block of 8 rows (the wave x transform)
            const size_t nparts = std::max<size_t>(PM_CHUNKS, (c->gd.jtot + 7)/8);
            MHH_CHECK(check_hip(hipMalloc(&c->pm_part, sizeof(double)*K*nparts), "hipMalloc(pm_part)"));
            MHH_CHECK(check_hip(hipMalloc(&c->pm_mean, sizeof(double)*K), "hipMalloc(pm_mean)"));
            MHH_CHECK(check_hip(hipMalloc(&c->pbar, sizeof(double)*nk), "hipMalloc(pbar)"));
            MHH_CHECK(check_hip(hipMalloc(&c->dpbar, sizeof(float)*nk), "hipMalloc(dpbar)"));
            MHH_CHECK(check_hip(hipMemset(c->pbar, 0, sizeof(double)*nk), "hipMemset(pbar)"));
            MHH_CHECK(check_hip(hipMemset(c->dpbar, 0, sizeof(float)*nk), "hipMemset(dpbar)"));
            // elimination of the mean mode (lambda = 0; Neumann bottom, Dirichlet
            // top, src/pres_2.cxx:306-324): reciprocal pivots and gamma, FP64
            const Gd& g = c->gd;
            const int Kc = g.ktot;
            std::vector<double> av(Kc), cv(Kc), coef(2*static_cast<size_t>(Kc), 0.);
            for (int k = 0; k < Kc; ++k)
            {
                av[k] = c->h_dz[k+g.kgc] * c->h_rhorefh[k+g.kgc  ]*c->h_dzhi[k+g.kgc  ];
                cv[k] = c->h_dz[k+g.kgc] * c->h_rhorefh[k+g.kgc+1]*c->h_dzhi[k+g.kgc+1];
            }
            auto bcoef = [&](int k) {
                double b = -(av[k] + cv[k]);
                if (k == 0) b += av[0];
                if (k == Kc-1) b -= cv[Kc-1];
                return b;
            };
            double w2 = bcoef(0);
            coef[0] = 1./w2;
            for (int k = 1; k < Kc; ++k)
            {
                const double gk = cv[k-1]/w2;
                coef[Kc + k] = gk;
                w2 = bcoef(k) - av[k]*gk;
                coef[k] = 1./w2;
            }
            MHH_CHECK(check_hip(hipMalloc(&c->pm_coef, sizeof(double)*coef.size()), "hipMalloc(pm_coef)"));
            MHH_CHECK(check_hip(hipMemcpy(c->pm_coef, coef.data(), sizeof(double)*coef.size(), hipMemcpyHostToDevice),
                                "hipMemcpy(pm_coef)"));
        }
        return 0;
    }

    int settle_tendencies(mhh_ctx* c)
    {
        if (!c->defer_pending) return 0;
        c->defer_pending = false;
        return c->precision == MHH_FP64 ? settle<double>(c, c->pd) : settle<float>(c, c->pf);
    }

    void pres_free(mhh_ctx* c)
    {
        dft_free(c);
        free_tables(c->td);
        free_tables(c->tf);
        for (void* b : {static_cast<void*>(c->pm_part), static_cast<void*>(c->pm_mean), static_cast<void*>(c->pm_coef),
                        static_cast<void*>(c->pbar), static_cast<void*>(c->dpbar)})
            if (b) (void)hipFree(b);
    }
}

extern "C" {

int mhh_pres_2_exec(mhh_ctx* c, double dt)
{
    MHH_REQUIRE_BOUND(c);
    if (!(dt > 0)) return mhh::fail(MHH_EINVAL, "pres_2: dt must be positive");
    return c->precision == MHH_FP64 ? exec<double>(c, c->pd, c->td, dt) : exec<float>(c, c->pf, c->tf, dt);
}

int mhh_pres_2_exec_rk3(mhh_ctx* c, double dt, int substep, double rkdt, int flags)
{
    MHH_REQUIRE_BOUND(c);
    if (!(dt > 0)) return mhh::fail(MHH_EINVAL, "pres_2: dt must be positive");
    if (substep < 0 || substep > 2) return mhh::fail(MHH_EINVAL, "rk3 substep must be 0, 1 or 2");
    if (flags & ~(MHH_RK3_SCALARS | MHH_RK3_DEFER)) return mhh::fail(MHH_EINVAL, "pres_2: unknown flags");
    const bool scalars = flags & MHH_RK3_SCALARS, defer = flags & MHH_RK3_DEFER;
    return c->precision == MHH_FP64 ? exec<double>(c, c->pd, c->td, dt, substep, rkdt, scalars, defer)
                                    : exec<float>(c, c->pf, c->tf, dt, substep, rkdt, scalars, defer);
}

int mhh_tendency_settle(mhh_ctx* c)
{
    MHH_REQUIRE_BOUND(c);
    return mhh::settle_tendencies(c);
}

int mhh_pres_2_mean_profile(mhh_ctx* c, double* out)
{
    MHH_NOT_IN_BATCH(c, "mhh_pres_2_mean_profile");
    if (!c || !out) return mhh::fail(MHH_EINVAL, "mhh_pres_2_mean_profile: null argument");
    const size_t nk = static_cast<size_t>(c->gd.kcells);
    if (!c->mixed)
    {
        std::fill(out, out + nk, 0.);
        return 0;
    }
    MHH_CHECK(mhh::check_hip(c->stream ? hipStreamSynchronize(c->stream) : hipDeviceSynchronize(), "sync"));
    return mhh::check_hip(hipMemcpy(out, c->pbar, sizeof(double)*nk, hipMemcpyDeviceToHost), "hipMemcpy(pbar)");
}

int mhh_pres_2_divergence(mhh_ctx* c, double* out)
{
    MHH_REQUIRE_BOUND(c);
    MHH_NOT_IN_BATCH(c, "mhh_pres_2_divergence");
    if (!out) return mhh::fail(MHH_EINVAL, "null output");
    return c->precision == MHH_FP64 ? divergence<double>(c, c->pd, out) : divergence<float>(c, c->pf, out);
}

int mhh_pres_2_divergence_noalloc(mhh_ctx* c, double* divmax_dev)
{
    MHH_REQUIRE_BOUND(c);
    MHH_NOT_IN_BATCH(c, "mhh_pres_2_divergence_noalloc");
    if (!divmax_dev) return mhh::fail(MHH_EINVAL, "null output");
    return c->precision == MHH_FP64 ? divergence_noalloc<double>(c, c->pd, divmax_dev)
                                    : divergence_noalloc<float>(c, c->pf, divmax_dev);
}

} // extern "C"
