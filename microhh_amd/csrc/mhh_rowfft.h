// mhh_rowfft.h -- FFTs of rows of any length with prime factors up to 13, by
// lane groups of a wavefront.
//
// A group of L lanes (L = 8, 16, 32 or 64; 64/L rows per wave) transforms one
// row in its LDS by the Stockham autosort algorithm: butterfly j of a pass of
// radix R takes the elements j + r n/R into the registers of lane j mod L and puts
// its outputs back into the same row.  A row belongs to one wave: no block barrier
// inside a transform.  The radices are make_plan's.  Two kinds of butterflies:
//   ROW_RADIX8  radices 8, 4, 2, 3 and 5
//   ROW_DIRECT  any radix up to 13 by its definition, the sums in the order of
//               fft_row_pingpong
// Order and roundings are those of the block-wide engines that the lane groups took
// over from: built with the compiler of ROCm 7.2, the projection of 42 grids
// returned the same bits as with those, in FP64, FP32 and the mixed mode.  turn() writes
// the roundings of the twiddle products out; those inside dft<> are left to
// contraction, so another compiler may move the last bits.  Composite radices up to 16
// would save a pass (960 x 500 x 58 FP64 projection 1.26 ms instead of 1.36), but
// rounding in another order shows: plain FP32 carries the horizontal mean through
// transforms and sweeps (4e-3 of a velocity after two steps), and the FP64 eddy
// viscosity, a square root clipped where the flow is stable, moves by 1e-9 there
// when the last bits of the velocities do.
#pragma once

#include <type_traits>

#include <hip/hip_runtime.h>

#include "mhh_fft.h"
#include "mhh_internal.h"
#include "mhh_stencil.h"

namespace mhh
{
    constexpr int ROW_VALS = 16, ROW_VALS_WIDE = 32;   // complex values a lane holds in a pass
    enum { ROW_RADIX8 = 0, ROW_DIRECT = 1 };
    enum { ROW_X_FWD, ROW_Y_FWD, ROW_Y_INV, ROW_X_INV };
    // Butterflies of radix r that a lane holds in a pass: as many as its values allow,
    // up to a limit.  4 for ROW_RADIX8: 256 on 64 lanes, the most that make_plan
    // calls fast.  8 for ROW_DIRECT bounds the unrolled code; it is not tuned
    // (1920 = 4 4 8 3 5 would need ten of radix 3, whose 30 values fit in the 32).
    __host__ __device__ constexpr int row_rounds(int r, int vals, int arith)
    {
        const int most = arith == ROW_DIRECT ? 8 : 4;
        return vals/r < most ? vals/r : most;
    }

    // The plan of a launch over `rows` rows: the lanes per row with the least work
    // per element, each pass's rounds of L butterflies times their cost (their
    // values and twiddles through LDS and the arithmetic), times the lanes, idle
    // ones included, in the instance with the fewest values per lane that holds
    // the row.  False if there is none (long rows, a single point).  Few rows
    // take more lanes each, so that the launch still has about ROW_WAVES waves (two
    // per SIMD): what a lane does in turn is latency then (90 x 75 x 60 FP64, 8
    // lanes per row instead of 64: forward x transform 19.2 instead of 13.8 us).
    constexpr int ROW_WAVES = 2048;
    inline bool make_row_plan(int n, long long rows, Row_plan& p)
    {
        p.n = 0;
        Plan f;
        if (n < 2 || n > 64*ROW_VALS_WIDE || !make_plan(n, f) || f.npass > ROW_MAXPASS) return false;
        int lmin = 3;
        while (lmin < 6 && (rows << lmin) < 64ll*ROW_WAVES) ++lmin;
        const int arith = f.fast ? ROW_RADIX8 : ROW_DIRECT;
        double best = 1.e300;
        for (int vals : {ROW_VALS, ROW_VALS_WIDE})
        {
            for (int lsh = lmin; lsh <= 6; ++lsh)
            {
                const int L = 1 << lsh;
                double cost = 6.*L*f.npass;     // a pass's trip through LDS
                bool fits = true;
                for (int q = 0; q < f.npass; ++q)
                {
                    const int R = f.radix[q], rounds = (n/R + L - 1)/L;
                    if (rounds > row_rounds(R, vals, arith)) { fits = false; break; }
                    cost += rounds*L*R*((q > 0 ? 3. : 2.) + (R > 5 && R != 8 ? 0.5*R : 1.));
                }
                if (!fits || cost >= best) continue;
                best = cost;
                p.n = n; p.npass = f.npass; p.lsh = lsh; p.vals = vals; p.arith = arith;
                int ns = 1;
                for (int q = 0; q < f.npass; ++q)
                {
                    const int R = f.radix[q];
                    p.radix[q] = R; p.nb[q] = n/R; p.ns[q] = ns; p.ts[q] = n/(ns*R);
                    p.mg[q] = static_cast<unsigned int>(((1ll << 22) + ns - 1)/ns);
                    ns *= R;
                }
            }
            if (p.n) return true;
        }
        return false;
    }

    // LDS slots of a row (element x at lpad(x)); an odd number, so that equal
    // elements of neighbouring rows sit in different banks.
    __host__ __device__ inline int row_stride(int n) { return (lpad(n - 1) + 1) | 1; }

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

    // Calls f with the pass's radix as a constant (uniform).
    template<int ARITH, typename F>
    __device__ __forceinline__ void with_radix(int R, F f)
    {
        constexpr bool D = ARITH == ROW_DIRECT;
#define MHH_RADIX(N) case N: f(std::integral_constant<int, N>{}); break
        switch (R)
        {
            MHH_RADIX(2);
            MHH_RADIX(3);
            MHH_RADIX(4);
            MHH_RADIX(5);
            case 7: if constexpr (D) f(std::integral_constant<int, 7>{}); break;
            case 11: if constexpr (D) f(std::integral_constant<int, 11>{}); break;
            case 13: if constexpr (D) f(std::integral_constant<int, 13>{}); break;
            default: f(std::integral_constant<int, 8>{}); break;
        }
#undef MHH_RADIX
    }

    // a*w with the roundings written out (left to contraction, the compiler may
    // round either product of a part first, and which one differs between
    // kernels): the imaginary part rounds a.x w.y first, or a.y w.x (LATE).
    template<bool LATE, typename T> __device__ __forceinline__ T turn(T a, T w)
    {
        T r;
        r.x = fma(a.x, w.x, -mul_rn(a.y, w.y));
        r.y = LATE ? fma(a.x, w.y, mul_rn(a.y, w.x)) : fma(a.y, w.x, mul_rn(a.x, w.y));
        return r;
    }

    // The transform DIR of one row, in place in the group's LDS, by its L lanes;
    // tw: the table of n roots in LDS.  Every lane of the wave calls it.
    template<typename TF, int VALS, int ARITH, int DIR>
    __device__ __forceinline__ void row_fft(cplx<TF>* row, const cplx<TF>* tw, const Row_plan& p, int l)
    {
        using T = cplx<TF>;
        constexpr int sign = DIR == ROW_X_FWD || DIR == ROW_Y_FWD ? -1 : 1;
        const int L = 1 << p.lsh;
        for (int q = 0; q < p.npass; ++q)
        {
            wave_lds_sync();
            with_radix<ARITH>(p.radix[q], [&](auto rc) {
                constexpr int R = decltype(rc)::value, NB = row_rounds(R, VALS, ARITH);
                const int nb = p.nb[q], ns = p.ns[q], ts = p.ts[q];
                const unsigned int mg = p.mg[q];
                auto root = [&](int t) {
                    T w = tw[lpad(t)];
                    if (sign > 0) w.y = -w.y;
                    return w;
                };
                T v[NB*R];
                #pragma unroll
                for (int b = 0; b < NB; ++b)
                    if (b*L < nb)
                    {
                        const int j = min(l + b*L, nb - 1);
                        #pragma unroll
                        for (int r = 0; r < R; ++r) v[b*R + r] = row[lpad(j + r*nb)];
                    }
                wave_lds_sync();
                #pragma unroll
                for (int b = 0; b < NB; ++b)
                    if (b*L < nb)
                    {
                        const int j = min(l + b*L, nb - 1);
                        int d = j;                  // j / ns
                        if (q > 0)
                        {
                            d = static_cast<int>((static_cast<unsigned int>(j)*mg) >> 22);
                            const int kt = (j - d*ns)*ts;
                            #pragma unroll
                            for (int r = 1; r < R; ++r)
                            {
                                // (the FP32 forward x kernel's one exception)
                                if (sizeof(TF) == 4 && DIR == ROW_X_FWD && R == 8 && ARITH == ROW_RADIX8 && r == 1)
                                    v[b*R + r] = turn<true>(v[b*R + r], root(r*kt));
                                else v[b*R + r] = turn<false>(v[b*R + r], root(r*kt));
                            }
                        }
                        const bool keep = l + b*L < nb;
                        const int o = j + d*ns*(R - 1);
                        if constexpr (ARITH == ROW_DIRECT)
                        {
                            #pragma unroll
                            for (int y = 0; y < R; ++y)
                            {
                                T acc = v[b*R];
                                #pragma unroll
                                for (int r = 1; r < R; ++r)
                                    acc = cadd(acc, turn<DIR != ROW_X_INV>(v[b*R + r], root(((r*y) % R)*nb)));
                                if (keep) row[lpad(o + y*ns)] = acc;
                            }
                        }
                        else
                        {
                            dft<TF, R>(v + b*R, sign);
                            if (keep)
                            {
                                #pragma unroll
                                for (int r = 0; r < R; ++r) row[lpad(o + r*ns)] = v[b*R + r];
                            }
                        }
                    }
            });
        }
        wave_lds_sync();
    }
}
