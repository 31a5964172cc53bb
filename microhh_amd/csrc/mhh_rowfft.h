// mhh_rowfft.h -- FFTs of rows of any length with prime factors up to 13, by
// lane groups of a wavefront.
//
// A group of L lanes (L = 8, 16, 32 or 64; 64/L rows per wave) transforms one
// row in its LDS by the Stockham autosort algorithm, in two to four passes of
// radices up to 16: butterfly j of a pass of radix R takes the elements j + r n/R
// into the registers of lane j mod L and puts its outputs back into the same
// row.  A row belongs to one wave: no block barrier inside a transform.  Large
// composite radices are what keeps the passes few: 384 = 16 6 4 and 360 = 15 6 4
// take three, where radices up to 8 and 5 need four.
//
// Only the forward transform (exp(-2 pi i ..)) is written; the inverse swaps the
// real and imaginary parts of its inputs and outputs.
#pragma once

#include <type_traits>

#include <hip/hip_runtime.h>

#include "mhh_fft.h"
#include "mhh_internal.h"

namespace mhh
{
    constexpr int ROW_VALS = 16, ROW_VALS_WIDE = 32;   // complex values a lane holds in a pass
    constexpr int ROW_ROUNDS = 4;                      // and butterflies

    // Whether the engine has a codelet of this radix.
    inline bool row_radix(int r) { return (r >= 2 && r <= 13) || r == 15 || r == 16; }

    // The factorisation and the lanes per row with the least work per element:
    // for each pass the rounds of L butterflies times their cost (their values
    // through LDS and the arithmetic), times the lanes, idle ones included,
    // among those that hold at most `vals` values per lane.  False if there is
    // none (lengths above 64 vals, primes above 13).
    struct Row_search
    {
        int n, vals, lmin, cur[ROW_MAXPASS];
        double best; Row_plan plan;
    };

    inline void row_search(Row_search& s, int rest, int pass, int maxr)
    {
        if (rest == 1)
        {
            for (int lsh = s.lmin; lsh <= 6; ++lsh)
            {
                const int L = 1 << lsh;
                double cost = 6.*L*pass;     // a pass's trip through LDS
                bool fits = true;
                for (int p = 0; p < pass; ++p)
                {
                    const int R = s.cur[p], rounds = (s.n/R + L - 1)/L;
                    if (rounds*R > s.vals || rounds > ROW_ROUNDS) { fits = false; break; }
                    const bool prime = R == 7 || R == 11 || R == 13;
                    // values and twiddles through LDS, and arithmetic
                    cost += rounds*L*R*((p > 0 ? 3. : 2.) + (prime ? 0.5*R : R > 8 ? 2. : 1.));
                }
                if (fits && cost < s.best)
                {
                    s.best = cost;
                    s.plan.n = s.n; s.plan.npass = pass; s.plan.lsh = lsh; s.plan.vals = s.vals;
                    int ns = 1;
                    for (int p = 0; p < pass; ++p)
                    {
                        const int R = s.cur[p];
                        s.plan.radix[p] = R; s.plan.nb[p] = s.n/R; s.plan.ns[p] = ns; s.plan.ts[p] = s.n/(ns*R);
                        s.plan.mg[p] = static_cast<unsigned int>(((1ll << 22) + ns - 1)/ns);
                        ns *= R;
                    }
                }
            }
            return;
        }
        if (pass == ROW_MAXPASS) return;
        for (int r = maxr < rest ? maxr : rest; r >= 2; --r)
            if (rest % r == 0 && row_radix(r))
            {
                s.cur[pass] = r;
                row_search(s, rest/r, pass + 1, r);
            }
    }

    // The plan of a launch over `rows` rows.  Few rows take more lanes each, so
    // that the launch still has about ROW_WAVES waves (two per SIMD): what a
    // lane does in turn is latency then (90 x 75 x 60 FP64, 8 lanes per row
    // instead of 64: forward x transform 19.2 instead of 13.8 us).
    constexpr int ROW_WAVES = 2048;
    inline bool make_row_plan(int n, long long rows, Row_plan& p)
    {
        p.n = 0;
        if (n < 2 || n > 64*ROW_VALS_WIDE) return false;
        int lmin = 3;
        while (lmin < 6 && (rows << lmin) < 64ll*ROW_WAVES) ++lmin;
        for (int vals : {ROW_VALS, ROW_VALS_WIDE})
        {
            Row_search s{};
            s.n = n; s.vals = vals; s.lmin = lmin; s.best = 1.e300;
            row_search(s, n, 0, 16);
            if (s.best < 1.e300) { p = s.plan; return true; }
        }
        return false;
    }

    // LDS slots of a row (element x at lpad(x)); an odd number, so that equal
    // elements of neighbouring rows sit in different banks.
    __host__ __device__ inline int row_stride(int n) { return (lpad(n - 1) + 1) | 1; }

    // ------------------------------------------------------------ codelets
    template<typename T> __host__ __device__ __forceinline__ T hcadd(T a, T b) { T r; r.x = a.x + b.x; r.y = a.y + b.y; return r; }
    template<typename T> __host__ __device__ __forceinline__ T hcsub(T a, T b) { T r; r.x = a.x - b.x; r.y = a.y - b.y; return r; }

    // cos and sin of 2 pi m / R, m = 1 .. (R-1)/2
    template<int R> struct Prime_trig;
    template<> struct Prime_trig<5>
    {
        static constexpr double c[2] = {0.30901699437494742410, -0.80901699437494742410};
        static constexpr double s[2] = {0.95105651629515357212, 0.58778525229247312917};
    };
    template<> struct Prime_trig<7>
    {
        static constexpr double c[3] = {0.62348980185873353053, -0.22252093395631440429, -0.90096886790241912624};
        static constexpr double s[3] = {0.78183148246802980871, 0.97492791218182360702, 0.43388373911755812048};
    };
    template<> struct Prime_trig<11>
    {
        static constexpr double c[5] = {0.84125353283118116886, 0.41541501300188642553, -0.14231483827328514044,
                                        -0.65486073394528506406, -0.95949297361449738989};
        static constexpr double s[5] = {0.54064081745559758211, 0.90963199535451837141, 0.98982144188093273238,
                                        0.75574957435425828377, 0.28173255684142969771};
    };
    template<> struct Prime_trig<13>
    {
        static constexpr double c[6] = {0.88545602565320989590, 0.56806474673115580251, 0.12053668025532305335,
                                        -0.35460488704253562597, -0.74851074817110109863, -0.97094181742605202716};
        static constexpr double s[6] = {0.46472317204376854566, 0.82298386589365639458, 0.99270887409805399280,
                                        0.93501624268541482344, 0.66312265824079520238, 0.23931566428755776715};
    };

    template<int R> constexpr int codelet_a() { return R == 6 ? 2 : R == 10 ? 2 : R == 12 ? 4 : R == 15 ? 3 : 0; }

    // Forward DFT of R values in registers.
    template<typename TF, int R>
    __host__ __device__ __forceinline__ void rdft(cplx<TF>* v)
    {
        using T = cplx<TF>;
        if constexpr (R == 2)
        {
            const T a = v[0], b = v[1];
            v[0] = hcadd(a, b); v[1] = hcsub(a, b);
        }
        else if constexpr (R == 3)
        {
            const TF h = TF(0.86602540378443864676);  // sqrt(3)/2
            const T s = hcadd(v[1], v[2]), d = hcsub(v[1], v[2]);
            T m; m.x = v[0].x - TF(0.5)*s.x; m.y = v[0].y - TF(0.5)*s.y;
            v[0] = hcadd(v[0], s);
            v[1].x = m.x + h*d.y; v[1].y = m.y - h*d.x;
            v[2].x = m.x - h*d.y; v[2].y = m.y + h*d.x;
        }
        else if constexpr (R == 4)
        {
            const T t0 = hcadd(v[0], v[2]), t1 = hcsub(v[0], v[2]), t2 = hcadd(v[1], v[3]), t3 = hcsub(v[1], v[3]);
            v[0] = hcadd(t0, t2); v[2] = hcsub(t0, t2);
            v[1].x = t1.x + t3.y; v[1].y = t1.y - t3.x;
            v[3].x = t1.x - t3.y; v[3].y = t1.y + t3.x;
        }
        else if constexpr (R == 8)
        {
            T e[4] = {v[0], v[2], v[4], v[6]};
            T o[4] = {v[1], v[3], v[5], v[7]};
            rdft<TF, 4>(e);
            rdft<TF, 4>(o);
            const TF h = TF(0.70710678118654752440);
            T w1; w1.x = h*(o[1].x + o[1].y); w1.y = h*(o[1].y - o[1].x);
            T w2; w2.x = o[2].y; w2.y = -o[2].x;
            T w3; w3.x = h*(o[3].y - o[3].x); w3.y = -h*(o[3].x + o[3].y);
            v[0] = hcadd(e[0], o[0]); v[4] = hcsub(e[0], o[0]);
            v[1] = hcadd(e[1], w1);   v[5] = hcsub(e[1], w1);
            v[2] = hcadd(e[2], w2);   v[6] = hcsub(e[2], w2);
            v[3] = hcadd(e[3], w3);   v[7] = hcsub(e[3], w3);
        }
        else if constexpr (R == 5 || R == 7 || R == 11 || R == 13)
        {
            // pairs x_m +- x_(R-m): the cosine sums of the even part, the sine sums of the odd
            constexpr int H = (R - 1)/2;
            T s[H], d[H];
            #pragma unroll
            for (int m = 0; m < H; ++m) { s[m] = hcadd(v[m+1], v[R-1-m]); d[m] = hcsub(v[m+1], v[R-1-m]); }
            const T x0 = v[0];
            #pragma unroll
            for (int m = 0; m < H; ++m) v[0] = hcadd(v[0], s[m]);
            #pragma unroll
            for (int q = 1; q <= H; ++q)
            {
                T a = x0, b; b.x = TF(0); b.y = TF(0);
                #pragma unroll
                for (int m = 1; m <= H; ++m)
                {
                    const int t = (m*q) % R, i = (t <= H ? t : R - t) - 1;
                    const TF c = TF(Prime_trig<R>::c[i]), sn = TF(t <= H ? Prime_trig<R>::s[i] : -Prime_trig<R>::s[i]);
                    a.x += c*s[m-1].x; a.y += c*s[m-1].y;
                    b.x += sn*d[m-1].x; b.y += sn*d[m-1].y;
                }
                v[q].x = a.x + b.y; v[q].y = a.y - b.x;
                v[R-q].x = a.x - b.y; v[R-q].y = a.y + b.x;
            }
        }
        else if constexpr (R == 9 || R == 16)
        {
            // R = A A: input m = A a + b, output q = qa + A qb, twiddle w_R^(b qa)
            constexpr int A = R == 9 ? 3 : 4;
            constexpr double C9[5] = {1., 0.76604444311897803520, 0.17364817766693034885, -0.5, -0.93969262078590838405};
            constexpr double S9[5] = {0., 0.64278760968653932632, 0.98480775301220805937, 0.86602540378443864676,
                                      0.34202014332566873304};
            constexpr double C16[10] = {1., 0.92387953251128675613, 0.70710678118654752440, 0.38268343236508977173, 0.,
                                        -0.38268343236508977173, -0.70710678118654752440, -0.92387953251128675613, -1.,
                                        -0.92387953251128675613};
            constexpr double S16[10] = {0., 0.38268343236508977173, 0.70710678118654752440, 0.92387953251128675613, 1.,
                                        0.92387953251128675613, 0.70710678118654752440, 0.38268343236508977173, 0.,
                                        -0.38268343236508977173};
            T y[A][A];
            #pragma unroll
            for (int b = 0; b < A; ++b)
            {
                #pragma unroll
                for (int a = 0; a < A; ++a) y[b][a] = v[A*a + b];
                rdft<TF, A>(y[b]);
                #pragma unroll
                for (int qa = 1; qa < A; ++qa)
                    if (b > 0)
                    {
                        const int t = b*qa;   // at most 4 (R = 9) or 9 (R = 16)
                        const T z = y[b][qa];
                        if (R == 16 && t == 4) { y[b][qa].x = z.y; y[b][qa].y = -z.x; }
                        else
                        {
                            const TF c = TF(R == 9 ? C9[t < 5 ? t : 0] : C16[t]), sn = TF(R == 9 ? S9[t < 5 ? t : 0] : S16[t]);
                            y[b][qa].x = c*z.x + sn*z.y; y[b][qa].y = c*z.y - sn*z.x;
                        }
                    }
            }
            #pragma unroll
            for (int qa = 0; qa < A; ++qa)
            {
                T t[A];
                #pragma unroll
                for (int b = 0; b < A; ++b) t[b] = y[b][qa];
                rdft<TF, A>(t);
                #pragma unroll
                for (int qb = 0; qb < A; ++qb) v[qa + A*qb] = t[qb];
            }
        }
        else
        {
            // coprime factors A B: with input m = B a + A b (mod R) the DFT is that
            // of a over A and of b over B, output q = (q mod A, q mod B): no twiddles
            constexpr int A = codelet_a<R>(), B = R/A;
            T y[B][A];
            #pragma unroll
            for (int b = 0; b < B; ++b)
            {
                #pragma unroll
                for (int a = 0; a < A; ++a) y[b][a] = v[(B*a + A*b) % R];
                rdft<TF, A>(y[b]);
            }
            #pragma unroll
            for (int qa = 0; qa < A; ++qa)
            {
                T t[B];
                #pragma unroll
                for (int b = 0; b < B; ++b) t[b] = y[b][qa];
                rdft<TF, B>(t);
                #pragma unroll
                for (int q = 0; q < R; ++q)
                    if (q % A == qa) v[q] = t[q % B];
            }
        }
    }

    // -------------------------------------------------------------- passes
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

    // Calls f.template operator()<R>() of the pass's radix (uniform).
    template<typename F>
    __device__ __forceinline__ void with_radix(int R, F f)
    {
        switch (R)
        {
            case 2: f(std::integral_constant<int, 2>{}); break;
            case 3: f(std::integral_constant<int, 3>{}); break;
            case 4: f(std::integral_constant<int, 4>{}); break;
            case 5: f(std::integral_constant<int, 5>{}); break;
            case 6: f(std::integral_constant<int, 6>{}); break;
            case 7: f(std::integral_constant<int, 7>{}); break;
            case 8: f(std::integral_constant<int, 8>{}); break;
            case 9: f(std::integral_constant<int, 9>{}); break;
            case 10: f(std::integral_constant<int, 10>{}); break;
            case 11: f(std::integral_constant<int, 11>{}); break;
            case 12: f(std::integral_constant<int, 12>{}); break;
            case 13: f(std::integral_constant<int, 13>{}); break;
            case 15: f(std::integral_constant<int, 15>{}); break;
            default: f(std::integral_constant<int, 16>{}); break;
        }
    }

    // The transform of one row, in place in the group's LDS, by its L lanes; tw:
    // the table of n roots in LDS.  Every lane of the wave calls it.
    template<typename TF, int VALS>
    __device__ __forceinline__ void row_fft(cplx<TF>* row, const cplx<TF>* tw, const Row_plan& p, int l)
    {
        using T = cplx<TF>;
        const int L = 1 << p.lsh;
        for (int q = 0; q < p.npass; ++q)
        {
            wave_lds_sync();
            with_radix(p.radix[q], [&](auto rc) {
                constexpr int R = decltype(rc)::value, NB = VALS/R < ROW_ROUNDS ? VALS/R : ROW_ROUNDS;
                const int nb = p.nb[q], ns = p.ns[q], ts = p.ts[q];
                const unsigned int mg = p.mg[q];
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
                            for (int r = 1; r < R; ++r) v[b*R + r] = cmul(v[b*R + r], tw[lpad(r*kt)]);
                        }
                        rdft<TF, R>(v + b*R);
                        if (l + b*L < nb)
                        {
                            const int o = j + d*ns*(R - 1);
                            #pragma unroll
                            for (int r = 0; r < R; ++r) row[lpad(o + r*ns)] = v[b*R + r];
                        }
                    }
            });
        }
        wave_lds_sync();
    }
}
