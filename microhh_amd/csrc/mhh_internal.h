// mhh_internal.h -- shared definitions of the gfx950 kernels and the C ABI layer.
#pragma once

#include <hip/hip_runtime.h>
#include <climits>
#include <cstdint>
#include <map>
#include <string>
#include <utility>
#include <vector>

#include "microhh_amd.h"

namespace mhh
{
    // Loop bounds and strides passed by value to every kernel (Grid_data,
    // include/grid.h:49-138, serial share: imax = itot, jmax = jtot).
    struct Gd
    {
        int itot, jtot, ktot;
        int igc, jgc, kgc;
        int istart, iend, jstart, jend, kstart, kend;
        int icells, jcells, kcells, ijcells, ncells;
        double dx, dy, dxi, dyi;
    };

    // The per-level factors of the fused tendency kernel in one record, so
    // that one scalar load brings all of them for a level.
    template<typename TF>
    struct Level
    {
        TF rho, rhoh, rhohp;      // rhoref[k], rhorefh[k], rhorefh[k+1]
        TF dzi, dzhi, dzhip;      // dzi[k], dzhi[k], dzhi[k+1]
        TF cfac;                  // dzi/rhoref: vertical flux divergence factor of cell-centred fields
        TF wfac;                  // dzhi/rhorefh: the same for w
        TF gthi;                  // grav/threfh (0 without a base state)
        TF threfh_rel;            // threfh - offset of scalar 0
        TF n2fac;                 // grav/thref * 0.5 * dzi: N2 per theta difference over k-1..k+1
    };

    // Element i of a table that no kernel writes, read through the constant
    // address space: a load at a uniform index is then a scalar load, however
    // the pointer reached the kernel (a batched launch reads its pointers
    // from memory, which hides from the compiler that nothing stores there).
    template<typename T>
    __device__ __forceinline__ T ld_const(const T* p, int i)
    {
        static_assert(sizeof(T) % 4 == 0, "ld_const reads whole 32-bit words");
        using W = const __attribute__((address_space(4))) uint32_t;
        W* q = (W*)(p + i);
        uint32_t w[sizeof(T)/4];
        #pragma unroll
        for (int k = 0; k < static_cast<int>(sizeof(T)/4); ++k) w[k] = q[k];
        T t;
        __builtin_memcpy(&t, w, sizeof(T));
        return t;
    }

    // Device copies of the 1-D grid and base-state profiles in the element type.
    template<typename TF>
    struct Prof
    {
        TF* z = nullptr; TF* zh = nullptr; TF* dz = nullptr; TF* dzh = nullptr;
        TF* dzi = nullptr; TF* dzhi = nullptr; TF* rhoref = nullptr; TF* rhorefh = nullptr;
        TF* thref = nullptr; TF* threfh = nullptr;
        TF* threfh_rel = nullptr;   // threfh - offset of scalar 0 (the buoyancy difference)
        Level<TF>* lev = nullptr;   // kcells records
    };

    // Pressure-solver tables (Pres_2::set_values, src/pres_2.cxx:124-153) and
    // FFT twiddles.
    template<typename TF>
    struct Pres_tables
    {
        TF* bmati = nullptr;    // itot
        TF* bmatj = nullptr;    // jtot
        TF* a = nullptr;        // kmax
        TF* c = nullptr;        // kmax
        TF* ac = nullptr;       // kmax: a + c
        TF* dz2 = nullptr;      // kmax: dz*dz
        TF* dz2rho = nullptr;   // kmax: dz*dz*rhoref
        double* twx = nullptr;  // itot complex roots exp(-2 pi i t / itot), (re, im) pairs
        double* twy = nullptr;  // jtot complex roots
        // Elimination of the tridiagonal systems, which depend on the mode
        // only through lambda = bmati[kx] + bmatj[ky] (bmatj[ky] =
        // bmatj[jtot-ky]): one system per l = kx*(jtot/2+1) + min(ky, jtot-ky),
        // nsys of them, stored [k][l].
        int nsys = 0;
        TF* tri_wi = nullptr;   // ktot x nsys: reciprocal pivots
        TF* tri_gam = nullptr;  // ktot x nsys: gamma (k >= 1)
    };
}

namespace mhh
{
    // Plan of a transform by lane groups (mhh_rowfft.h).
    constexpr int ROW_MAXPASS = 8;
    struct Row_plan
    {
        int n = 0;                  // 0: no plan
        int npass;
        int lsh;                    // 1 << lsh lanes per row
        int vals;                   // the kernel instance: ROW_VALS or ROW_VALS_WIDE values per lane
        int arith;                  // and its butterflies: ROW_RADIX8 or ROW_DIRECT
        int radix[ROW_MAXPASS];
        int nb[ROW_MAXPASS];        // butterflies n/R
        int ns[ROW_MAXPASS];        // product of the radices before
        int ts[ROW_MAXPASS];        // twiddle stride n/(ns R)
        unsigned int mg[ROW_MAXPASS];   // j/ns = (j mg) >> 22 for j < 2048, ns >= 2 (32-bit product)
    };
}

struct mhh_surface_state;
struct mhh_buffer_state;

struct mhh_ctx
{
    int precision = MHH_FP64;   // element type of the fields: MHH_FP64 or MHH_FP32
    bool mixed = false;         // MHH_MIXED: FP32 fields, FP64 tridiagonal and divergence
    double s_offset[MHH_MAX_SCALARS] = {};
    // Mixed mode: the horizontal mean of the pressure, solved in FP64.
    double* pm_part = nullptr;   // ktot x PM_CHUNKS partial plane sums of the RHS
    double* pm_mean = nullptr;   // ktot: plane mean of the RHS
    double* pm_coef = nullptr;   // 2 ktot: reciprocal pivots and gamma of the mean-mode elimination
    double* pbar = nullptr;      // kcells: mean pressure per level
    float* dpbar = nullptr;      // kcells: pbar[k] - pbar[k-1], the mean's part of the z gradient
    hipStream_t stream = nullptr;
    int device = 0;
    mhh::Gd gd{};
    std::vector<double> h_z, h_zh, h_dz, h_dzh, h_dzi, h_dzhi, h_rhoref, h_rhorefh, h_thref, h_threfh;
    mhh::Prof<double> pd;
    mhh::Prof<float> pf;
    mhh::Pres_tables<double> td;
    mhh::Pres_tables<float> tf;
    bool have_base_state = false;
    mhh_field_set f{};
    bool bound = false;
    // Levels per block of the fused tendency kernel and of the viscosity
    // plane-ring kernel (0: the built-in choice, march_kchunk).
    int tend_kchunk = 0;
    int visc_kchunk = 0;
    // Spectral transforms through the general LDS engine only (no kernels
    // specialised for n = 128, 256, 512): a check of the specialised ones.
    bool fft_generic = false;
    // y transforms and tridiagonal sweep as separate passes even where the
    // fused ones apply (a check of the fused kernels).
    bool ytri_split = false;
    // Plans of the x and y transforms by lane groups.
    mhh::Row_plan row_px, row_py;
    // Mixed mode, length 1024: x and y transforms as DFT-as-GEMM on the matrix
    // cores (mhh_dft.hip) instead of by lane groups; tables per context.
    bool dft_mfma = true;
    int visc_mode = 0;            // the viscosity with the tendencies: 0 by grid size, 1 two passes, 2 one pass
    void* sfc_keep = nullptr;     // du/dz, dv/dz, db/dz kept for the viscosity (three planes)
    bool sfc_kept = false;        // sfc_keep holds the gradients of the coming viscosity
    void* dft_tab = nullptr;     // 32 x 4 FP16: hi and lo of cos and sin of 2 pi m / 32
    void* dft_tw = nullptr;      // 1024 float2: cos and sin of 2 pi m / 1024
    // A deferred end of the RK3 update (MHH_RK3_DEFER): ut, vt, wt and st[0]
    // hold the tendencies as they were before the pressure gradient and the
    // cA scaling; the reference's values are cA (at - grad p) with the p of
    // the last solve (cA at for the scalar).  The fused tendency pass
    // completes them on the fly; every other call that touches tendencies or
    // p completes them first (settle_tendencies).
    bool defer_pending = false;
    double defer_cA = 0.;
    // Scalars advected with the Koren flux limiter ([advec] fluxlimit_list).
    int fluxlimit[MHH_MAX_SCALARS] = {};
    // Reduction scratch: per-block partial maxima and one result slot.
    double* red = nullptr;
    int red_capacity = 0;
    double* h_red = nullptr;  // pinned host slot for the reduction result
    // Smagorinsky length per level, cs*(dx*dy*dz[k])^(1/3), computed on the host
    // as the reference does (src/diff_smag2.cxx:163) and cached per cs.
    double mlen_cs = -1.;
    double* mlen_d = nullptr;
    float* mlen_f = nullptr;
    // Fixed-flux forcing (mhh_force.hip): the body force and the partial
    // plane sums of u and ut (1 + 2 ktot plane_chunks), and dz (kcells),
    // allocated on first use.
    double* force_buf = nullptr;
    double* force_dz = nullptr;
    // Surface layer and buffer sponge (mhh_surface.hip), when initialised.
    mhh_surface_state* sfc = nullptr;
    mhh_buffer_state* buf = nullptr;
    // Kernel timing: per kernel name, a pool of (start, stop) event pairs and
    // the number recorded since the last reset.
    bool timing = false;
    std::string timing_only;   // non-empty: time only the kernel family of this name
    struct Event_pool { std::vector<std::pair<hipEvent_t, hipEvent_t>> ev; int used = 0; };
    std::map<std::string, Event_pool> timers;
    // While a batch records (mhh_batch_begin .. mhh_batch_end): the batch and
    // this context's member index in it; launches are recorded, not issued.
    mhh_batch* rec = nullptr;
    int rec_member = -1;
};

namespace mhh
{
    void set_error(const std::string& msg);
    int fail(int code, const std::string& msg);
    int check_launch(const char* what);
    int check_hip(hipError_t e, const char* what);
    bool fits_int(long long v);

    // Rows of blocks in k for the 3-D point kernels.
    constexpr int BX = 64;
    constexpr int BY = 4;

    inline dim3 grid3(const Gd& g, int kfirst, int klast)
    {
        return dim3((g.itot + BX - 1)/BX, (g.jtot + BY - 1)/BY, klast > kfirst ? klast - kfirst : 0);
    }

    // XCD-contiguous block order.  Workgroups are dealt to the 8 XCDs round
    // robin (block b to XCD b % 8), each with its own L2; a 1-D grid of nb
    // blocks (nb a multiple of 8) mapped through xcd_tile gives every XCD a
    // contiguous range of tiles, so the rows and planes neighbouring tiles
    // share are fetched into one L2, not eight.
    __host__ __device__ inline int xcd_tile(int b, int nb) { return (b % 8)*(nb/8) + b/8; }
    inline int xcd_blocks(int ntiles) { return (ntiles + 7)/8*8; }

    // Levels per block of the k-marching plane-ring kernels: 64, or fewer
    // on small grids, so that a launch still has about 4 blocks per CU (each
    // chunk reads a few levels past its ends again; 8 levels is the floor), and
    // down to 2 levels while the launch has fewer than `least` blocks and the
    // halved chunks give at most `most`: a level costs a block a trip to memory,
    // and reading the ends again costs little where most of the chip is idle.
    // The results do not depend on it.
    // least: a block per CU for the tendency passes, whose chunks begin with a
    // dozen planes (32^3 FP32, 32 blocks of 8 levels: 27.6 us, 128 of 2: 14.5; but
    // 90 x 75 x 60 FP64, 304 blocks of 8, gains nothing from 4, and 150 x 100 x 75
    // FP32, 750 of 8, loses a fifth), four for the viscosity (32^3 13.5 and 8.5 us).
    constexpr int MARCH_LEAST_TEND = 256, MARCH_LEAST_VISC = 1024;
    inline int march_kchunk(int ntiles_xy, int ktot, int least, int most)
    {
        auto blocks = [&](int kc) { return static_cast<long>(ntiles_xy)*((ktot + kc - 1)/kc); };
        int kc = 64;
        while (kc > 8 && blocks(kc) < 1024) kc /= 2;
        while (kc > 2 && blocks(kc) < least && blocks(kc/2) <= most) kc /= 2;
        return kc;
    }

    // most, for the viscosity: the blocks of its kernels that run at once (their
    // VGPRs leave 8 on a CU in FP32, 7 with Mason damping, 5 with the limits, and 4 in FP64
    // with the surface model or the limits).  Beyond that the short chunks run in a second
    // round, which costs what they saved: 128 x 128 x 96 FP64 with the surface
    // model, 768 blocks of 8 levels 24.7 us, 1536 of 4 27.8; 96 x 96 x 64, 768
    // of 4 14.5, 1536 of 2 17.9; 256 x 160 x 24 FP32 with Mason damping, 960 of 4
    // 12.8, 1920 of 2 15.6.  FP64 without a surface model has 5 on a CU and
    // gains up to 6 (128 x 128 x 96 20.5 us by 768, 19.0 by 1536; 192 x 144 x 64 22.7 by 864, 24.2 by 1728).
    inline int visc_most(bool fp64, bool limits, bool sfc, bool mason)
    {
        if (fp64) return sfc || limits ? 1024 : 1536;
        return limits ? 1280 : sfc && mason ? 1792 : 2048;
    }

    // While a context records into a batch its marching kernels run
    // merged with the other members', which fill the chip together, so each
    // member marches 32 levels per chunk (64-member ensemble step: 8.30 ms,
    // against 8.83 with 64 levels and 8.49 with 16).
    inline int march_kchunk(const mhh_ctx* c, int ntiles_xy, int ktot, int least, int most = INT_MAX)
    {
        return c->rec ? 32 : march_kchunk(ntiles_xy, ktot, least, most);
    }

    // Max-reductions: each thread folds a chunk of RED_KCHUNK levels of its
    // column, each block writes one partial, one block folds the partials.
    constexpr int RED_KCHUNK = 32;
    inline dim3 grid_red(const Gd& g)
    {
        return dim3((g.itot + BX - 1)/BX, (g.jtot + BY - 1)/BY, (g.ktot + RED_KCHUNK - 1)/RED_KCHUNK);
    }

    // Maximum over a device array of per-block partial maxima, returned on the host.
    int reduce_max_partials(mhh_ctx* ctx, int npartials, double* out);
    int reduce_max_partials_at(mhh_ctx* ctx, double* base, int npartials, double* out);
    int ensure_reduction(mhh_ctx* ctx, int nblocks);

    // This device's copy of the allocation-free reductions' scratch array
    // (MHH_NOALLOC_SCRATCH_BYTES), looked up when the first context on the
    // device was created; null before that.
    double* static_scratch(int device);
    // Folds npartials device partial maxima into the device double *out on
    // the context stream, without a host copy or synchronisation.
    int fold_max_to_device(mhh_ctx* ctx, const double* partials, int npartials, double* out);

    // Brackets the launches issued during its lifetime with HIP events on the
    // context stream when timing is enabled.
    class Timer
    {
        public:
            Timer(mhh_ctx* c, const char* name);
            ~Timer();
        private:
            mhh_ctx* c;
            hipEvent_t stop = nullptr;
    };

    // Periodic halos of one field (Boundary_cyclic::exec; mhh_boundary.hip).
    int cyclic_field(mhh_ctx* c, void* field, int edge);

    // Zero the ghost cells of a tendency field (mhh_boundary.hip).
    template<typename TF> int zero_tendency_ghosts(mhh_ctx* c, TF* const* at, int n);
    // RK3 update of one field and its tendency (a += cBdt*at; at = zero ? 0 :
    // cAn*at), the tendency's ghost cells cleared when zero.
    template<typename TF> int rk3_field(mhh_ctx* c, TF* a, TF* at, TF cBdt, TF cAn, int zero);

    // Partial sums per level of the mixed mode's plane mean.
    constexpr int PM_CHUNKS = 16;

    // Completes a deferred RK3 tendency update, if one is pending (mhh_pres.hip).
    int settle_tendencies(mhh_ctx* ctx);

    // Uploads what the Smagorinsky viscosity of these parameters needs once
    // (the length scale per level), so that later calls queue kernels only
    // (mhh_diff.hip).
    int smag_prepare(mhh_ctx* ctx, const mhh_smag_params& par);

    // Pressure solver setup (mhh_pres.hip).
    int pres_init(mhh_ctx* ctx);
    void pres_free(mhh_ctx* ctx);

    // DFT-as-GEMM transforms of length 1024 in the mixed mode (mhh_dft.hip):
    // whether they replace the lane groups for a length n, their tables,
    // and the forward x (real rows of P minus the plane mean -> C[k][kx][j]),
    // y (in place on C's rows, sign -1 forward, +1 inverse with 1/jtot) and
    // inverse x (C -> ghosted p with halos, 1/itot) passes.
    bool dft_applies(const mhh_ctx* ctx, int n);
    int dft_init(mhh_ctx* ctx);
    void dft_free(mhh_ctx* ctx);
    int dft_x_fwd(mhh_ctx* ctx, const float* P, float2* C, const double* pmean);
    int dft_y(mhh_ctx* ctx, float2* C, int nrows, int sign);
    int dft_x_bwd(mhh_ctx* ctx, const float2* C, float* p);

    // Transforms by lane groups for lengths without kernels of their own
    // (mhh_rowfft.hip): the plans of a context (n = 0 where there
    // is none); the forward x transform of the projection's right-hand side,
    // evaluated in it or (mixed mode) read from P minus the plane means pm_mean, into
    // C[k][kx][j]; the y transforms in place on C's rows (sign -1 forward, +1
    // inverse with 1/jtot); the inverse x transform into the ghosted p with halos,
    // 1/itot.
    void row_plans_init(mhh_ctx* ctx);
    template<typename TF, typename T>
    int row_x_fwd(mhh_ctx* ctx, const TF* P, T* C, const double* tw, const Prof<TF>& p, TF dxi, TF dyi, TF dti);
    template<typename TF, typename T> int row_y(mhh_ctx* ctx, T* C, const double* tw, int sign, int nrows, const char* name);
    template<typename TF, typename T> int row_x_bwd(mhh_ctx* ctx, const T* C, TF* p, const double* tw);

    // Surface layer and buffer state (mhh_surface.hip).
    void surface_free(mhh_ctx* ctx);

    // Plane sums and means (mhh_stats.hip) of nf fields in one pass, FP64 sums
    // over the interior in a fixed order.  plane_sums: partial sums of the levels
    // k0 .. k0+nk-1, part[(field*nk + level)*plane_chunks + chunk].
    // mean_profiles: the horizontal means of every level
    // (src/field3d_operators.cxx:46-66) into the device array
    // prof[field*kcells + level]; part: nf*kcells*plane_chunks values of scratch.
    template<typename TF> struct Plane_fields { const TF* a[3 + MHH_MAX_SCALARS]; };
    int plane_chunks(const Gd& g);
    template<typename TF> int plane_sums(mhh_ctx* c, const Plane_fields<TF>& f, int nf, int k0, int nk, double* part);
    template<typename TF> int mean_profiles(mhh_ctx* c, const Plane_fields<TF>& f, int nf, double* part, double* prof);
}

#define MHH_CHECK(call) do { int _rc = (call); if (_rc) return _rc; } while (0)
#define MHH_REQUIRE_BOUND(ctx) do { \
    if (!(ctx)) return mhh::fail(MHH_EINVAL, "null context"); \
    if (!(ctx)->bound) return mhh::fail(MHH_ESTATE, "fields are not bound (call mhh_fields_bind)"); } while (0)
