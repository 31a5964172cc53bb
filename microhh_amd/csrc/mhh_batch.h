// mhh_batch.h -- kernels as functors, launched for one context or batched
// over the contexts of an ensemble.
//
// A kernel of the batchable path is a trivially copyable struct K holding its
// arguments, with NT / MINB (its launch bounds) and a device operator()(Bid)
// that does one block's work.  launch() either runs it on the context's own
// stream (one_g<K>, blockIdx as the block index), or, while the context
// records into a batch (mhh_batch_begin .. mhh_batch_end), appends K, its grid
// and block to the context's sequence.  At the end of the recording the
// sequences of all members are merged: the members whose next kernel is of the
// same type run it in one launch of batch_g<K>, whose blocks are dealt to the
// members through a table of first blocks, so an ensemble of small, uneven
// grids fills the chip with one launch per kernel type instead of one per
// member and kernel.
#pragma once

#include <type_traits>

#include "mhh_internal.h"

namespace mhh
{
    // Block index and grid of one context's launch.
    struct Bid { int x, y, z, nx, ny, nz; };

    template<typename K>
    __device__ __forceinline__ void run_one(const K& k)
    {
        k(Bid{static_cast<int>(blockIdx.x), static_cast<int>(blockIdx.y), static_cast<int>(blockIdx.z),
              static_cast<int>(gridDim.x), static_cast<int>(gridDim.y), static_cast<int>(gridDim.z)});
    }

    // One member's share of a batched launch: blocks first .. first + nx ny nz
    // - 1 (first a multiple of 8, so a block still runs on the XCD its index
    // selects, b % 8, for the kernels whose tile order relies on it), its
    // functor at byte `off` of the argument buffer.
    struct Batch_slot { int first, nx, ny, nz; unsigned int off; int pad[3]; };

    template<typename K>
    __device__ __forceinline__ void run_batch(const Batch_slot* __restrict__ slot, int n,
                                              const unsigned char* __restrict__ args)
    {
        // the member of this block: the last slot whose first block is <= b
        const int b = static_cast<int>(blockIdx.x);
        int lo = 0, hi = n - 1;
        while (lo < hi)
        {
            const int mid = (lo + hi + 1) >> 1;
            if (slot[mid].first <= b) lo = mid; else hi = mid - 1;
        }
        const int first = slot[lo].first, nx = slot[lo].nx, ny = slot[lo].ny, nz = slot[lo].nz;
        const int l = b - first, nxy = nx*ny;
        if (l >= nxy*nz) return;   // blocks that pad the next member's start to a multiple of 8
        const K& k = *reinterpret_cast<const K*>(args + slot[lo].off);
        k(Bid{l % nx, (l / nx) % ny, l / nxy, nx, ny, nz});
    }

    // The kernels: K::NT threads per block at most and, for K::MINB > 0, at
    // least K::MINB waves per SIMD (amdgpu_waves_per_eu); K::MINB = 0 leaves
    // the occupancy to the compiler's scheduler.
    template<typename K>
    __global__ void __launch_bounds__(K::NT, K::MINB) one_g(K k) { run_one(k); }
    template<typename K>
    __global__ void __launch_bounds__(K::NT) one_g0(K k) { run_one(k); }
    template<typename K>
    __global__ void __launch_bounds__(K::NT, K::MINB) batch_g(const Batch_slot* __restrict__ slot, int n,
                                                              const unsigned char* __restrict__ args)
    { run_batch<K>(slot, n, args); }
    template<typename K>
    __global__ void __launch_bounds__(K::NT) batch_g0(const Batch_slot* __restrict__ slot, int n,
                                                      const unsigned char* __restrict__ args)
    { run_batch<K>(slot, n, args); }

    // Launches batch_g<K> over n slots; the type-erased entry of a recording.
    using Batch_fn = int (*)(const Batch_slot* slot, int n, const unsigned char* args, int nblocks, dim3 block,
                             size_t lds, hipStream_t stream);

    template<typename K>
    int batch_launch(const Batch_slot* slot, int n, const unsigned char* args, int nblocks, dim3 block, size_t lds,
                     hipStream_t stream)
    {
        if constexpr (K::MINB > 0) batch_g<K><<<nblocks, block, lds, stream>>>(slot, n, args);
        else batch_g0<K><<<nblocks, block, lds, stream>>>(slot, n, args);
        return check_launch("batched launch");
    }

    // Bytes of an argument buffer that is made for `size` bytes.  Twice as many: the
    // substeps of a step differ (12 members FP32: 47, 19, 64 and 67 kB), and a buffer that
    // has to grow in the middle of a step waits for the GPU and is allocated
    // anew (1.1 to 1.6 ms of a first step of 3.5).
    inline size_t batch_capacity(size_t size)
    {
        const size_t cap = (2*size + 4095)/4096*4096;
        return cap > 65536 ? cap : 65536;
    }

    // Appends one launch to the sequence of the recording context (mhh_batch.hip).
    void batch_record(mhh_ctx* c, Batch_fn fn, const void* k, size_t size, dim3 grid, dim3 block, size_t lds);
    // A device double that the end of the recording copies to *dst (the
    // result of a reduction the recording context would have read at once).
    void batch_readback(mhh_ctx* c, const double* src, double* dst);
    // Device memory that recorded launches may use, freed after they ran.
    void batch_defer_free(mhh_ctx* c, void* ptr);

    // Records a kernel that runs as a functor only in a batch (its form outside
    // one is a kernel of its own).
    template<typename K>
    void record(mhh_ctx* c, const K& k, dim3 grid, dim3 block, size_t lds = 0)
    {
        static_assert(std::is_trivially_copyable<K>::value, "kernel functors are copied bytewise");
        static_assert(alignof(K) <= 16, "kernel functors are stored at 16-byte boundaries");
        if (grid.x == 0 || grid.y == 0 || grid.z == 0) return;
        batch_record(c, &batch_launch<K>, &k, sizeof(K), grid, block, lds);
    }

    template<typename K>
    void launch(mhh_ctx* c, const K& k, dim3 grid, dim3 block, size_t lds = 0)
    {
        if (c->rec) return record(c, k, grid, block, lds);
        if (grid.x == 0 || grid.y == 0 || grid.z == 0) return;
        if constexpr (K::MINB > 0) one_g<K><<<grid, block, lds, c->stream>>>(k);
        else one_g0<K><<<grid, block, lds, c->stream>>>(k);
    }
}

// Entry points whose kernels are not functors (or that read results back at
// once) refuse to run while their context records into a batch.
#define MHH_NOT_IN_BATCH(ctx, name) do { \
    if ((ctx) && (ctx)->rec) return mhh::fail(MHH_ESTATE, std::string(name) + " cannot be recorded into a batch"); \
    } while (0)
