// mhh_batch.hip -- batched launches over the contexts of an ensemble.
//
// The reference advances one model per process (src/model.cxx:356-545).  An
// ensemble of small, uneven grids issued model by model leaves the chip
// mostly idle: a 32^3 member's kernels have a few dozen blocks each, and the
// run is bound by the launch rate.  A batch records the members' kernel
// sequences (mhh_batch.h: every kernel of the fused substep is a functor) and
// runs them merged: the members whose next kernel is of the same type run it
// in one launch, whose blocks a table of first blocks deals to the members.
// Members of different sizes take different transform kernels (the wave
// kernels for 128, 256, 512 points, lane groups otherwise); the merge
// then issues each kernel type once over the members that use it.
#include <algorithm>
#include <cstring>

#include "mhh_batch.h"

struct mhh_batch
{
    std::vector<mhh_ctx*> ctx;
    hipStream_t stream = nullptr;
    bool recording = false;

    // one recorded launch: the type-erased batched launcher (one per functor
    // type, so equal pointers mean the same kernel), the functor's bytes
    struct Item { mhh::Batch_fn fn; size_t off, size; dim3 grid, block; size_t lds; };
    std::vector<std::vector<Item>> items;   // per member, in issue order
    std::vector<unsigned char> bytes;       // the recorded functors
    struct Readback { const double* src; double* dst; };
    std::vector<Readback> readbacks;
    std::vector<void*> deferred_free;

    // the merged launches of the last end(): argument and slot offsets
    // within the uploaded buffer
    struct Launch { mhh::Batch_fn fn; dim3 block; size_t lds; int nslots, nblocks; size_t slot_off; };
    std::vector<Launch> launches;
    int recorded = 0;

    // uploads: a pinned staging buffer (reused once the event says its last
    // copy is done) and a few device buffers, each keeping the blob it holds
    // so that a repeated substep (same arguments) needs no copy
    unsigned char* h_stage = nullptr;
    size_t h_cap = 0;
    hipEvent_t staged = nullptr;
    struct Dev_buf { unsigned char* d = nullptr; size_t cap = 0; std::vector<unsigned char> blob; long use = -1; };
    Dev_buf dev[4];
    long uses = 0;
    double* h_rb = nullptr;   // pinned slots of the readbacks
    double* d_rb = nullptr;   // their device staging
    int rb_cap = 0;
};

namespace
{
    // The readback values of a batch gathered into one array, so that one
    // copy brings them to the host.
    __global__ void gather_g(const double* const* __restrict__ src, double* __restrict__ dst, int n)
    {
        const int i = blockIdx.x*blockDim.x + threadIdx.x;
        if (i < n) dst[i] = *src[i];
    }

    using mhh::fail;
    using mhh::check_hip;
    using mhh::Batch_slot;
    using mhh::batch_capacity;

    constexpr size_t ALIGN = 16;
    size_t align_up(size_t x, size_t a) { return (x + a - 1)/a*a; }

    bool same_kernel(const mhh_batch::Item& a, const mhh_batch::Item& b)
    {
        return a.fn == b.fn && a.block.x == b.block.x && a.block.y == b.block.y && a.block.z == b.block.z;
    }

    // Merge the members' sequences into launches and build the blob that
    // goes to the device: every functor at a 16-byte boundary, then the slot
    // tables.  Order: repeatedly take a kernel type that is next for some
    // members and run it for all of them, keeping each member's own order
    // (members are independent of each other).  Preferred is a type that no
    // other member still has waiting further down its sequence (running it
    // now cannot split it into two launches), and among those the one next
    // for the most members (ties: the lowest member index); without such a
    // type, the one next for the most members.
    int merge(mhh_batch* b, std::vector<unsigned char>& blob, size_t* rb_off)
    {
        const int n = static_cast<int>(b->ctx.size());
        b->launches.clear();
        std::vector<size_t> head(n, 0);
        std::vector<std::vector<std::pair<int, size_t>>> groups;   // per launch: (member, item)
        for (;;)
        {
            int best = -1, best_count = 0;
            bool best_free = false;
            for (int m = 0; m < n; ++m)
            {
                if (head[m] >= b->items[m].size()) continue;
                const auto& it = b->items[m][head[m]];
                // each type once: at the first member that has it next
                bool seen = false;
                for (int q = 0; q < m && !seen; ++q)
                    seen = head[q] < b->items[q].size() && same_kernel(b->items[q][head[q]], it);
                if (seen) continue;
                int count = 0;
                bool free = true;
                for (int q = 0; q < n; ++q)
                {
                    const auto& seq = b->items[q];
                    if (head[q] >= seq.size()) continue;
                    if (same_kernel(seq[head[q]], it)) { ++count; continue; }
                    for (size_t r = head[q] + 1; r < seq.size() && free; ++r)
                        free = !same_kernel(seq[r], it);
                }
                if ((free && !best_free) || (free == best_free && count > best_count))
                {
                    best = m; best_count = count; best_free = free;
                }
            }
            if (best < 0) break;
            const auto key = b->items[best][head[best]];
            std::vector<std::pair<int, size_t>> grp;
            for (int m = 0; m < n; ++m)
            {
                if (head[m] >= b->items[m].size()) continue;
                if (same_kernel(b->items[m][head[m]], key))
                    grp.emplace_back(m, head[m]++);
            }
            groups.push_back(std::move(grp));
        }
        // functors first
        blob.clear();
        std::vector<std::vector<unsigned int>> offs(groups.size());
        for (size_t l = 0; l < groups.size(); ++l)
            for (const auto& mi : groups[l])
            {
                const auto& it = b->items[mi.first][mi.second];
                const size_t o = align_up(blob.size(), ALIGN);
                if (o + it.size > 0xffffffffu) return fail(MHH_EINVAL, "mhh_batch_end: arguments exceed 4 GB");
                blob.resize(o + it.size);
                std::memcpy(blob.data() + o, b->bytes.data() + it.off, it.size);
                offs[l].push_back(static_cast<unsigned int>(o));
            }
        // then one slot table per launch
        for (size_t l = 0; l < groups.size(); ++l)
        {
            const size_t so = align_up(blob.size(), ALIGN);
            const int ns = static_cast<int>(groups[l].size());
            blob.resize(so + sizeof(Batch_slot)*ns);
            Batch_slot* slot = reinterpret_cast<Batch_slot*>(blob.data() + so);
            long long first = 0;
            size_t lds = 0;
            for (int s = 0; s < ns; ++s)
            {
                const auto& it = b->items[groups[l][s].first][groups[l][s].second];
                const long long nb = static_cast<long long>(it.grid.x)*it.grid.y*it.grid.z;
                Batch_slot sl{};
                sl.first = static_cast<int>(first);
                sl.nx = static_cast<int>(it.grid.x); sl.ny = static_cast<int>(it.grid.y);
                sl.nz = static_cast<int>(it.grid.z);
                sl.off = offs[l][s];
                std::memcpy(slot + s, &sl, sizeof(sl));
                first += (nb + 7)/8*8;
                if (first >= 0x7fffffffLL) return fail(MHH_EINVAL, "mhh_batch_end: a merged launch exceeds 2^31 blocks");
                lds = std::max(lds, it.lds);
            }
            const auto& k0 = b->items[groups[l][0].first][groups[l][0].second];
            b->launches.push_back({k0.fn, k0.block, lds, ns, static_cast<int>(first), so});
        }
        // the source addresses of the readbacks
        *rb_off = align_up(blob.size(), ALIGN);
        blob.resize(*rb_off + sizeof(const double*)*b->readbacks.size());
        for (size_t r = 0; r < b->readbacks.size(); ++r)
            std::memcpy(blob.data() + *rb_off + r*sizeof(const double*), &b->readbacks[r].src, sizeof(const double*));
        return 0;
    }

    // A device buffer holding blob: one that holds it already, else the least
    // recently used one, refilled through the pinned staging buffer.
    int upload(mhh_batch* b, const std::vector<unsigned char>& blob, unsigned char** out)
    {
        ++b->uses;
        for (auto& db : b->dev)
            if (db.d && db.blob.size() == blob.size() && std::memcmp(db.blob.data(), blob.data(), blob.size()) == 0)
            {
                db.use = b->uses;
                *out = db.d;
                return 0;
            }
        auto* victim = &b->dev[0];
        for (auto& db : b->dev) if (db.use < victim->use) victim = &db;
        if (victim->cap < blob.size())
        {
            // the stream may still read the old buffer: free it after the queued work
            if (victim->d)
            {
                MHH_CHECK(check_hip(hipStreamSynchronize(b->stream), "hipStreamSynchronize"));
                (void)hipFree(victim->d);
                victim->d = nullptr;
                victim->cap = 0;
            }
            const size_t cap = batch_capacity(blob.size());
            MHH_CHECK(check_hip(hipMalloc(&victim->d, cap), "hipMalloc(batch arguments)"));
            victim->cap = cap;
        }
        if (b->h_cap < blob.size())
        {
            MHH_CHECK(check_hip(hipEventSynchronize(b->staged), "hipEventSynchronize"));
            if (b->h_stage) (void)hipHostFree(b->h_stage);
            b->h_stage = nullptr;
            b->h_cap = 0;
            const size_t cap = batch_capacity(blob.size());
            MHH_CHECK(check_hip(hipHostMalloc(reinterpret_cast<void**>(&b->h_stage), cap, hipHostMallocDefault),
                                "hipHostMalloc(batch staging)"));
            b->h_cap = cap;
        }
        // the staging buffer's previous copy must be done before it is rewritten
        MHH_CHECK(check_hip(hipEventSynchronize(b->staged), "hipEventSynchronize"));
        std::memcpy(b->h_stage, blob.data(), blob.size());
        // the copy is ordered after the launches that may still read this
        // device buffer's previous contents (one stream)
        MHH_CHECK(check_hip(hipMemcpyAsync(victim->d, b->h_stage, blob.size(), hipMemcpyHostToDevice, b->stream),
                            "hipMemcpyAsync(batch arguments)"));
        MHH_CHECK(check_hip(hipEventRecord(b->staged, b->stream), "hipEventRecord"));
        victim->blob = blob;
        victim->use = b->uses;
        *out = victim->d;
        return 0;
    }

    // Upload the merged launches' arguments, run them, and deliver the readbacks.
    int issue(mhh_batch* b, const std::vector<unsigned char>& blob, size_t rb_off, int nrb)
    {
        if (b->launches.empty() && nrb == 0) return 0;
        if (nrb > b->rb_cap)
        {
            MHH_CHECK(check_hip(hipStreamSynchronize(b->stream), "hipStreamSynchronize"));
            if (b->h_rb) (void)hipHostFree(b->h_rb);
            if (b->d_rb) (void)hipFree(b->d_rb);
            b->h_rb = nullptr; b->d_rb = nullptr;
            b->rb_cap = 0;
            MHH_CHECK(check_hip(hipHostMalloc(reinterpret_cast<void**>(&b->h_rb), sizeof(double)*nrb,
                                              hipHostMallocDefault), "hipHostMalloc(batch readbacks)"));
            MHH_CHECK(check_hip(hipMalloc(&b->d_rb, sizeof(double)*nrb), "hipMalloc(batch readbacks)"));
            b->rb_cap = nrb;
        }
        unsigned char* d = nullptr;
        MHH_CHECK(upload(b, blob, &d));
        for (const auto& l : b->launches)
            MHH_CHECK(l.fn(reinterpret_cast<const Batch_slot*>(d + l.slot_off), l.nslots, d, l.nblocks, l.block,
                           l.lds, b->stream));
        if (nrb == 0) return 0;
        gather_g<<<(nrb + 255)/256, 256, 0, b->stream>>>(reinterpret_cast<const double* const*>(d + rb_off),
                                                         b->d_rb, nrb);
        MHH_CHECK(mhh::check_launch("batch readbacks"));
        MHH_CHECK(check_hip(hipMemcpyAsync(b->h_rb, b->d_rb, sizeof(double)*nrb, hipMemcpyDeviceToHost, b->stream),
                            "hipMemcpyAsync(batch readbacks)"));
        MHH_CHECK(check_hip(hipStreamSynchronize(b->stream), "hipStreamSynchronize"));
        for (int r = 0; r < nrb; ++r) *b->readbacks[r].dst = b->h_rb[r];
        return 0;
    }

    void stop_recording(mhh_batch* b)
    {
        for (mhh_ctx* c : b->ctx) { c->rec = nullptr; c->rec_member = -1; }
        b->recording = false;
    }

    void release(mhh_batch* b)
    {
        if (b->stream) (void)hipStreamSynchronize(b->stream);
        if (b->recording) stop_recording(b);
        for (auto& db : b->dev) if (db.d) (void)hipFree(db.d);
        if (b->h_stage) (void)hipHostFree(b->h_stage);
        if (b->h_rb) (void)hipHostFree(b->h_rb);
        if (b->d_rb) (void)hipFree(b->d_rb);
        if (b->staged) (void)hipEventDestroy(b->staged);
        delete b;
    }
}

namespace mhh
{
    void batch_record(mhh_ctx* c, Batch_fn fn, const void* k, size_t size, dim3 grid, dim3 block, size_t lds)
    {
        mhh_batch* b = c->rec;
        const size_t off = align_up(b->bytes.size(), ALIGN);
        b->bytes.resize(off + size);
        std::memcpy(b->bytes.data() + off, k, size);
        b->items[c->rec_member].push_back({fn, off, size, grid, block, lds});
    }

    void batch_readback(mhh_ctx* c, const double* src, double* dst)
    {
        c->rec->readbacks.push_back({src, dst});
    }

    void batch_defer_free(mhh_ctx* c, void* ptr)
    {
        c->rec->deferred_free.push_back(ptr);
    }
}

extern "C" {

int mhh_batch_create(mhh_ctx* const* ctx, int n, mhh_batch** out)
{
    if (!ctx || !out || n < 1) return fail(MHH_EINVAL, "mhh_batch_create: bad argument");
    if (n > MHH_BATCH_MAX) return fail(MHH_EINVAL, "mhh_batch_create: more than MHH_BATCH_MAX members");
    *out = nullptr;
    for (int m = 0; m < n; ++m)
    {
        if (!ctx[m]) return fail(MHH_EINVAL, "mhh_batch_create: null context");
        if (!ctx[m]->bound) return fail(MHH_ESTATE, "mhh_batch_create: fields are not bound");
        if (ctx[m]->rec) return fail(MHH_ESTATE, "mhh_batch_create: a context is recording into another batch");
        if (ctx[m]->stream != ctx[0]->stream)
            return fail(MHH_EINVAL, "mhh_batch_create: the members of a batch share one stream");
        if (ctx[m]->device != ctx[0]->device)
            return fail(MHH_EINVAL, "mhh_batch_create: the members of a batch are on one device");
        if (ctx[m]->precision != ctx[0]->precision || ctx[m]->mixed != ctx[0]->mixed)
            return fail(MHH_EINVAL, "mhh_batch_create: the members of a batch have one precision");
        for (int q = 0; q < m; ++q)
            if (ctx[q] == ctx[m]) return fail(MHH_EINVAL, "mhh_batch_create: a context appears twice");
    }
    auto* b = new mhh_batch();
    b->ctx.assign(ctx, ctx + n);
    b->stream = ctx[0]->stream;
    b->items.resize(n);
    if (int rc = check_hip(hipEventCreateWithFlags(&b->staged, hipEventDisableTiming), "hipEventCreate"))
    {
        release(b);
        return rc;
    }
    *out = b;
    return 0;
}

int mhh_batch_begin(mhh_batch* b)
{
    if (!b) return fail(MHH_EINVAL, "mhh_batch_begin: null batch");
    if (b->recording) return fail(MHH_ESTATE, "mhh_batch_begin: the batch is recording already");
    for (mhh_ctx* c : b->ctx)
        if (c->rec) return fail(MHH_ESTATE, "mhh_batch_begin: a member records into another batch");
    for (auto& v : b->items) v.clear();
    b->bytes.clear();
    b->readbacks.clear();
    for (size_t m = 0; m < b->ctx.size(); ++m) { b->ctx[m]->rec = b; b->ctx[m]->rec_member = static_cast<int>(m); }
    b->recording = true;
    return 0;
}

int mhh_batch_end(mhh_batch* b)
{
    if (!b) return fail(MHH_EINVAL, "mhh_batch_end: null batch");
    if (!b->recording) return fail(MHH_ESTATE, "mhh_batch_end: the batch is not recording");
    stop_recording(b);
    b->recorded = 0;
    for (const auto& v : b->items) b->recorded += static_cast<int>(v.size());
    std::vector<unsigned char> blob;
    size_t rb_off = 0;
    MHH_CHECK(merge(b, blob, &rb_off));
    const int nrb = static_cast<int>(b->readbacks.size());
    const int rc = issue(b, blob, rb_off, nrb);
    // buffers the members replaced during the recording: hipFree waits for
    // the launches that use them
    for (void* ptr : b->deferred_free) (void)hipFree(ptr);
    b->deferred_free.clear();
    return rc;
}

int mhh_batch_stats(const mhh_batch* b, int* launches, int* recorded)
{
    if (!b) return fail(MHH_EINVAL, "mhh_batch_stats: null batch");
    if (launches) *launches = static_cast<int>(b->launches.size());
    if (recorded) *recorded = b->recorded;
    return 0;
}

int mhh_batch_destroy(mhh_batch* b)
{
    if (!b) return 0;
    release(b);
    return 0;
}

} // extern "C"
