// gbsw_api.cpp -- C ABI of the engine (include/gbsw.h): contexts and resident
// batches over the pipeline of gbsw_exec.cpp.
//
// Replaces the host pipeline of driver.cpp:15-243 / 245-489 (packing, chunking,
// two-stream copies, host newMin between the passes, pinned result arrays) with a
// batch uploaded once into HBM, a forward->reverse hand-off that never leaves the
// device, and status codes instead of exit() (utils.hpp:5-21).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <mutex>
#include <string>
#include <thread>
#include <vector>

#include "gbsw_internal.hpp"

using namespace gbsw;

namespace gbsw {
const char* last_error_text();
}

namespace {

// Residue order of the reference's protein table (driver.cpp:252-258 maps each
// of these letters to its index; every other byte below 91 maps to 0).
const char kAaOrder[] = "ARNDCQEGHILKMFPSTWYVBZX*";

} // namespace

struct gbsw_batch;
struct gbsw_context {
    int device = 0;
    int num_cu = 0;
    Exec ex;
    gbsw_batch* oneshot = nullptr; // gbsw_align's batch, reused across calls
    // gbsw_align_noalloc: its own streams and events, and a batch whose device
    // buffers are views of the device's static scratch (set up at creation)
    Exec nx;
    gbsw_batch* nbatch = nullptr;
    std::string nx_error;          // why the allocation-free set-up failed ("" if it did not)
    // staging of large uploads from pageable memory, shared by the context's batches
    std::mutex up_mu;
    PinnedBuffer up_ring;
    std::vector<hipEvent_t> up_events;
    ~gbsw_context()
    {
        for (hipEvent_t e : up_events) (void)hipEventDestroy(e);
    }
};

struct gbsw_batch {
    gbsw_context* ctx = nullptr;
    Job job;
    DeviceBuffer input;                       // one block: ref_off, qry_off, ref, qry (views)
    DeviceBuffer ref, ref_off, qry, qry_off, out, order;
    PinnedBuffer stage;                       // a small input block
    PinnedBuffer results;                     // of a one-shot call
    DeviceBuffer keys, keys_sorted, vals, sort_temp;
    uint8_t lut[256];
    uint8_t code_of[24]; // protein: reference code of each residue code present
    gbsw_stats stats{};
    std::vector<LaunchRec> launches; // of the last gbsw_batch_align
    JobGraph graph;
    bool one_shot = false; // a gbsw_align batch: aligned once, never worth a graph
    bool aligned = false;  // results of a gbsw_batch_align are in `out`
    // alignment paths: per-pair tables, run buffers, tightness scratch
    DeviceBuffer tb_meta, tb_temp, tb_runs, tb_dir, tb_dst, tb_tables;
    PinnedBuffer tb_host;
    std::vector<hipEvent_t> tb_events;
    ~gbsw_batch()
    {
        for (hipEvent_t e : tb_events) (void)hipEventDestroy(e);
    }
};

namespace gbsw {

// Residue table of an alphabet: protein uses the reference encoding; DNA maps each
// distinct byte present in `bytes` to its own code (raw-byte equality).  Returns
// the number of codes, or a negative status.
int build_alphabet(int32_t alphabet, const uint8_t* const* bytes, const uint64_t* lens, int nbuf, uint8_t* lut)
{
    std::memset(lut, 0xFF, 256);
    if (alphabet == GBSW_PROTEIN) {
        for (int c = 0; c < 91; ++c) {
            const char* f = std::strchr(kAaOrder, c);
            lut[c] = (uint8_t)((f && c) ? (f - kAaOrder) : 0);
        }
        for (int k = 0; k < nbuf; ++k)
            for (uint64_t i = 0; i < lens[k]; ++i)
                if (bytes[k][i] >= 91)
                    return fail(GBSW_E_RESIDUE, "protein residue byte >= 91 (the reference encoding table has 91 entries)");
        return 24;
    }
    bool seen[256] = {false};
    for (int k = 0; k < nbuf; ++k)
        for (uint64_t i = 0; i < lens[k]; ++i) seen[bytes[k][i]] = true;
    int A = 0;
    for (int c = 0; c < 256; ++c)
        if (seen[c]) lut[c] = (uint8_t)A++;
    if (A > kMaxAlpha) return fail(GBSW_E_RESIDUE, "more than 31 distinct DNA bytes in one batch");
    return std::max(A, 1);
}

// build_alphabet from the set of byte values present (bit b of mask[b / 32]),
// as scanned on the device after the upload.  Protein: only the reference codes
// that occur get a residue code (in code order), so the kernels' profiles hold
// no rows for absent residues; code_of[k] is the reference code (row of the
// caller's 24x24 matrix) of residue code k.
int alphabet_from_mask(int32_t alphabet, const uint32_t* mask, uint8_t* lut, uint8_t* code_of)
{
    auto present = [&](int c) { return (mask[c >> 5] >> (c & 31)) & 1u; };
    std::memset(lut, 0xFF, 256);
    if (alphabet == GBSW_PROTEIN) {
        for (int c = 91; c < 256; ++c)
            if (present(c))
                return fail(GBSW_E_RESIDUE, "protein residue byte >= 91 (the reference encoding table has 91 entries)");
        uint8_t enc[256];
        build_alphabet(alphabet, nullptr, nullptr, 0, enc);
        bool used[24] = {false};
        for (int c = 0; c < 91; ++c)
            if (present(c)) used[enc[c]] = true;
        uint8_t compact[24];
        int A = 0;
        for (int k = 0; k < 24; ++k)
            if (used[k]) {
                compact[k] = (uint8_t)A;
                code_of[A++] = (uint8_t)k;
            }
        if (A == 0) code_of[A++] = 0; // an empty batch: one code
        for (int c = 0; c < 91; ++c) lut[c] = used[enc[c]] ? compact[enc[c]] : 0xFF;
        return A;
    }
    int A = 0;
    for (int c = 0; c < 256; ++c)
        if (present(c)) lut[c] = (uint8_t)A++;
    if (A > kMaxAlpha) return fail(GBSW_E_RESIDUE, "more than 31 distinct DNA bytes in one batch");
    return std::max(A, 1);
}

} // namespace gbsw

namespace gbsw {

// Device block of a batch's input: byte offsets of its parts.
struct InputLayout {
    size_t ref_off, qry_off, ref, qry, total;
};
InputLayout input_layout(int64_t n, uint64_t ref_bytes, uint64_t qry_bytes)
{
    auto up = [](uint64_t x) { return (size_t)((x + 255) & ~(uint64_t)255); };
    const uint64_t offs = sizeof(uint64_t) * ((uint64_t)std::max<int64_t>(n, 1) + 1);
    InputLayout L;
    L.ref_off = 0;
    L.qry_off = L.ref_off + up(offs);
    L.ref = L.qry_off + up(offs);
    L.qry = L.ref + up(std::max<uint64_t>(ref_bytes, 16));
    L.total = L.qry + up(std::max<uint64_t>(qry_bytes, 16));
    return L;
}
void input_views(gbsw_batch* b, const InputLayout& L)
{
    uint8_t* d = b->input.as<uint8_t>();
    b->ref_off.view(d + L.ref_off, L.qry_off - L.ref_off);
    b->qry_off.view(d + L.qry_off, L.ref - L.qry_off);
    b->ref.view(d + L.ref, L.qry - L.ref);
    b->qry.view(d + L.qry, L.total - L.qry);
}

struct HostPart {
    void* dst;
    const void* src;
    size_t bytes;
};

// Copy parts to the device.  From pageable memory, large: several threads move pieces
// into a ring of pinned memory and start each one's transfer, since one thread's copy
// is slower than the link (100 MB: pinned 1.8 ms, the runtime's pageable copy 3.7 and
// more for memory it has not pinned before, this 2.4; 2, 4 and 8 MB pieces 2.7, 2.4 and
// 2.3, two to eight threads alike).  `meanwhile` runs on the calling thread, before it
// joins in.  Blocks until the sources may be reused.  False: there is no pinned memory
// for the ring, and nothing was done.
constexpr size_t kUpPiece = (size_t)4 << 20;
constexpr int kUpSlots = 6, kUpThreads = 4;
template <class F>
bool upload_large(gbsw_context* ctx, hipStream_t st, const HostPart* parts, int nparts, F&& meanwhile, hipError_t* result)
{
    std::lock_guard<std::mutex> lock(ctx->up_mu);
    hipError_t e = ctx->up_ring.reserve(kUpPiece * kUpSlots);
    if (e != hipSuccess) {
        (void)hipGetLastError();
        return false;
    }
    while (e == hipSuccess && ctx->up_events.size() < (size_t)kUpSlots) {
        hipEvent_t ev;
        e = hipEventCreateWithFlags(&ev, hipEventDisableTiming);
        if (e == hipSuccess) ctx->up_events.push_back(ev);
    }
    *result = e;
    if (e != hipSuccess) return true;
    std::vector<HostPart> pieces;
    for (int x = 0; x < nparts; ++x)
        for (size_t at = 0; at < parts[x].bytes; at += kUpPiece)
            pieces.push_back({(uint8_t*)parts[x].dst + at, (const uint8_t*)parts[x].src + at,
                              std::min(kUpPiece, parts[x].bytes - at)});
    std::atomic<size_t> next{0};
    std::atomic<int> error{(int)hipSuccess};
    std::atomic<size_t> started[kUpSlots]; // pieces whose transfer from the slot has been started
    for (auto& v : started) v.store(0);
    uint8_t* ring = ctx->up_ring.as<uint8_t>();
    auto work = [&]() {
        hipError_t me = hipSetDevice(ctx->device);
        for (;;) {
            const size_t c = next.fetch_add(1);
            if (c >= pieces.size()) break;
            const size_t slot = c % kUpSlots, turn = c / kUpSlots;
            // the slot's previous piece: its transfer started (by the thread that holds
            // it, before that thread takes another) and done
            while (started[slot].load(std::memory_order_acquire) < turn) std::this_thread::yield();
            if (me == hipSuccess && turn > 0) me = hipEventSynchronize(ctx->up_events[slot]);
            if (me == hipSuccess && error.load() == (int)hipSuccess) {
                std::memcpy(ring + slot * kUpPiece, pieces[c].src, pieces[c].bytes);
                me = hipMemcpyAsync(pieces[c].dst, ring + slot * kUpPiece, pieces[c].bytes, hipMemcpyHostToDevice, st);
                if (me == hipSuccess) me = hipEventRecord(ctx->up_events[slot], st);
            }
            if (me != hipSuccess) error.store((int)me);
            started[slot].store(turn + 1, std::memory_order_release);
        }
    };
    std::vector<std::thread> helpers;
    const int want = (int)std::min<size_t>({(size_t)kUpThreads, pieces.size(),
                                            std::max<size_t>(1, std::thread::hardware_concurrency() / 2)});
    try {
        for (int x = 1; x < want; ++x) helpers.emplace_back(work);
    } catch (...) { // fewer threads, then
    }
    meanwhile();
    work();
    for (std::thread& t : helpers) t.join();
    const hipError_t se = hipStreamSynchronize(st); // the ring is free again
    *result = error.load() != (int)hipSuccess ? (hipError_t)error.load() : se;
    return true;
}

bool is_pinned(const void* p)
{
    hipPointerAttribute_t at;
    if (hipPointerGetAttributes(&at, p) != hipSuccess) {
        (void)hipGetLastError();
        return false;
    }
    return at.type == hipMemoryTypeHost;
}

// Upload pairs into batch b (new, or one reused: its device buffers only grow),
// with ex's stream and geometry model.  `staged` (not for the allocation-free entry
// point): through pinned staging; a block of up to kUpStaged bytes is then one
// transfer, and may still be under way on ex.stream on return.  Where pinned memory is
// not to be had, the same copies go from pageable memory.
constexpr size_t kUpStaged = (size_t)1 << 20, kUpLarge = (size_t)8 << 20;
// Residues whose set of byte values the host finds (about a byte per cycle: 20 us at
// most); more are scanned on the device, which costs a launch and a wait (about 30 us).
constexpr uint64_t kHostScan = 65536;
static int batch_fill(gbsw_batch* b, gbsw_context* ctx, Exec& ex, bool staged, int32_t alphabet, int64_t n,
                      const char* ref, const uint64_t* ref_off, const char* query, const uint64_t* query_off)
{
    if (!ctx || n < 0 || (n > 0 && (!ref_off || !query_off)))
        return fail(GBSW_E_ARGUMENT, "null argument or negative pair count");
    if (alphabet != GBSW_DNA && alphabet != GBSW_PROTEIN) return fail(GBSW_E_ARGUMENT, "unknown alphabet");
    if (n > (int64_t)0x7FFFFFFF) return fail(GBSW_E_RANGE, "more than 2^31-1 pairs in one batch");
    const uint64_t ref_bytes = n ? ref_off[n] - ref_off[0] : 0;
    const uint64_t qry_bytes = n ? query_off[n] - query_off[0] : 0;
    if ((ref_bytes && !ref) || (qry_bytes && !query)) return fail(GBSW_E_ARGUMENT, "sequence buffer is null");
    GBSW_HIP_TRY(hipSetDevice(ctx->device));

    b->ctx = ctx;
    b->job = Job{};
    b->graph.reset();
    b->aligned = false;
    b->stats = gbsw_stats{};
    b->launches.clear();
    Job& job = b->job;
    job.alphabet = alphabet;
    job.n = n;
    bool valid = true;
    for (int64_t p = 0; p < n; ++p) { // (a decreasing offset gives a huge length)
        const uint64_t lr = ref_off[p + 1] - ref_off[p], lq = query_off[p + 1] - query_off[p];
        valid &= (lr <= 65000) & (lq <= 65000);
    }
    for (int64_t p = 0; !valid && p < n; ++p) {
        if (ref_off[p + 1] < ref_off[p] || query_off[p + 1] < query_off[p])
            return fail(GBSW_E_ARGUMENT, "offsets must be non-decreasing");
        if (ref_off[p + 1] - ref_off[p] > 65000 || query_off[p + 1] - query_off[p] > 65000)
            return fail(GBSW_E_RANGE, "sequences longer than 65000 residues are not supported");
    }
    const uint8_t* rp = (const uint8_t*)ref + (n ? ref_off[0] : 0);
    const uint8_t* qp = (const uint8_t*)query + (n ? query_off[0] : 0);
    job.lut_host = b->lut;
    job.kmodel = ex.kmodel;
    size_t sort_bytes = 0;
    int rc = sort_scratch_bytes(n, &sort_bytes);
    if (rc) return rc;
    const size_t np = (size_t)std::max<int64_t>(n, 1);
    const InputLayout L = input_layout(n, ref_bytes, qry_bytes);
    hipStream_t st = ex.stream;
    hipError_t e = b->input.reserve(L.total);
    if (e == hipSuccess) input_views(b, L);
    if (e == hipSuccess) e = b->out.reserve(sizeof(int32_t) * 5 * np);
    if (e == hipSuccess) e = b->keys.reserve(std::max<size_t>(4 * np, 32));
    if (e == hipSuccess) e = b->keys_sorted.reserve(4 * np);
    if (e == hipSuccess) e = b->vals.reserve(4 * np);
    if (e == hipSuccess) e = b->order.reserve(4 * np);
    if (e == hipSuccess) e = b->sort_temp.reserve(sort_bytes);
    const size_t offs_bytes = L.ref - L.ref_off, masks_bytes = 32 * kPresenceBlocks;
    bool one_block = staged && L.total <= kUpStaged;
    bool pinned_offs = staged && b->one_shot; // (kept for the next call)
    bool host_scan = ref_bytes + qry_bytes <= kHostScan;
    const size_t masks_at = one_block ? L.total : pinned_offs ? offs_bytes : 0;
    if (staged && b->stage.reserve(masks_at + masks_bytes) != hipSuccess) {
        (void)hipGetLastError();
        staged = one_block = pinned_offs = false;
        host_scan = true; // (nowhere for the device's masks)
    }
    std::vector<uint64_t> offs;
    uint8_t* h = b->stage.as<uint8_t>();
    if (e == hipSuccess && !one_block && !pinned_offs) {
        offs.resize(offs_bytes / sizeof(uint64_t));
        h = (uint8_t*)offs.data();
    }
    job.buckets.reserve(kClasses); // (no allocation beside running threads)
    job.fine.reserve(kFineClasses);
    // what takes a pass over the pairs: offsets from 0, classes
    auto pairs_pass = [&]() {
        uint64_t *ro = (uint64_t*)(h + L.ref_off), *qo = (uint64_t*)(h + L.qry_off);
        Bucket classes[kClasses], fine[kFineClasses];
        ro[0] = qo[0] = 0;
        for (int64_t p = 0; p < n; ++p) {
            const uint64_t lr = ref_off[p + 1] - ref_off[p], lq = query_off[p + 1] - query_off[p];
            ro[p + 1] = ro[p] + lr;
            qo[p + 1] = qo[p] + lq;
            const int32_t rows = (int32_t)std::max(lr, lq), cols = (int32_t)std::min(lr, lq);
            job.max_rows = std::max(job.max_rows, rows);
            job.max_cols = std::max(job.max_cols, cols);
            job.cells += (int64_t)(lr * lq);
            fine[fine_class(cols)].add(cols, rows);
        }
        for (const Bucket& f : fine)
            if (f.count) classes[length_class(f.max_cols)].add(f);
        place_buckets(job.buckets, classes, kClasses);
        place_buckets(job.fine, fine, kFineClasses);
    };
    if (e == hipSuccess) e = hipMemsetAsync(b->out.ptr, 0, sizeof(int32_t) * 5 * np, st);
    uint8_t* dev = b->input.as<uint8_t>();
    const HostPart parts[2] = {{dev + L.ref, rp, ref_bytes}, {dev + L.qry, qp, qry_bytes}};
    if (e == hipSuccess) {
        if (one_block) {
            pairs_pass();
            if (ref_bytes) std::memcpy(h + L.ref, rp, ref_bytes);
            if (qry_bytes) std::memcpy(h + L.qry, qp, qry_bytes);
            e = hipMemcpyAsync(dev, h, L.qry + qry_bytes, hipMemcpyHostToDevice, st);
        } else {
            if (!(staged && L.total >= kUpLarge && !(ref_bytes && is_pinned(rp)) && !(qry_bytes && is_pinned(qp)) &&
                  upload_large(ctx, st, parts, 2, pairs_pass, &e))) {
                for (const HostPart& x : parts)
                    if (e == hipSuccess && x.bytes) e = hipMemcpyAsync(x.dst, x.src, x.bytes, hipMemcpyHostToDevice, st);
                pairs_pass();
            }
            if (e == hipSuccess) e = hipMemcpyAsync(dev, h, offs_bytes, hipMemcpyHostToDevice, st);
            if (e == hipSuccess) e = hipStreamSynchronize(st);
        }
    }
    // The residue codes need the set of byte values in the batch (every distinct
    // DNA byte is a code; protein bytes must be < 91).
    uint32_t seen[8] = {0};
    if (e == hipSuccess && host_scan) {
        uint8_t has[256] = {0};
        for (uint64_t x = 0; x < ref_bytes; ++x) has[rp[x]] = 1;
        for (uint64_t x = 0; x < qry_bytes; ++x) has[qp[x]] = 1;
        for (int x = 0; x < 256; ++x) seen[x >> 5] |= (uint32_t)has[x] << (x & 31);
    } else if (e == hipSuccess) {
        // one mask per workgroup, in pinned memory
        uint32_t* masks = (uint32_t*)(staged ? b->stage.as<uint8_t>() + masks_at : ex.tables_host.as<uint8_t>());
        std::memset(masks, 0, masks_bytes);
        e = byte_presence(b->ref.as<uint8_t>(), ref_bytes, b->qry.as<uint8_t>(), qry_bytes, masks, st);
        if (e == hipSuccess) e = hipStreamSynchronize(st);
        for (int x = 0; x < 8 * kPresenceBlocks; ++x) seen[x & 7] |= masks[x];
    }
    if (e == hipSuccess && one_block && !b->one_shot) e = hipStreamSynchronize(st);
    if (e != hipSuccess) {
        (void)hipStreamSynchronize(st);
        return fail(e == hipErrorOutOfMemory ? GBSW_E_MEMORY : GBSW_E_DEVICE,
                    std::string("batch upload: ") + hipGetErrorString(e));
    }
    {
        const int A = alphabet_from_mask(alphabet, seen, b->lut, b->code_of);
        if (A < 0) {
            (void)hipStreamSynchronize(st);
            return A;
        }
        job.alpha = A;
        job.code_of = alphabet == GBSW_PROTEIN ? b->code_of : nullptr;
    }
    job.ref = b->ref.as<uint8_t>();
    job.qry = b->qry.as<uint8_t>();
    job.ref_off = b->ref_off.as<uint64_t>();
    job.qry_off = b->qry_off.as<uint64_t>();
    job.out = b->out.as<int32_t>();
    job.keys = b->keys.as<uint32_t>();
    job.keys_sorted = b->keys_sorted.as<uint32_t>();
    job.vals = b->vals.as<int32_t>();
    job.order = b->order.as<int32_t>();
    job.sort_temp = b->sort_temp.ptr;
    job.sort_temp_bytes = sort_bytes;
    b->stats.cells = job.cells;
    return GBSW_OK;
}

} // namespace gbsw

namespace {

// Both passes of every pair of batch b on ex's streams, blocking; the results also to
// `results` (pinned, 5 n) if given.
int batch_align_on(gbsw_batch* b, Exec& ex, const gbsw_scoring* sc, int32_t mode, int32_t* results = nullptr)
{
    if (mode != GBSW_PLAIN && mode != GBSW_BATCHED) return fail(GBSW_E_ARGUMENT, "unknown mode");
    GBSW_HIP_TRY(hipSetDevice(b->ctx->device));
    b->stats = gbsw_stats{};
    b->stats.cells = b->job.cells;
    b->launches.clear();
    // a resident batch captures its work into a graph; gbsw_align's one-off
    // batch does not
    b->job.graph = b->one_shot ? nullptr : &b->graph;
    int rc = enqueue_job(ex, b->job, sc, mode);
    if (rc) {
        (void)hipStreamSynchronize(ex.stream);
        return rc;
    }
    const size_t bytes = sizeof(int32_t) * 5 * (size_t)b->job.n;
    if (results && bytes) GBSW_HIP_TRY(hipMemcpyAsync(results, b->out.ptr, bytes, hipMemcpyDeviceToHost, ex.stream));
    double ms = 0.0;
    rc = complete_job(ex, b->job, sc, &ms);
    if (results && bytes) {
        if (rc == GBSW_OK && ex.late_results) // (aligned again: recomputed pairs)
            GBSW_HIP_TRY(hipMemcpyAsync(results, b->out.ptr, bytes, hipMemcpyDeviceToHost, ex.stream));
        GBSW_HIP_TRY(hipStreamSynchronize(ex.stream));
    }
    b->launches = ex.launches;
    b->stats.device_ms = ms;
    b->stats.launches = (int32_t)b->launches.size();
    b->stats.buckets = mode == GBSW_PLAIN ? 1 : (int32_t)b->job.buckets.size();
    b->stats.graph = ex.graph_state;
    for (const LaunchRec& L : b->launches) b->stats.main_kernel_ms = std::max(b->stats.main_kernel_ms, L.ms);
    b->aligned = rc == GBSW_OK;
    return rc;
}

// Five result arrays of n that are one block.
bool back_to_back(int32_t* const* dst, size_t n)
{
    for (int f = 0; f < 5; ++f)
        if (!dst[0] || dst[f] != dst[0] + f * n) return false;
    return true;
}

// Carve the device scratch of gbsw_align_noalloc for one call of n pairs:
// tables, then the batch's arrays, then the redo list; what is left holds the
// strip-boundary rows (7/8) and the split form's bookkeeping (1/8).  Every
// buffer becomes a view (never grown, never freed).
int noalloc_carve(gbsw_context* ctx, int64_t n, uint64_t ref_bytes, uint64_t qry_bytes)
{
    uint8_t* base = (uint8_t*)noalloc_scratch(ctx->device);
    if (!base || !ctx->nx.stream)
        return fail(GBSW_E_DEVICE, "the allocation-free scratch is not set up on this device: " + ctx->nx_error);
    size_t sort_bytes = 0;
    if (int rc = sort_scratch_bytes(n, &sort_bytes)) return rc;
    const size_t np = (size_t)std::max<int64_t>(n, 1);
    size_t at = 0;
    auto take = [&](DeviceBuffer& d, size_t bytes) {
        const size_t p = at;
        at = (at + bytes + 255) & ~(size_t)255;
        if (at <= kNoallocScratchBytes) d.view(base + p, bytes);
    };
    Exec& x = ctx->nx;
    gbsw_batch* b = ctx->nbatch;
    take(x.status, sizeof(int32_t) * kStatusWords);
    take(x.queue, sizeof(uint32_t) * kXcds * 64);
    take(x.sub, sizeof(int16_t) * 1024);
    take(x.lut, 256);
    take(x.colmax, sizeof(int16_t) * 32);
    take(b->input, input_layout(n, ref_bytes, qry_bytes).total);
    take(b->out, sizeof(int32_t) * 5 * np);
    take(b->keys, std::max<size_t>(4 * np, 32));
    take(b->keys_sorted, 4 * np);
    take(b->vals, 4 * np);
    take(b->order, 4 * np);
    take(b->sort_temp, sort_bytes);
    take(x.redo, sizeof(int32_t) * np);
    // at least 1 MiB for boundary rows (a wide pair on one workgroup)
    constexpr size_t kMinRest = (size_t)1 << 20;
    if (at + kMinRest > kNoallocScratchBytes)
        return fail(GBSW_E_RANGE, "gbsw_align_noalloc: " + std::to_string(n) + " pairs of " +
                                      std::to_string(ref_bytes + qry_bytes) + " residue bytes need " +
                                      std::to_string(at + kMinRest) + " bytes of scratch; the limit is " +
                                      std::to_string(kNoallocScratchBytes));
    const size_t rest = kNoallocScratchBytes - at;
    const size_t split_bytes = (rest / 8) & ~(size_t)255;
    take(x.split_buf, split_bytes);
    take(x.bnd, kNoallocScratchBytes - at);
    return GBSW_OK;
}

} // namespace

extern "C" {

const char* gbsw_last_error(void) { return gbsw::last_error_text(); }

const char* gbsw_version(void) { return "gbsw-mi355x 0.2 (gfx950, packed int16 wavefront)"; }

int gbsw_device_memory(int32_t device, uint64_t* bytes)
{
    if (!bytes) return fail(GBSW_E_ARGUMENT, "bytes is null");
    hipDeviceProp_t prop;
    GBSW_HIP_TRY(hipGetDeviceProperties(&prop, device));
    *bytes = (uint64_t)prop.totalGlobalMem;
    return GBSW_OK;
}

int gbsw_context_create(int32_t device, gbsw_context** out)
{
    if (!out) return fail(GBSW_E_ARGUMENT, "out is null");
    *out = nullptr;
    int count = 0;
    GBSW_HIP_TRY(hipGetDeviceCount(&count));
    if (device < 0 || device >= count) return fail(GBSW_E_ARGUMENT, "no such device");
    GBSW_HIP_TRY(hipSetDevice(device));
    hipDeviceProp_t prop;
    GBSW_HIP_TRY(hipGetDeviceProperties(&prop, device));
    gbsw_context* ctx = new gbsw_context();
    ctx->device = device;
    ctx->num_cu = prop.multiProcessorCount;
    const int rc = ctx->ex.init(device, ctx->num_cu);
    if (rc) {
        ctx->ex.destroy();
        delete ctx;
        return rc;
    }
    // set-up of the allocation-free entry point: the device address of this
    // device's scratch, its streams and events; a failure here only disables
    // gbsw_align_noalloc (which then reports it)
    int nrc = noalloc_setup(device);
    if (!nrc) nrc = ctx->nx.init_views(device, ctx->num_cu);
    if (nrc) ctx->nx_error = gbsw_last_error();
    ctx->nbatch = new gbsw_batch();
    ctx->nbatch->one_shot = true;
    set_error("");
    *out = ctx;
    return GBSW_OK;
}

int gbsw_context_set_option(gbsw_context* ctx, int32_t option, int64_t value)
{
    if (!ctx) return fail(GBSW_E_ARGUMENT, "context is null");
    switch (option) {
    case GBSW_OPT_STREAMS:
        if (value < 1 || value > kAuxStreams + 1) return fail(GBSW_E_ARGUMENT, "streams must be 1..8");
        if (int rc = ctx->ex.ensure_streams((int)value)) return rc;
        ctx->ex.streams = (int)value;
        return GBSW_OK;
    case GBSW_OPT_F16:
        if (value != 0 && value != 1) return fail(GBSW_E_ARGUMENT, "f16 option is 0 or 1");
        ctx->ex.f16 = value != 0;
        return GBSW_OK;
    case GBSW_OPT_GRAPHS:
        if (value != 0 && value != 1) return fail(GBSW_E_ARGUMENT, "graphs option is 0 or 1");
        ctx->ex.graphs = value != 0;
        return GBSW_OK;
    case GBSW_OPT_SPLIT:
        if (value != 0 && value != 1) return fail(GBSW_E_ARGUMENT, "split option is 0 or 1");
        ctx->ex.split = value != 0;
        return GBSW_OK;
    case GBSW_OPT_GEOMETRY:
        if (value < 0 || value >= kGeometryModels) return fail(GBSW_E_ARGUMENT, "geometry model is 0..5");
        ctx->ex.kmodel = (int)value;
        return GBSW_OK;
    default:
        return fail(GBSW_E_ARGUMENT, "unknown option");
    }
}

int gbsw_context_destroy(gbsw_context* ctx)
{
    if (!ctx) return GBSW_OK;
    (void)hipSetDevice(ctx->device);
    delete ctx->oneshot;
    delete ctx->nbatch;
    ctx->nx.destroy();
    ctx->ex.destroy();
    delete ctx;
    return GBSW_OK;
}

int gbsw_batch_create(gbsw_context* ctx, int32_t alphabet, int64_t n, const char* ref,
                      const uint64_t* ref_off, const char* query, const uint64_t* query_off,
                      gbsw_batch** out)
{
    if (!out) return fail(GBSW_E_ARGUMENT, "out is null");
    *out = nullptr;
    gbsw_batch* b = new gbsw_batch();
    const int rc = ctx ? batch_fill(b, ctx, ctx->ex, true, alphabet, n, ref, ref_off, query, query_off)
                       : fail(GBSW_E_ARGUMENT, "context is null");
    if (rc) {
        const std::string err = gbsw_last_error();
        delete b;
        set_error(err);
        return rc;
    }
    *out = b;
    return GBSW_OK;
}

int gbsw_batch_destroy(gbsw_batch* b)
{
    if (!b) return GBSW_OK;
    (void)hipSetDevice(b->ctx->device);
    delete b;
    return GBSW_OK;
}

int gbsw_batch_align(gbsw_batch* b, const gbsw_scoring* sc, int32_t mode)
{
    if (!b || !sc) return fail(GBSW_E_ARGUMENT, "null argument");
    return batch_align_on(b, b->ctx->ex, sc, mode);
}

int gbsw_batch_traceback(gbsw_batch* b, const gbsw_scoring* sc, int64_t capacity, uint32_t* cigar,
                         int64_t* cigar_offsets, int32_t* path_score, double* device_ms)
{
    if (!b || !sc || !cigar_offsets) return fail(GBSW_E_ARGUMENT, "null argument");
    if (capacity < 0 || (capacity > 0 && !cigar)) return fail(GBSW_E_ARGUMENT, "bad cigar buffer");
    if (!b->aligned) return fail(GBSW_E_ARGUMENT, "the batch has no alignment results (gbsw_batch_align first)");
    if (sc->gap_open > sc->gap_extend)
        return fail(GBSW_E_SCORING, "alignment paths need gap_open <= gap_extend (a gap run is one gap)");
    gbsw_context* ctx = b->ctx;
    GBSW_HIP_TRY(hipSetDevice(ctx->device));
    const Job& job = b->job;
    std::vector<int16_t> sub;
    int32_t max_sub = 0;
    bool p8 = false;
    if (int rc = prepare_scoring(job, sc, sub, &max_sub, &p8)) return rc;
    const int64_t n = job.n;
    cigar_offsets[0] = 0;
    if (n == 0) {
        if (device_ms) *device_ms = 0.0;
        return GBSW_OK;
    }
    hipStream_t st = ctx->ex.stream;
    // the int32 cells hold (rows + columns) x the largest |score| below 2^28
    int64_t big = std::max(std::abs((int64_t)sc->gap_open), std::abs((int64_t)sc->gap_extend));
    int32_t min_sub = 0;
    for (int16_t v : sub) {
        big = std::max<int64_t>(big, std::abs((int32_t)v));
        min_sub = std::min<int32_t>(min_sub, v);
    }
    const int64_t go = -(int64_t)sc->gap_open, ge = -(int64_t)sc->gap_extend;
    // device tables: run capacities and their offsets, offsets of the result (n + 1
    // int64 each); runs per pair (n + 1), path scores, order and its keys (n int32
    // each); counts
    const int64_t n1 = n + 1;
    GBSW_HIP_TRY(b->tb_meta.reserve(sizeof(int64_t) * (size_t)(3 * n1) + sizeof(int32_t) * (size_t)(n1 + 5 * n) +
                                    sizeof(TbCounts) + 64));
    int64_t* d_cap = b->tb_meta.as<int64_t>();
    int64_t* d_cap_off = d_cap + n1;
    int64_t* d_dst_off = d_cap_off + n1;
    int32_t* d_nruns = (int32_t*)(d_dst_off + n1);
    int32_t* d_score = d_nruns + n1;
    int32_t* d_vals = d_score + n;
    int32_t* d_order = d_vals + n;
    uint32_t* d_keys = (uint32_t*)(d_order + n);
    uint32_t* d_keys_sorted = d_keys + n;
    TbCounts* d_counts = (TbCounts*)(d_keys_sorted + n);
    size_t sort_bytes = 0, scan_bytes = 0, scan32_bytes = 0;
    GBSW_HIP_TRY(sort_pairs(nullptr, sort_bytes, d_keys, d_keys_sorted, d_vals, d_order, (int)n, kTbKeyBits, st));
    GBSW_HIP_TRY(tb_scan(nullptr, scan_bytes, d_cap, d_cap_off, n1, st));
    GBSW_HIP_TRY(tb_scan(nullptr, scan32_bytes, d_nruns, d_dst_off, n1, st));
    size_t temp_bytes = std::max({sort_bytes, scan_bytes, scan32_bytes, (size_t)16});
    GBSW_HIP_TRY(b->tb_temp.reserve(temp_bytes));
    GBSW_HIP_TRY(b->tb_tables.reserve(256 + sizeof(int16_t) * sub.size()));
    // pinned host memory, kept with the batch: the tables to upload and the counts, later
    // the result's offsets and the path scores
    const size_t tables = 256 + sizeof(int16_t) * sub.size();
    const size_t host_words = sizeof(int64_t) * (size_t)n1 + sizeof(int32_t) * (size_t)n;
    GBSW_HIP_TRY(b->tb_host.reserve(std::max(host_words, 4096 + sizeof(TbCounts) + sizeof(int64_t))));
    uint8_t* h_tables = b->tb_host.as<uint8_t>();
    TbCounts& counts = *(TbCounts*)(h_tables + 4096);
    int64_t& cap_total = *(int64_t*)(h_tables + 4096 + sizeof(TbCounts));
    static_assert(sizeof(TbCounts) % 8 == 0, "cap_total is aligned");
    if (tables > 4096) return fail(GBSW_E_INTERNAL, "residue alphabet too large");
    std::memcpy(h_tables, b->lut, 256);
    std::memcpy(h_tables + 256, sub.data(), sizeof(int16_t) * sub.size());
    uint8_t* d_lut = b->tb_tables.as<uint8_t>();
    TbArgs a{};
    a.ref = b->ref.as<uint8_t>();
    a.qry = b->qry.as<uint8_t>();
    a.ref_off = b->ref_off.as<uint64_t>();
    a.qry_off = b->qry_off.as<uint64_t>();
    a.out = b->out.as<int32_t>();
    a.n = n;
    a.lut = d_lut;
    a.sub = (const int16_t*)(d_lut + 256);
    a.alpha = job.alpha;
    a.gap_open = sc->gap_open;
    a.gap_extend = sc->gap_extend;
    a.max_sub = max_sub;
    a.order = d_order;
    a.cap_off = d_cap_off;
    a.nruns = d_nruns;
    a.path_score = d_score;
    Exec& ex = ctx->ex;
    constexpr int kTbStreams = 4;
    if (int rc = ex.ensure_streams(kTbStreams)) return rc;
    GBSW_HIP_TRY(hipEventRecord(ex.ev_start, st));
    GBSW_HIP_TRY(hipMemcpyAsync(d_lut, h_tables, tables, hipMemcpyHostToDevice, st));
    GBSW_HIP_TRY(hipMemsetAsync(d_counts, 0, sizeof(TbCounts), st));
    GBSW_HIP_TRY(tb_keys(a, d_keys, d_vals, d_cap, d_counts, st));
    GBSW_HIP_TRY(hipMemcpyAsync(&counts, d_counts, sizeof(TbCounts), hipMemcpyDeviceToHost, st));
    GBSW_HIP_TRY(tb_scan(b->tb_temp.ptr, temp_bytes, d_cap, d_cap_off, n1, st));
    GBSW_HIP_TRY(hipMemcpyAsync(&cap_total, d_cap_off + n, sizeof(int64_t), hipMemcpyDeviceToHost, st));
    GBSW_HIP_TRY(sort_pairs(b->tb_temp.ptr, temp_bytes, d_keys, d_keys_sorted, d_vals, d_order, (int)n, kTbKeyBits, st));
    GBSW_HIP_TRY(hipStreamSynchronize(st));
    if (counts.bad) return fail(GBSW_E_INTERNAL, "a pair with a positive score has an empty rectangle");
    if ((int64_t)counts.span * big >= ((int64_t)1 << 28))
        return fail(GBSW_E_RANGE, "path scores may exceed the int32 cells' range");
    GBSW_HIP_TRY(b->tb_runs.reserve(sizeof(uint32_t) * (size_t)std::max<int64_t>(1, cap_total)));
    a.runs = b->tb_runs.as<uint32_t>();

    // Substitution scores, biased by o + g: bytes of four times that (in registers for up
    // to four codes) where they fit, else words.
    const int64_t lo = min_sub + go + ge, hi = max_sub + go + ge;
    const int form = lo >= 0 && hi <= 63 ? (job.alpha <= kRegAlpha ? kProfRegs : kProfBytes) : kProfWords;
    const bool words16 = lo >= -8000 && hi <= 8000;
    // no 16-bit value is negative: H >= -2 o (all of one sequence, then all of the
    // other, against gaps), Ho >= H - o, and a diagonal sum adds at least min_sub to Ho
    const int64_t base = 1 + std::max(3 * go, 2 * go - min_sub);
    a.base = (int32_t)std::min<int64_t>(base, 1 << 28);
    // cells of a class: the narrowest that holds its largest value bound
    auto cells_of = [&](int64_t value) {
        const int64_t top = value + base + 1;
        return !words16 || top >= kTbTop16Wide ? kTbCells32 : top >= kTbTop16 ? kTbCells16Wide : kTbCells16;
    };

    // Launches: stretches of classes, largest first, of one cell type, one group width
    // and regions that do not differ much, in turn on four streams with a quarter of the
    // scratch each: the tail of one runs beside the next.  All scratch: at most 12 GiB, or a
    // third of the free device memory when less (but room for one pair).
    // (12 waves per CU: 8, 12 and 16 took 4.84, 4.43 and 4.38 ms for 300k pairs of the DNA
    // mix, 15.5, 14.3 and 14.1 for a million, and scratch is per wave.  One stream less
    // than needed is worse: on two the 300k pairs took 5.4 ms.)
    struct Launch {
        int cells, G, kmax, grid, lds;
        int64_t p0, count, region;
    };
    size_t free_bytes = 0, total_bytes = 0;
    if (hipMemGetInfo(&free_bytes, &total_bytes) != hipSuccess) {
        (void)hipGetLastError();
        free_bytes = (size_t)24 << 30;
    }
    free_bytes += b->tb_dir.bytes;
    const int64_t part_max =
        std::max<int64_t>((int64_t)64 << 20, std::min<int64_t>((int64_t)3 << 30, (int64_t)(free_bytes / 12)));
    // 64 lanes per two pairs take more steps in all than 16 per two (a stripe's
    // anti-diagonals are longer) but a quarter of the time of each: the classes from
    // `wide_from` on use them, where that makes the sum per SIMD or the longest set,
    // whichever is larger, least.  A lone wave issues at about half a SIMD's rate.
    int wide_from = kTbAreas;
    {
        const double simds = 4.0 * ctx->num_cu;
        double best = 1e300, work64 = 0.0, work16 = 0.0, long64 = 0.0;
        std::vector<double> w16(kTbAreas), w64(kTbAreas), l16(kTbAreas + 1, 0.0), l64(kTbAreas);
        for (int c = 0; c < kTbAreas; ++c) {
            const double k = counts.pairs[c];
            const int kmax = tb_kmax(cells_of(counts.value[c]), form);
            // (every set as its class's largest rows and columns)
            const double s16 = k ? tb_set_cost((int)counts.rows[c], (int)counts.cols[c], 16, kmax) : 0.0;
            const double s64 = k ? tb_set_cost((int)counts.rows[c], (int)counts.cols[c], 64, kmax) : 0.0;
            w16[c] = std::ceil(k / 8) * s16;
            w64[c] = std::ceil(k / 2) * s64;
            l16[c + 1] = std::max(l16[c], s16);
            l64[c] = s64;
            work16 += w16[c];
        }
        for (int x = kTbAreas; x >= 0; --x) { // classes x and up with 64 lanes
            if (x < kTbAreas) {
                work64 += w64[x];
                work16 -= w16[x];
                long64 = std::max(long64, l64[x]);
            }
            const double t = std::max((work64 + work16) / simds, 2.0 * std::max(long64, l16[x])) +
                             0.25 * (work64 + work16) / simds;
            if (t < best * 0.999) {
                best = t;
                wide_from = x;
            }
        }
    }
    std::vector<Launch> launches;
    int64_t part_bytes[kTbStreams] = {};
    {
        int64_t at = 0;
        uint32_t top_value[kTbAreas]; // largest bound of a class and those below it
        for (int c = 0; c < kTbAreas; ++c) top_value[c] = std::max(counts.value[c], c ? top_value[c - 1] : 0u);
        for (int c = kTbAreas - 1; c >= 0;) {
            if (!counts.pairs[c]) {
                --c;
                continue;
            }
            Launch L{};
            L.cells = cells_of(top_value[c]);
            L.G = c >= wide_from ? 64 : 16;
            L.kmax = tb_kmax(L.cells, form);
            L.p0 = at;
            L.lds = tb_lds_bytes(L.cells, L.G, form, L.kmax, job.alpha);
            const int64_t slots =
                (int64_t)ctx->num_cu * std::min(12, tb_occupancy(L.cells, L.G, form, L.lds));
            const int np = 2 * (64 / L.G);
            auto region_of = [&](int x) { // room for a set of the class, if that is not out of proportion
                const int64_t one = (int64_t)counts.scratch[L.G == 64][x] << 8;
                const int64_t set =
                    tb_region_bytes((int)counts.rows[x], (int)counts.cols[x], L.G, L.kmax, L.cells, np / 2);
                return (std::max(one, std::min({set, np * one, part_max})) + 255) & ~(int64_t)255;
            };
            const int64_t first = region_of(c);
            const bool last = launches.size() + 1 == kTbLaunches;
            for (; c >= 0; --c) {
                if (!counts.pairs[c]) continue;
                const int64_t r = region_of(c);
                if (L.count && !last && (cells_of(top_value[c]) != L.cells || (c >= wide_from ? 64 : 16) != L.G ||
                                         (2 * r < first && first * slots > part_max / 4)))
                    break;
                L.count += counts.pairs[c];
                L.region = std::max(L.region, r);
            }
            at += L.count;
            const int64_t sets = (L.count + np - 1) / np;
            L.grid = (int)std::max<int64_t>(1, std::min({slots, sets, part_max / L.region}));
            int64_t& part = part_bytes[launches.size() % kTbStreams];
            part = std::max(part, L.region * L.grid);
            launches.push_back(L);
        }
    }
    int64_t part_at[kTbStreams + 1] = {};
    for (int x = 0; x < kTbStreams; ++x) part_at[x + 1] = part_at[x] + part_bytes[x];
    GBSW_HIP_TRY(b->tb_dir.reserve((size_t)std::max<int64_t>(256, part_at[kTbStreams])));
    while (b->tb_events.size() < kTbStreams) {
        hipEvent_t e;
        GBSW_HIP_TRY(hipEventCreateWithFlags(&e, hipEventDisableTiming));
        b->tb_events.push_back(e);
    }
    const int streams = (int)std::min<size_t>(launches.size(), kTbStreams);
    if (streams > 1) GBSW_HIP_TRY(hipEventRecord(b->tb_events[0], st));
    for (int x = 1; x < streams; ++x) GBSW_HIP_TRY(hipStreamWaitEvent(ex.aux[x - 1], b->tb_events[0], 0));
    for (size_t c = 0; c < launches.size(); ++c) {
        const Launch& L = launches[c];
        const int x = (int)(c % kTbStreams);
        a.p0 = L.p0;
        a.count = L.count;
        a.kmax = L.kmax;
        a.region_bytes = L.region;
        a.queue = d_counts->queue + c;
        a.dir = b->tb_dir.as<uint8_t>() + part_at[x];
        GBSW_HIP_TRY(tb_launch(a, L.cells, L.G, form, L.grid, L.lds, x ? ex.aux[x - 1] : st));
    }
    for (int x = 1; x < streams; ++x) {
        GBSW_HIP_TRY(hipEventRecord(b->tb_events[x], ex.aux[x - 1]));
        GBSW_HIP_TRY(hipStreamWaitEvent(st, b->tb_events[x], 0));
    }
    GBSW_HIP_TRY(tb_scan(b->tb_temp.ptr, temp_bytes, d_nruns, d_dst_off, n1, st));
    GBSW_HIP_TRY(hipEventRecord(ex.ev_stop, st)); // device_ms: the path kernels
    int64_t* h_off = b->tb_host.as<int64_t>();
    int32_t* h_score = (int32_t*)(h_off + n1);
    GBSW_HIP_TRY(hipMemcpyAsync(h_off, d_dst_off, sizeof(int64_t) * (size_t)n1, hipMemcpyDeviceToHost, st));
    if (path_score)
        GBSW_HIP_TRY(hipMemcpyAsync(h_score, d_score, sizeof(int32_t) * (size_t)n, hipMemcpyDeviceToHost, st));
    GBSW_HIP_TRY(hipStreamSynchronize(st));
    std::memcpy(cigar_offsets, h_off, sizeof(int64_t) * (size_t)n1);
    if (path_score) std::memcpy(path_score, h_score, sizeof(int32_t) * (size_t)n);
    const int64_t total = cigar_offsets[n];
    if (device_ms) {
        float ms = 0.f;
        GBSW_HIP_TRY(hipEventElapsedTime(&ms, ex.ev_start, ex.ev_stop));
        *device_ms = ms;
    }
    if (total > capacity) {
        return fail(GBSW_E_RANGE, "cigar capacity " + std::to_string(capacity) + " < " + std::to_string(total) +
                                      " words needed (cigar_offsets holds the layout)");
    }
    GBSW_HIP_TRY(b->tb_dst.reserve(sizeof(uint32_t) * (size_t)std::max<int64_t>(1, total)));
    GBSW_HIP_TRY(tb_compact(a.runs, d_cap_off, d_nruns, d_dst_off, b->tb_dst.as<uint32_t>(), n, st));
    if (total)
        GBSW_HIP_TRY(hipMemcpyAsync(cigar, b->tb_dst.ptr, sizeof(uint32_t) * (size_t)total, hipMemcpyDeviceToHost, st));
    GBSW_HIP_TRY(hipStreamSynchronize(st));
    return GBSW_OK;
}

int gbsw_batch_results(gbsw_batch* b, int32_t* score, int32_t* ref_begin, int32_t* ref_end,
                       int32_t* query_begin, int32_t* query_end)
{
    if (!b) return fail(GBSW_E_ARGUMENT, "batch is null");
    GBSW_HIP_TRY(hipSetDevice(b->ctx->device));
    int32_t* dst[5] = {score, ref_begin, ref_end, query_begin, query_end};
    const size_t n = (size_t)b->job.n;
    if (n && back_to_back(dst, n)) {
        GBSW_HIP_TRY(hipMemcpy(dst[0], b->out.ptr, sizeof(int32_t) * 5 * n, hipMemcpyDeviceToHost));
        return GBSW_OK;
    }
    for (int f = 0; f < 5; ++f)
        if (dst[f] && n)
            GBSW_HIP_TRY(hipMemcpy(dst[f], b->out.as<int32_t>() + (size_t)f * n, sizeof(int32_t) * n,
                                   hipMemcpyDeviceToHost));
    return GBSW_OK;
}

int gbsw_batch_device_results(gbsw_batch* b, const int32_t** d_out)
{
    if (!b || !d_out) return fail(GBSW_E_ARGUMENT, "null argument");
    *d_out = b->out.as<int32_t>();
    return GBSW_OK;
}

int gbsw_batch_stats(const gbsw_batch* b, gbsw_stats* out)
{
    if (!b || !out) return fail(GBSW_E_ARGUMENT, "null argument");
    *out = b->stats;
    return GBSW_OK;
}

int gbsw_batch_launch_stats(const gbsw_batch* b, int32_t index, gbsw_launch_stat* out)
{
    if (!b || !out) return fail(GBSW_E_ARGUMENT, "null argument");
    if (index < 0 || (size_t)index >= b->launches.size()) return fail(GBSW_E_ARGUMENT, "launch index out of range");
    const LaunchRec& L = b->launches[(size_t)index];
    out->kind = L.kind;
    out->columns_per_lane = L.K;
    out->workgroups = L.grid;
    out->pairs = L.pairs;
    out->cells = L.cells;
    out->ms = L.ms;
    return GBSW_OK;
}

int gbsw_batch_autotune(gbsw_batch* b, const gbsw_scoring* sc, int32_t repeats, int32_t* model, double* ms)
{
    if (!b || !sc) return fail(GBSW_E_ARGUMENT, "null argument");
    if (repeats < 1) repeats = 1;
    gbsw_context* ctx = b->ctx;
    GBSW_HIP_TRY(hipSetDevice(ctx->device));
    Job& job = b->job;
    // (the plan of the next align follows the model)
    auto use_model = [&](int m) { job.kmodel = m; };
    // the batch's current model first; another one must beat it by more than
    // kTuneMargin (run-to-run noise of a batch is about 1 %)
    constexpr double kTuneMargin = 0.015;
    const int current = job.kmodel;
    int best = -1;
    double best_ms = 1e300;
    std::vector<std::string> tried;
    for (int i = 0; i < kGeometryModels; ++i) {
        const int m = i == 0 ? current : (i <= current ? i - 1 : i);
        use_model(m);
        // models whose plan is one already timed add nothing
        std::string plan;
        int rc = batched_plan_text(ctx->ex, job, sc, &plan);
        if (rc) return rc;
        if (std::find(tried.begin(), tried.end(), plan) != tried.end()) continue;
        tried.push_back(std::move(plan));
        double m_ms = 1e300;
        for (int r = 0; !rc && r < repeats + 1; ++r) {
            rc = gbsw_batch_align(b, sc, GBSW_BATCHED);
            if (!rc && r > 0) m_ms = std::min(m_ms, b->stats.device_ms); // the first run captures the graph
        }
        if (rc) return rc;
        if (best < 0 || m_ms < best_ms * (1.0 - kTuneMargin)) { best_ms = m_ms; best = m; }
    }
    use_model(best);
    ctx->ex.kmodel = best; // batches created afterwards start from it
    if (model) *model = best;
    if (ms) *ms = best_ms;
    return GBSW_OK;
}

int gbsw_align(gbsw_context* ctx, const gbsw_scoring* sc, int32_t mode, int64_t n, const char* ref,
               const uint64_t* ref_off, const char* query, const uint64_t* query_off, int32_t* score,
               int32_t* ref_begin, int32_t* ref_end, int32_t* query_begin, int32_t* query_end)
{
    if (!sc || !ctx) return fail(GBSW_E_ARGUMENT, "null argument");
    // the context's one-shot batch: its device buffers are kept and only grow, so
    // repeated calls allocate and free nothing (a free would also wait for the
    // whole device)
    if (!ctx->oneshot) {
        ctx->oneshot = new gbsw_batch();
        ctx->oneshot->one_shot = true;
    }
    gbsw_batch* b = ctx->oneshot;
    int rc = batch_fill(b, ctx, ctx->ex, true, sc->alphabet, n, ref, ref_off, query, query_off);
    // few results: copied behind the kernels, with the one wait of the call
    constexpr int64_t kStagedResults = 16384;
    int32_t* pinned = nullptr;
    if (!rc && n && n <= kStagedResults) {
        if (b->results.reserve(sizeof(int32_t) * 5 * (size_t)n) == hipSuccess) pinned = b->results.as<int32_t>();
        else (void)hipGetLastError(); // (copied after the job, then)
    }
    if (!rc) {
        rc = batch_align_on(b, ctx->ex, sc, mode, pinned);
        if (rc) {
            const std::string err = gbsw_last_error();
            (void)hipStreamSynchronize(ctx->ex.stream); // (the input block may be under way)
            set_error(err);
        }
    }
    if (!rc && pinned) {
        int32_t* dst[5] = {score, ref_begin, ref_end, query_begin, query_end};
        for (int f = 0; f < 5; ++f)
            if (dst[f]) std::memcpy(dst[f], pinned + (size_t)f * (size_t)n, sizeof(int32_t) * (size_t)n);
    } else if (!rc) {
        rc = gbsw_batch_results(b, score, ref_begin, ref_end, query_begin, query_end);
    }
    return rc;
}

int gbsw_align_noalloc(gbsw_context* ctx, const gbsw_scoring* sc, int32_t mode, int64_t n, const char* ref,
                       const uint64_t* ref_off, const char* query, const uint64_t* query_off, int32_t* score,
                       int32_t* ref_begin, int32_t* ref_end, int32_t* query_begin, int32_t* query_end)
{
    if (!sc || !ctx) return fail(GBSW_E_ARGUMENT, "null argument");
    if (n < 0 || (n > 0 && (!ref_off || !query_off))) return fail(GBSW_E_ARGUMENT, "null offsets or negative pair count");
    GBSW_HIP_TRY(hipSetDevice(ctx->device));
    const uint64_t rb = n ? ref_off[n] - ref_off[0] : 0;
    const uint64_t qb = n ? query_off[n] - query_off[0] : 0;
    int rc = noalloc_carve(ctx, n, rb, qb);
    gbsw_batch* b = ctx->nbatch;
    if (!rc) rc = batch_fill(b, ctx, ctx->nx, false, sc->alphabet, n, ref, ref_off, query, query_off);
    if (!rc) rc = batch_align_on(b, ctx->nx, sc, mode);
    if (!rc) rc = gbsw_batch_results(b, score, ref_begin, ref_end, query_begin, query_end);
    return rc;
}

} // extern "C"
