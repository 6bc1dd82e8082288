// gbsw_exec.cpp -- the alignment pipeline of one job: geometry choice, length
// buckets, device binning, kernel launches on concurrent streams, the int32
// recompute of saturated pairs, and timing.
//
// Replaces the per-chunk body of driver.cpp:88-221 (pack, two-stream copies,
// forward launch, host newMin, reverse launch, copies back).
#include <algorithm>
#include <climits>
#include <cmath>
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>

#include "gbsw_internal.hpp"

namespace gbsw {

namespace {
thread_local std::string g_err;
}

void set_error(const std::string& msg) { g_err = msg; }
int fail(int code, const std::string& msg)
{
    g_err = msg;
    return code;
}
const char* last_error_text() { return g_err.c_str(); }

void DeviceBuffer::release()
{
    if (ptr && owned) (void)hipFree(ptr);
    ptr = nullptr;
    bytes = 0;
    owned = true;
}

hipError_t DeviceBuffer::reserve(size_t b)
{
    if (b <= bytes) return hipSuccess;
    if (!owned) return hipErrorOutOfMemory; // a view never grows
    release();
    hipError_t e = hipMalloc(&ptr, b);
    if (e == hipSuccess) bytes = b;
    else ptr = nullptr;
    return e;
}

void PinnedBuffer::release()
{
    if (ptr) (void)hipHostFree(ptr);
    ptr = nullptr;
    bytes = 0;
}

hipError_t PinnedBuffer::reserve(size_t b)
{
    if (b <= bytes) return hipSuccess;
    release();
    hipError_t e = hipHostMalloc(&ptr, b, hipHostMallocDefault);
    if (e == hipSuccess) bytes = b;
    else ptr = nullptr;
    return e;
}

namespace {

// Defaults of the per-context options.  GBSW_F16=0 keeps every bucket on the
// int16 kernels; GBSW_STREAMS=1 serialises the buckets (per-kernel timing and
// counters).
bool default_f16()
{
    const char* e = std::getenv("GBSW_F16");
    return !(e && std::atoi(e) == 0);
}

bool default_graphs()
{
    const char* e = std::getenv("GBSW_GRAPHS");
    return !(e && std::atoi(e) == 0);
}

bool default_split()
{
    const char* e = std::getenv("GBSW_SPLIT");
    return !(e && std::atoi(e) == 0);
}

int default_kmodel()
{
    const char* e = std::getenv("GBSW_KMODEL");
    const int m = e ? std::atoi(e) : kModelOccupancy;
    return (m >= 0 && m < kGeometryModels) ? m : kModelOccupancy;
}

int default_streams()
{
    const char* e = std::getenv("GBSW_STREAMS");
    const int v = e ? std::atoi(e) : kDefaultStreams;
    return std::max(1, std::min(kAuxStreams + 1, v));
}

// LDS bytes of a workgroup; bnd_bytes = 4 (packed int16) or 8 (int32 kernel).
int lds_for(int K, int alpha, bool p8, int bnd_bytes = 4)
{
    return lds_layout(prof_row_bytes(K, p8), alpha, bnd_bytes).total;
}

// Lanes per pair of the sweep kernel with eight pairs per wave (16 lanes for two).
constexpr int kLanesPerTwo = kLanesPerPair / 2;

int sweep_lds_for(int K, int alpha, int form, int G)
{
    return G == kLanesPerTwo ? pairs_lds(K, alpha).total : sweep_lds(G, K, form, alpha, 4).total;
}

int grid_for(const Exec& ex, int kind, int K, int lds, int64_t nquads)
{
    int occ = kernel_occupancy(kind, K, lds);
    if (occ < 1) occ = 1;
    const int64_t full = (int64_t)occ * ex.num_cu, simds = 4 * (int64_t)ex.num_cu;
    // Work items that would all be resident, at least two per SIMD: a whole number per
    // SIMD, the rest from the queue.  The first to finish takes them then; resident from
    // the start, they slow SIMDs whose long items decide the end.  (Short reads, 2,100
    // to 2,500 sets on 1,024 SIMDs: 0.310 - 0.344 ms against 0.348 - 0.383; 3,500 and
    // 4,000 sets 0.406 and 0.425 against 0.459 and 0.474; 3,000 sets 0.394 and 0.387.)
    if (nquads < full && nquads >= 2 * simds) return (int)(nquads / simds * simds);
    return (int)std::max<int64_t>(1, std::min<int64_t>(full, nquads));
}

// A kind as launch statistics report it.
int reported_kind(int kind)
{
    if (kind & kHalfPairs) return kByteProfile | kReportedPairs;
    return kind & kReportedKind;
}

// Launch one kernel between two timing events.
int launch_timed(Exec& ex, hipStream_t stream, int kind, int K, int grid, int lds, KernelArgs& a, void* bnd)
{
    const size_t slot = ex.launches.size();
    a.bnd = bnd;
    while (ex.kev.size() < 2 * (slot + 1)) {
        hipEvent_t e;
        GBSW_HIP_TRY(hipEventCreate(&e));
        ex.kev.push_back(e);
    }
    GBSW_HIP_TRY(hipEventRecord(ex.kev[2 * slot], stream));
    GBSW_HIP_TRY(kernel_launch(kind, K, grid, lds, stream, a));
    GBSW_HIP_TRY(hipEventRecord(ex.kev[2 * slot + 1], stream));
    ex.launches.push_back({reported_kind(kind), K, grid, 0, 0, 0.0});
    return GBSW_OK;
}

// Tables (staged in pinned memory) and status words; the caller adds the rest.
PrepareArgs prepare_args(const Exec& ex, const Job& job, size_t sub_bytes)
{
    PrepareArgs p{};
    const uint8_t* th = ex.tables_host.as<uint8_t>();
    p.n = job.n;
    p.h_sub = (const int16_t*)th;
    p.h_lut = th + 2048;
    p.h_colmax = (const int16_t*)(th + 2304);
    p.sub = ex.sub.as<int16_t>();
    p.lut = ex.lut.as<uint8_t>();
    p.colmax = ex.colmax.as<int16_t>();
    p.status = ex.status.as<uint32_t>();
    p.queue = ex.queue.as<uint32_t>();
    p.split = ex.split_buf.as<uint32_t>();
    p.nsub = (int32_t)(sub_bytes / sizeof(int16_t));
    p.alpha = job.alpha;
    p.nstatus = kStatusWords;
    return p;
}

KernelArgs base_args(const Exec& ex, const Job& job, const gbsw_scoring* sc)
{
    KernelArgs a;
    std::memset(&a, 0, sizeof(a));
    a.ref = job.ref;
    a.ref_off = job.ref_off;
    a.qry = job.qry;
    a.qry_off = job.qry_off;
    a.n = job.n;
    a.out = job.out;
    a.status = ex.status.as<int32_t>();
    a.redo = ex.redo.as<int32_t>();
    a.lut = ex.lut.as<uint8_t>();
    a.sub = ex.sub.as<int16_t>();
    a.colmax = ex.colmax.as<int16_t>();
    a.alpha = job.alpha;
    a.gap_min = std::min(-(int32_t)sc->gap_open, -(int32_t)sc->gap_extend);
    a.gap_open = sc->gap_open;
    a.gap_extend = sc->gap_extend;
    a.sat_limit = 32767 - ex.max_sub;
    a.asym = table_is_asymmetric(sc, job) ? 1 : 0;
    a.bnd_rows = std::max(1, job.max_rows);
    return a;
}

} // namespace

int Exec::init(int dev, int ncu)
{
    device = dev;
    num_cu = ncu;
    streams = default_streams();
    f16 = default_f16();
    split = default_split();
    graphs = default_graphs();
    kmodel = default_kmodel();
    hipError_t e = hipStreamCreateWithFlags(&stream, hipStreamNonBlocking);
    if (e == hipSuccess) e = hipEventCreate(&ev_start);
    if (e == hipSuccess) e = hipEventCreate(&ev_stop);
    if (e == hipSuccess) e = hipEventCreateWithFlags(&ev_fork, hipEventDisableTiming);
    if (e == hipSuccess && ensure_streams(streams) != GBSW_OK) e = hipErrorOutOfMemory;
    if (e == hipSuccess) e = status.reserve(sizeof(int32_t) * kStatusWords);
    if (e == hipSuccess) e = status_host.reserve(sizeof(int32_t) * kStatusWords);
    if (e == hipSuccess) e = tables_host.reserve(4096);
    if (e == hipSuccess) e = queue.reserve(sizeof(uint32_t) * 64);
    if (e == hipSuccess) e = sub.reserve(sizeof(int16_t) * 1024);
    if (e == hipSuccess) e = lut.reserve(256);
    if (e == hipSuccess) e = colmax.reserve(sizeof(int16_t) * 32);
    if (e != hipSuccess) return fail(GBSW_E_DEVICE, std::string("stream/scratch setup: ") + hipGetErrorString(e));
    return GBSW_OK;
}

int Exec::init_views(int dev, int ncu)
{
    device = dev;
    num_cu = ncu;
    streams = default_streams();
    f16 = default_f16();
    split = default_split();
    graphs = false;
    fixed = true;
    kmodel = default_kmodel();
    GBSW_HIP_TRY(hipStreamCreateWithFlags(&stream, hipStreamNonBlocking));
    GBSW_HIP_TRY(hipEventCreate(&ev_start));
    GBSW_HIP_TRY(hipEventCreate(&ev_stop));
    GBSW_HIP_TRY(hipEventCreateWithFlags(&ev_fork, hipEventDisableTiming));
    // every stream a job may use, and the launch events, now: a job then creates nothing
    if (int rc = ensure_streams(kAuxStreams + 1)) return rc;
    while (kev.size() < 2 * (size_t)kNoallocLaunchEvents) {
        hipEvent_t e;
        GBSW_HIP_TRY(hipEventCreate(&e));
        kev.push_back(e);
    }
    GBSW_HIP_TRY(status_host.reserve(sizeof(int32_t) * kStatusWords));
    GBSW_HIP_TRY(tables_host.reserve(4096));
    return GBSW_OK;
}

int Exec::ensure_streams(int n)
{
    for (int i = 0; i < std::min(kAuxStreams, n - 1); ++i) {
        if (aux[i]) continue;
        GBSW_HIP_TRY(hipStreamCreateWithFlags(&aux[i], hipStreamNonBlocking));
        GBSW_HIP_TRY(hipEventCreateWithFlags(&ev_join[i], hipEventDisableTiming));
    }
    return GBSW_OK;
}

void Exec::destroy()
{
    if (stream) (void)hipStreamSynchronize(stream);
    for (int i = 0; i < kAuxStreams; ++i)
        if (aux[i]) (void)hipStreamSynchronize(aux[i]);
    for (hipEvent_t e : kev) (void)hipEventDestroy(e);
    kev.clear();
    if (ev_start) (void)hipEventDestroy(ev_start);
    if (ev_stop) (void)hipEventDestroy(ev_stop);
    if (ev_fork) (void)hipEventDestroy(ev_fork);
    for (int i = 0; i < kAuxStreams; ++i) {
        if (ev_join[i]) (void)hipEventDestroy(ev_join[i]);
        if (aux[i]) (void)hipStreamDestroy(aux[i]);
        ev_join[i] = nullptr;
        aux[i] = nullptr;
    }
    bnd.release(); queue.release(); status.release(); sub.release(); lut.release(); colmax.release(); redo.release();
    split_buf.release();
    status_host.release();
    tables_host.release();
    if (stream) (void)hipStreamDestroy(stream);
    stream = nullptr;
    ev_start = ev_stop = ev_fork = nullptr;
}

int max_k_for(int alpha, bool p8)
{
    int nk = 0;
    const int* ks = kernel_k_list(&nk);
    int best = ks[0];
    for (int i = 0; i < nk; ++i)
        if (lds_for(ks[i], alpha, p8) <= 65536) best = ks[i];
    return best;
}

double occupancy_threshold(int model)
{
    static const double thr[kGeometryModels] = {0.0, 2.5, 2.0, 3.0, 4.0, 1.5};
    return (model > 0 && model < kGeometryModels) ? thr[model] : 0.0;
}

// Share of the VALU issue rate `waves` per SIMD reach: the int16 kernels' large
// buckets issue 0.96 VALU instructions per CU per cycle at 4 waves per SIMD, 0.82
// at 2.75, 0.78 at 2 and 0.62 at 1.5 (rocprofv3 counters), so min(1, waves /
// threshold), threshold 2.5 by default.
double issue_share(double waves, double threshold)
{
    return (waves > 0 && threshold > 0) ? std::min(1.0, waves / threshold) : 1.0;
}

int k_for_cols(int cols, int alpha, int model)
{
    const bool p8 = byte_profile_alphabet(alpha);
    const int kmax = max_k_for(alpha, p8);
    int nk = 0;
    const int* ks = kernel_k_list(&nk);
    int best = ks[0];
    double best_cost = 1e300;
    for (int i = 0; i < nk; ++i) {
        const int K = ks[i];
        if (K > kmax) break;
        const int64_t strips = std::max<int64_t>(1, (cols + kVirtPerPair * K - 1) / (kVirtPerPair * K));
        // padded columns and the per-step cost, per strip
        double cost = (double)(strips * (K + 2) * 4 + (strips - 1));
        if (model != kModelClassic) // (one wave per workgroup)
            cost /= issue_share(kernel_occupancy(with_profile(kBatched, p8), K, lds_for(K, alpha, p8)) / 4.0,
                                occupancy_threshold(model));
        if (cost < best_cost) { best_cost = cost; best = K; }
    }
    return best;
}

void place_buckets(std::vector<Bucket>& out, const Bucket* by_class, int classes)
{
    out.clear();
    int64_t at = 0;
    for (int c = classes - 1; c >= 0; --c) { // the sort order: longest class first
        if (by_class[c].count == 0) continue;
        out.push_back(by_class[c]);
        out.back().begin = at;
        at += by_class[c].count;
    }
}

int wide_grid_cap(const Exec& ex, int alpha)
{
    int occ = 1;
    for (int form = alpha <= kRegAlpha ? kProfRegs : kProfBytes; form <= kProfWords; ++form)
        occ = std::max(occ, kernel_occupancy(sweep_kind(kBatchedF16, form, kWideGroup), 1,
                                             sweep_lds_for(1, alpha, form, kWave)));
    return occ * ex.num_cu;
}

bool f16_high_byte_exact(int32_t s)
{
    // an integer is an f16 value with a zero low byte when it has at most three
    // significant bits (leading one and two mantissa bits) below 2^11
    const int32_t a = s < 0 ? -s : s;
    if (a >= 2048) return false;
    return a == 0 || (a >> __builtin_ctz((uint32_t)a)) < 8;
}

SweepChoice sweep_choice(const std::vector<int16_t>& sub, int alpha, int32_t gap_open, int32_t gap_extend,
                         int32_t max_sub, bool bytes, int32_t max_cols)
{
    SweepChoice c;
    const int32_t ge = -gap_extend, go = -gap_open, cost = ge + go;
    int32_t lo = 1 << 30, hi = -(1 << 30);
    for (int r = 0; r < alpha; ++r)
        for (int q = 0; q < alpha; ++q) {
            lo = std::min<int32_t>(lo, sub[(size_t)(r * alpha + q)]);
            hi = std::max<int32_t>(hi, sub[(size_t)(r * alpha + q)]);
        }
    // Tables hold score + bias; 0 is padding, which must score below zero.  The step adds
    // score + open + extend: as it stands in the tables where that fits (bias = cost),
    // else, as bytes, from the smallest score up, the rest by `shift` (Sweep16Shifted).
    // (100,000 proteins with gaps of -2/-1 8.2 ms, with a 16-bit profile 11.6; a million
    // reads with gaps that cost nothing 27.9 ms, with a 16-bit profile 39.8, on the int16
    // kernels 47.6.)
    c.bias = cost;
    int32_t pad = cost > 0 ? -cost : -1; // (16-bit tables hold a padding word)
    c.form = kProfWords;
    if (bytes && cost > 0 && lo + cost >= 0 && hi + cost <= 255) {
        c.form = kProfBytes;
    } else if (bytes && hi - std::min(lo, -1) <= 255) {
        c.form = kProfBytes;
        c.bias = -std::min(lo, -1);
        pad = -c.bias;
    }
    if (c.form == kProfBytes && alpha <= kRegAlpha) c.form = kProfRegs;
    c.shift = cost - c.bias;
    // every value stays non-negative: the smallest is a zero cell's Ho plus the
    // smallest score
    c.base = go + std::max(0, -(std::min(lo, pad) + cost)) + 4;
    const int64_t offset = (int64_t)c.base + (int64_t)ge * (kRebase + 40);
    // int32 cells: any range; the profile holds the biased scores in 16 bits
    c.wide_ok = cost >= 1 && lo + cost > -32768 && hi + cost < 32768;
    // a pair below this never formed a value past 0x7C00 (largest offset, gap step
    // and one substitution on top of its best; the strict reverse pass keeps kRevLow
    // below zero)
    c.sat_limit = (int32_t)(0x7C00 - kRevLow - offset - 2 * ge - max_sub - 4);
    // The running offset and the scores leave most of the range to the cell values, or
    // enough for any pair of the job.  (A million reads with gaps of -600/-100 25.4 ms, on
    // the int16 kernels 33.7.)
    c.ok = (offset <= 8192 || (offset <= 24576 && (int64_t)max_cols * max_sub < c.sat_limit)) && max_sub <= 4096 &&
           lo + cost > -16384 && hi + cost < 16384;
    double same = 0, all = 0;
    for (int r = 0; r < alpha; ++r) same += sub[(size_t)(r * alpha + r)];
    for (int16_t v : sub) all += v;
    c.typical = 0.875 * same / alpha + (alpha > 1 ? 0.125 * (all - same) / ((double)alpha * (alpha - 1)) : 0.0);
    return c;
}

int sort_scratch_bytes(int64_t n, size_t* bytes)
{
    size_t tb = 0;
    GBSW_HIP_TRY(sort_pairs(nullptr, tb, nullptr, nullptr, nullptr, nullptr, (int)std::max<int64_t>(1, n), kSortBits,
                            nullptr));
    *bytes = std::max<size_t>(tb, 16);
    return GBSW_OK;
}

bool table_is_asymmetric(const gbsw_scoring* sc, const Job& job)
{
    if (sc->alphabet != GBSW_PROTEIN) return false;
    for (int r = 0; r < job.alpha; ++r)
        for (int c = 0; c < r; ++c) {
            const int cr = job.code_of ? job.code_of[r] : r, cc = job.code_of ? job.code_of[c] : c;
            if (sc->matrix[cr * 24 + cc] != sc->matrix[cc * 24 + cr]) return true;
        }
    return false;
}

int prepare_scoring(const Job& job, const gbsw_scoring* sc, std::vector<int16_t>& sub, int* max_sub, bool* p8,
                    bool* f16p8)
{
    if (sc->alphabet != job.alphabet) return fail(GBSW_E_ARGUMENT, "scoring alphabet differs from the batch alphabet");
    if (sc->gap_open > 0 || sc->gap_extend > 0) return fail(GBSW_E_SCORING, "gap_open and gap_extend must be <= 0");
    const int A = job.alpha;
    sub.assign((size_t)std::max(1, A * A), 0);
    int mx = 0;
    if (job.alphabet == GBSW_DNA) {
        for (int r = 0; r < A; ++r)
            for (int c = 0; c < A; ++c) sub[(size_t)(r * A + c)] = r == c ? sc->match : sc->mismatch;
        mx = std::max<int>(sc->match, sc->mismatch);
    } else {
        // the caller's table indexed enc(row)*24 + enc(col) (kernel.cpp:785-788),
        // restricted to the residue codes of the batch
        for (int r = 0; r < A; ++r)
            for (int c = 0; c < A; ++c) {
                const int cr = job.code_of ? job.code_of[r] : r, cc = job.code_of ? job.code_of[c] : c;
                const int16_t v = sc->matrix[cr * 24 + cc];
                sub[(size_t)(r * A + c)] = v;
                mx = std::max<int>(mx, v);
            }
    }
    for (int16_t v : sub)
        if (v < -16000 || v > 16000) return fail(GBSW_E_SCORING, "substitution scores must lie in [-16000, 16000]");
    *max_sub = std::max(0, mx);
    int lo = 0;
    for (int16_t v : sub) lo = std::min<int>(lo, v);
    *p8 = byte_profile_alphabet(A) && lo >= -127 && mx <= 127;
    if (f16p8) {
        // small alphabets hold scores of at most three significant bits as bytes (the byte
        // tables would take any that span 255; +9/-11 takes a 16-bit profile: a million
        // reads 31.4 ms, 21.9 at +3/-3)
        *f16p8 = true;
        for (int16_t v : sub) *f16p8 = *f16p8 && f16_high_byte_exact(v);
    }
    // result keys hold scores in 23 bits; int16 saturation is handled per pair
    if ((int64_t)job.max_cols * *max_sub >= (1 << 23)) return fail(GBSW_E_RANGE, "possible score exceeds 2^23");
    return GBSW_OK;
}

namespace {

// One launch of the batched form: adjacent length classes.
struct BucketPlan {
    Bucket bk;
    int kind = 0, K = 0, grid = 0, lds = 0, strips = 1; // K: the widest geometry of the launch
    int G = kLanesPerPair; // lanes per pair (64: one pair per wave)
    int32_t sat_limit = 0;
    std::vector<SetRange> ranges;    // sweep launches: geometries by position within the launch
    double work = 0, unit = 0;       // estimated cycles: of the whole launch on the full GPU, of its longest item alone
    size_t bnd_at = 0, split_at = 0; // 32-bit word offsets into ex.bnd / ex.split_buf
    int pairs_per_wave() const { return kWave / G; }
    int64_t sets() const { return (bk.count + pairs_per_wave() - 1) / pairs_per_wave(); }
};

bool plan_is_split(const BucketPlan& b)
{
    const int k = b.kind & 0xFF;
    return k == kSplit || k == kSplitF16 || (b.kind & kSplitStrips);
}

// 32-bit words of a split launch's bookkeeping: keys (2 x count u64), progress
// words (2 slots per workgroup, u64), done counters (2 x sets), release epochs
// (one per slot), the placement table (kXcds) and the strip gates (count), padded
// to a multiple of 64 (256 bytes) so that the next launch's 64-bit keys and
// progress words stay 8-byte aligned.
size_t split_words_of(const BucketPlan& b)
{
    const size_t words = 5 * (size_t)b.bk.count + 2 * (size_t)b.sets() + 3 * (size_t)(2 * b.grid) + kXcds;
    return (words + 63) & ~(size_t)63;
}

// Cycles of one step of a wave with K columns per lane, with other waves on its
// SIMD and alone (measured: 126 and 194 cycles at K = 1, 193 at K = 5 beside others,
// 391 / 455 / 602 at K = 5 / 6 / 8 alone); a strip with boundary rows takes more.
double step_issue(int K, bool ms) { return 25.0 * K + 80 + (ms ? 20 : 0); }
double step_alone(int K, bool ms) { return 58.0 * K + 135 + (ms ? 55 : 0); }
// Eight pairs per wave, K columns per lane.  (Short reads, K = 10 against four pairs at
// K = 5: 5k, 10k, 20k, 30k, 50k, 100k and 300k pairs 0.33, 0.47, 0.59, 0.72, 0.91, 1.55
// and 4.15 ms against 0.32, 0.34, 0.56, 0.71, 1.01, 1.84 and 4.91.)
double pairs_issue(int K) { return 29.5 * K + 52; }
double pairs_alone(int K) { return 56.0 * K + 200; }
// Forward plus reverse pass, in forward passes.
constexpr double kPasses = 1.6;
// A strip of the split form starts once its predecessor has published the rows of
// its first three chunks, which leave the predecessor's last virtual lane 2G steps
// after they enter it.
int split_lag(int G) { return 2 * G + 3 * kChunk; }
// Geometries of the sweep kernels, ascending.
#define GBSW_ITEM(k) k,
constexpr int kSweepK16[] = {GBSW_SWEEP_K16(GBSW_ITEM) GBSW_SWEEP_K16_WIDE(GBSW_ITEM)};
constexpr int kSweepK64[] = {GBSW_SWEEP_K64(GBSW_ITEM)};
constexpr int kSweepSplitK[] = {GBSW_SWEEP_K64_SPLIT(GBSW_ITEM)};
#undef GBSW_ITEM
constexpr int kSweepNarrowMax = 8; // widest geometry of the narrow four-pair kernel
static_assert(kPairsCols == kVirtPerPair * kSweepNarrowMax, "eight pairs per wave: the narrow classes");

// Estimates of one class in one geometry: work (wave cycles over all SIMDs) and
// the longest item's time.
struct GeoCost {
    double work = 1e300, unit = 1e300;
    int K = 0, strips = 1;
};
GeoCost geo_cost(const Exec& ex, const Bucket& bk, int G, int K, bool split)
{
    const int vl = 2 * G;
    GeoCost c;
    c.K = K;
    c.strips = std::max(1, (bk.max_cols + vl * K - 1) / (vl * K));
    const double n = (double)std::max<int64_t>(1, bk.count);
    const double strips = c.strips == 1 ? 1.0 : std::max(1.0, (double)bk.cols / n / (vl * K) + 0.5);
    const double steps = (double)bk.rows / n + vl - 1, longest = bk.max_rows + vl - 1;
    c.work = n * G / kWave * strips * steps * step_issue(K, c.strips > 1) * kPasses * (split ? 1.4 : 1.0) /
             (4.0 * ex.num_cu);
    c.unit = (split ? longest + (c.strips - 1) * (double)split_lag(G) : c.strips * longest) *
             step_alone(K, c.strips > 1) * kPasses;
    return c;
}

// The same for eight pairs per wave.
GeoCost pairs_cost(const Exec& ex, const Bucket& bk, int K)
{
    GeoCost c;
    c.K = K;
    const double n = (double)std::max<int64_t>(1, bk.count);
    c.work = n / 8 * ((double)bk.rows / n + kLanesPerPair - 1) * pairs_issue(K) * kPasses / (4.0 * ex.num_cu);
    c.unit = ((double)bk.max_rows + kLanesPerPair - 1) * pairs_alone(K) * kPasses;
    return c;
}

// The launches of a job whose scoring runs the sweep kernels.
//
// Which geometry a class takes.  Four pairs per wave issue the fewest instructions
// per cell; one pair per wave finishes a pair about four times sooner and takes any
// number of strips; its strips on several waves (the split form) finish it sooner
// still.  The sort order puts long classes first, so the forms are three adjacent
// stretches of it (split, one pair per wave, four pairs per wave: wide, then narrow
// geometries), one launch each.  A job lasts at least as long as its instructions
// take on the whole GPU and as its longest item takes alone; the stretches are
// those of least max + kOverlap x min of the two.
//
// pairs: the narrow classes with eight pairs per wave (cls: the fine classes).
// Returns the estimate.
double plan_sweeps_over(const Exec& ex, const Job& job, const std::vector<Bucket>& cls, const SweepChoice& sw,
                        bool may_split, bool pairs, std::vector<BucketPlan>& plan)
{
    constexpr double kOverlap = 0.35;
    const size_t n = cls.size();
    const double thr = occupancy_threshold(job.kmodel);
    auto lds = [&](int G, int K) { return sweep_lds_for(K, job.alpha, sw.form, G); };
    auto kind_of = [&](int kind, int flags) { return sweep_kind(kind, sw.form, sw.shift ? flags | kShifted : flags); };
    // share of the issue rate of a launch whose widest geometry is K
    auto share = [&](int flags, int G, int K) {
        const int l = lds(G, K);
        if (l > 65536) return 0.0;
        return issue_share(kernel_occupancy(kind_of(kBatchedF16, flags), K, l) / 4.0, thr);
    };
    struct Option {
        std::vector<GeoCost> cost; // per class
        std::vector<double> work, unit; // sums / maxima over [0, i) (or [i, n) for four pairs per wave)
        int cap = 0;
    };
    auto prefix = [&](Option& o) {
        o.work.assign(n + 1, 0.0);
        o.unit.assign(n + 1, 0.0);
        for (size_t i = 0; i < n; ++i) {
            o.work[i + 1] = o.work[i] + o.cost[i].work;
            o.unit[i + 1] = std::max(o.unit[i], o.cost[i].unit);
        }
    };
    // four pairs per wave: the widest geometry (its LDS decides the launch's
    // occupancy) is that of the first class
    Option four;
    size_t first = n; // classes before it have no such geometry
    four.cost.resize(n);
    four.work.assign(n + 1, 0.0);
    four.unit.assign(n + 1, 0.0);
    for (size_t i = n; i-- > 0;) {
        double s = 0.0;
        if (pairs && cls[i].max_cols <= kPairsCols) {
            const int K = std::max(2, (cls[i].max_cols + 15) / 16);
            s = K > kPairsNarrowMax ? share(kHalfPairs | kWideLanes, kLanesPerTwo, kPairsCols / 16)
                                    : share(kHalfPairs, kLanesPerTwo, kPairsNarrowMax);
            four.cost[i] = pairs_cost(ex, cls[i], K);
        } else {
            int K = 0;
            for (int k : kSweepK16)
                if (cls[i].max_cols <= kVirtPerPair * k) { K = k; break; }
            if (K) s = share(K > kSweepNarrowMax ? kWideLanes : 0, kLanesPerPair, K);
            if (K) four.cost[i] = geo_cost(ex, cls[i], kLanesPerPair, K, false);
        }
        if (s <= 0) break;
        first = i;
        four.work[i] = four.work[i + 1] + four.cost[i].work / s;
        four.unit[i] = std::max(four.unit[i + 1], four.cost[i].unit);
    }
    // one pair per wave: per widest geometry, the strips of least work or of the
    // shortest item; split: one geometry per launch
    std::vector<Option> one, split;
    for (int cap : kSweepK64) {
        const double s = share(kWideGroup, kWave, cap);
        if (s <= 0) break;
        for (int quick = 0; quick < 2; ++quick) {
            Option o;
            o.cap = cap;
            for (const Bucket& bk : cls) {
                GeoCost best;
                for (int K : kSweepK64) {
                    if (K > cap) break;
                    const GeoCost c = geo_cost(ex, bk, kWave, K, false);
                    if (quick ? c.unit < best.unit : c.work < best.work) best = c;
                }
                best.work /= s;
                o.cost.push_back(best);
            }
            prefix(o);
            one.push_back(std::move(o));
        }
    }
    if (may_split)
        for (int K : kSweepSplitK) {
            if (lds(kWave, K) > 65536) break;
            const int kind = kind_of(kSplitF16, kWideGroup);
            const double s = issue_share(kernel_occupancy(kind, K, lds(kWave, K)) / 4.0, thr);
            Option o;
            o.cap = K;
            for (const Bucket& bk : cls) {
                o.cost.push_back(geo_cost(ex, bk, kWave, K, true));
                o.cost.back().work /= s;
            }
            prefix(o);
            split.push_back(std::move(o));
        }
    double best = 1e300;
    size_t i64 = 0, i16 = n, which_one = 0, which_split = 0;
    // launches beyond the first cost little beside a large job and show in a small one
    constexpr double kLaunch = 12000;
    // (more pairs than this fill the GPU unsplit)
    const int64_t most_split = 16 * (int64_t)ex.num_cu;
    for (size_t o = 0; o < one.size(); ++o)
        for (size_t b = first; b <= n; ++b) { // [b, n) four pairs per wave
            std::vector<double> unit_tail(b + 1, 0.0); // longest one-pair item of [i, b)
            for (size_t i = b; i-- > 0;) unit_tail[i] = std::max(unit_tail[i + 1], one[o].cost[i].unit);
            const double w4 = four.work[b], u4 = four.unit[b];
            auto consider = [&](size_t a, size_t s) { // [0, a) split
                double w = w4 + one[o].work[b] - one[o].work[a], u = std::max(u4, unit_tail[a]);
                if (a) {
                    w += split[s].work[a];
                    u = std::max(u, split[s].unit[a]);
                }
                const double m = std::max(w, u) + kOverlap * std::min(w, u) +
                                 kLaunch * ((a > 0 ? 1 : 0) + (b > a ? 1 : 0) + (n > b ? 1 : 0));
                if (m < best) { best = m; i64 = a; i16 = b; which_one = o; which_split = s; }
            };
            consider(0, 0);
            for (size_t s = 0; s < split.size(); ++s)
                for (size_t a = 1; a <= b && cls[a - 1].begin + cls[a - 1].count <= most_split; ++a) consider(a, s);
        }

    auto add = [&](size_t from, size_t to, int G, int flags, const Option& o, bool is_split) {
        if (from >= to) return;
        BucketPlan b;
        b.G = G;
        b.sat_limit = sw.sat_limit;
        b.bk.begin = cls[from].begin;
        for (size_t i = from; i < to; ++i) {
            const GeoCost& c = o.cost[i];
            b.bk.add(cls[i]);
            b.K = std::max(b.K, c.K);
            b.strips = std::max(b.strips, c.strips);
            b.work += c.work;
            b.unit = std::max(b.unit, c.unit);
            const int32_t end = (int32_t)b.bk.count;
            if (!b.ranges.empty() && b.ranges.back().K == c.K) b.ranges.back().end = end;
            else b.ranges.push_back({end, c.K});
        }
        b.kind = kind_of(is_split ? kSplitF16 : kBatchedF16, flags);
        b.lds = lds(G, b.K);
        plan.push_back(b);
    };
    size_t narrow = i16;
    while (narrow < n && cls[narrow].max_cols > kPairsCols) ++narrow;
    if (i64) add(0, i64, kWave, kWideGroup, split[which_split], true);
    add(i64, i16, kWave, kWideGroup, one[which_one], false);
    add(i16, narrow, kLanesPerPair, kWideLanes, four, false);
    if (pairs) {
        size_t few = narrow;
        while (few < n && four.cost[few].K > kPairsNarrowMax) ++few;
        add(narrow, few, kLanesPerTwo, kHalfPairs | kWideLanes, four, false);
        add(few, n, kLanesPerTwo, kHalfPairs, four, false);
    } else {
        add(narrow, n, kLanesPerPair, 0, four, false);
    }
    return best;
}

// int32 cells, one pair per wave, K columns per virtual lane (split: strips on several
// waves).
constexpr int kMostInt32 = 4; // widest geometry of the int32 kernels
void int32_geometry(const Job& job, int K, bool split, BucketPlan& b)
{
    b.G = kWave;
    b.K = K;
    b.kind = kBatchedWide | kWideGroup | (split ? kSplitStrips : 0);
    b.strips = std::max(1, (b.bk.max_cols + 2 * kWave * K - 1) / (2 * kWave * K));
    b.lds = sweep_lds(kWave, K, kProfWords, job.alpha, 8).total;
}
// The split form in the geometry whose chain of strips is shortest.  (An int32 step
// takes about twice a 16-bit one.)
void int32_split_geometry(const Job& job, BucketPlan& b)
{
    double best = 1e300;
    int K = kMostInt32;
    for (int k = 2; k <= kMostInt32; k += 2) {
        const double strips = std::ceil(b.bk.max_cols / (2.0 * kWave * k));
        const double t = (b.bk.max_rows + (strips - 1) * split_lag(kWave)) * step_alone(2 * k, true);
        if (t < best) { best = t; K = k; }
    }
    int32_geometry(job, K, true, b);
    b.unit = best * kPasses;
}

// The classes of the longest pairs, as far as an alike pair of them passes the 16-bit
// range (SweepChoice::typical per column, one residue in eight changed: 2.25 of +3/-3,
// 4.9 of BLOSUM62), take int32 cells at once, beside the others, where their strips'
// waves are few (two per SIMD).  Recomputed after the others, two of 400 long reads
// doubled the time, 21.5 ms where this takes 12.2, and 36 of 100 alike proteins of up to
// 8,192 columns 15.3 ms where this takes 8.2: their chain of strips is as long as
// everything else.  Pairs that are not alike pay for it: 100 unrelated proteins of up to
// 8,192 columns 8.3 ms, 7.2 in 16 bits.  (By the largest score of the table, 11 of W
// against W, proteins from 3,576 columns on paid too: 20, 100 and 500 of up to 4,096
// columns 4.8, 5.7 and 8.0 ms instead of 4.4, 4.8 and 6.7.)
size_t plan_int32(const Exec& ex, const Job& job, const SweepChoice& sw, std::vector<BucketPlan>& plan)
{
    if (ex.fixed || !sw.wide_ok) return 0;
    BucketPlan b;
    size_t n = 0;
    for (; n < job.buckets.size(); ++n) {
        const Bucket& bk = job.buckets[n];
        if (sw.typical * (double)bk.max_cols < (double)sw.sat_limit) break;
        b.bk.add(bk);
    }
    if (!n) return 0;
    b.bk.begin = job.buckets[0].begin;
    int32_split_geometry(job, b);
    if (b.strips < 2 || b.bk.count * b.strips > 8 * (int64_t)ex.num_cu) return 0;
    b.sat_limit = INT_MAX;
    b.ranges.push_back({(int32_t)b.bk.count, b.K});
    plan.push_back(b);
    return n;
}

// Whether a plan's stretches are those of the fine classes.
bool plan_is_fine(const std::vector<BucketPlan>& plan)
{
    for (const BucketPlan& b : plan)
        if (b.kind & kHalfPairs) return true;
    return false;
}

// Eight pairs per wave: jobs with two such waves per SIMD and more (fewer leave SIMDs
// idle) and register tables, where the estimate is less.
void plan_sweeps(const Exec& ex, const Job& job, const SweepChoice& sw, bool may_split, bool asym,
                 std::vector<BucketPlan>& plan)
{
    const size_t wide = may_split ? plan_int32(ex, job, sw, plan) : 0;
    if (wide) {
        const std::vector<Bucket> rest(job.buckets.begin() + (std::ptrdiff_t)wide, job.buckets.end());
        if (!rest.empty()) (void)plan_sweeps_over(ex, job, rest, sw, may_split, false, plan);
        return;
    }
    const double t = plan_sweeps_over(ex, job, job.buckets, sw, may_split, false, plan);
    if (sw.form != kProfRegs || asym || job.fine.empty() || job.n <= kSmallSort ||
        job.n < 8 * 2 * 4 * (int64_t)ex.num_cu)
        return;
    std::vector<BucketPlan> other;
    // (only with that kernel in it: the pairs are then sorted by the fine classes)
    if (plan_sweeps_over(ex, job, job.fine, sw, may_split, true, other) < t && plan_is_fine(other)) plan.swap(other);
}

// The launches of a job on the int16 kernels (scorings outside the sweep kernels'
// range, option F16 off): one per geometry.  A multi-strip launch is split when it
// has too few quads to keep every workgroup busy for two rounds (on the 200k-pair
// DNA mix: 1765 vs 827 GCUPS at 1.4 quads per workgroup; 988 vs 1275 on protein at
// 2.7).  one_launch: all pairs in one launch, in the geometry of the longest.
void plan_int16(const Exec& ex, const Job& job, int max_sub, bool p8, int kclamp, bool may_split, bool one_launch,
                std::vector<BucketPlan>& plan)
{
    for (const Bucket& bk : job.buckets) {
        const int K = std::min(kclamp, k_for_cols(one_launch ? job.max_cols : bk.max_cols, job.alpha, job.kmodel));
        const int strips = std::max(1, (bk.max_cols + kVirtPerPair * K - 1) / (kVirtPerPair * K));
        if (plan.empty() || (!one_launch && (plan.back().K != K || (plan.back().strips > 1) != (strips > 1)))) {
            plan.push_back(BucketPlan{});
            BucketPlan& b = plan.back();
            b.bk.begin = bk.begin;
            b.K = K;
            b.kind = with_profile(kBatched, p8);
            b.lds = lds_for(K, job.alpha, p8);
            b.sat_limit = 32767 - max_sub;
        }
        BucketPlan& b = plan.back();
        b.bk.add(bk);
        b.strips = std::max(b.strips, strips);
        const GeoCost c = geo_cost(ex, bk, kLanesPerPair, K, false);
        b.work += 1.4 * c.work;
        b.unit = std::max(b.unit, 1.4 * c.unit);
    }
    for (BucketPlan& b : plan) {
        const int64_t full = (int64_t)std::max(1, kernel_occupancy(b.kind, b.K, b.lds)) * ex.num_cu;
        const int skind = with_profile(kSplit, p8);
        if (may_split && b.strips > 1 && b.sets() < 2 * full && kernel_has(skind, b.K)) b.kind = skind;
    }
}

// Kernels, grids and scratch of every launch (host only; reserves the buffers).
int plan_batched(Exec& ex, const Job& job, int max_sub, bool p8, const SweepChoice& sw, bool asym, int kclamp,
                 std::vector<BucketPlan>& plan)
{
    plan.clear();
    // (an asymmetric table may need a third pass per pair, which strip items lack)
    const bool may_split = ex.split && !ex.split_misplaced && !asym;
    auto set_grid = [&](BucketPlan& b) {
        if (plan_is_split(b)) {
            // a multiple of kXcds: every XCD's counter serves every kXcds-th set, with a
            // workgroup for each of their strips at most, and two boundary slots each
            const int occ = std::max(1, kernel_occupancy(b.kind, b.K, b.lds));
            const int64_t busy = (b.sets() + kXcds - 1) / kXcds * b.strips * kXcds;
            b.grid = (int)std::max<int64_t>(kXcds, std::min<int64_t>((int64_t)occ * ex.num_cu / kXcds * kXcds, busy));
        } else {
            b.grid = grid_for(ex, b.kind, b.K, b.lds, b.sets());
        }
    };
    // boundary rows and split bookkeeping (keys: 2 x count u64, prog: slots u64,
    // done: 2 x sets u32, rel: slots u32, xcc, gate: count u32) in 32-bit words
    size_t bnd_words = 0, split_words = 0;
    auto sizes = [&]() {
        bnd_words = split_words = 0;
        for (BucketPlan& b : plan) {
            b.bnd_at = bnd_words;
            const size_t per_wg = (size_t)b.pairs_per_wave() * (size_t)std::max(1, b.bk.max_rows);
            if (plan_is_split(b)) {
                // (int32 rows are pairs of 64-bit alignment)
                const size_t row_words = b.kind & kSplitStrips ? 2 : 1;
                bnd_words = (bnd_words + 1) & ~(size_t)1;
                b.bnd_at = bnd_words;
                bnd_words += (size_t)2 * b.grid * per_wg * row_words;
                b.split_at = split_words;
                split_words += split_words_of(b);
            } else if (b.strips > 1) {
                // (a launch whose pairs all fit one strip hands no boundary rows on)
                bnd_words += (size_t)b.grid * per_wg;
            }
        }
    };
    auto make = [&](bool split, bool one_launch = false) {
        plan.clear();
        if (sw.ok) plan_sweeps(ex, job, sw, split, asym, plan);
        else plan_int16(ex, job, max_sub, p8, kclamp, split, one_launch, plan);
        for (BucketPlan& b : plan) set_grid(b);
        sizes();
    };
    make(may_split);
    for (const BucketPlan& b : plan)
        if (sw.ok && (b.ranges.empty() || b.ranges.size() > (size_t)kMaxRanges || b.ranges.back().end != b.bk.count))
            return fail(GBSW_E_INTERNAL, "the geometry ranges of a launch do not hold its pairs");
    if (ex.fixed) {
        // preallocated buffers (a serving slot): without the split form where its
        // boundary slots and bookkeeping do not fit
        if (bnd_words * sizeof(uint32_t) > ex.bnd.bytes || split_words * sizeof(uint32_t) > ex.split_buf.bytes) make(false);
        // then the widest multi-strip grids shrink (a persistent grid of any size
        // drains its queue) until the boundary rows fit
        while (bnd_words * sizeof(uint32_t) > ex.bnd.bytes) {
            BucketPlan* w = nullptr;
            for (BucketPlan& b : plan)
                if (!plan_is_split(b) && b.strips > 1 && b.grid > 1 && (!w || b.grid > w->grid)) w = &b;
            if (!w && plan.size() > 1 && !sw.ok) {
                // a workgroup per launch is too much still: all pairs in one launch, which
                // needs the rows of one workgroup (a server's slots hold that much at
                // least; sweep plans have one launch with boundary rows anyway)
                make(false, true);
                continue;
            }
            if (!w) return fail(GBSW_E_RANGE, "strip boundary rows exceed the preallocated scratch");
            w->grid = std::max(1, w->grid / 2);
            sizes();
        }
    }
    // Launches run concurrently on the streams, the ones whose single work item
    // takes longest first, so that few long pairs overlap the bulk instead of running
    // alone at the end; record_batched puts each on the least-loaded stream.
    std::sort(plan.begin(), plan.end(), [](const BucketPlan& x, const BucketPlan& y) {
        return x.unit != y.unit ? x.unit > y.unit : x.bk.begin < y.bk.begin;
    });
    const size_t nb = std::max<size_t>(plan.size(), 1);
    if (ex.queue.bytes < sizeof(uint32_t) * kXcds * nb) GBSW_HIP_TRY(ex.queue.reserve(sizeof(uint32_t) * kXcds * nb));
    if (split_words) GBSW_HIP_TRY(ex.split_buf.reserve(split_words * sizeof(uint32_t)));
    GBSW_HIP_TRY(ex.bnd.reserve(std::max<size_t>(bnd_words, 1) * sizeof(uint32_t)));
    return GBSW_OK;
}

// The split form's bookkeeping of launch b, at its place in ex.split_buf.
int set_split_args(const Exec& ex, const BucketPlan& b, KernelArgs& a)
{
    uint32_t* w = ex.split_buf.as<uint32_t>() + b.split_at;
    const int64_t nslots = 2 * (int64_t)b.grid;
    a.split.keys = (uint64_t*)w;
    a.split.prog = (uint64_t*)(w + 4 * b.bk.count);
    a.split.done = w + 4 * b.bk.count + 2 * nslots;
    a.split.rel = a.split.done + 2 * b.sets();
    a.split.xcc = a.split.rel + nslots;
    a.split.gate = a.split.xcc + kXcds;
    if (((uintptr_t)a.split.keys | (uintptr_t)a.split.prog) & 7)
        return fail(GBSW_E_INTERNAL, "split bookkeeping of a launch is not 8-byte aligned");
    a.split.strips = b.strips;
    a.split.slots = (int32_t)(nslots / kXcds);
    a.split.first = b.kind & kSplitStrips ? 1 : 0;
    return GBSW_OK;
}

// Stream work of the batched form (recorded eagerly or into a graph).
int record_batched(Exec& ex, const Job& job, KernelArgs a, const std::vector<BucketPlan>& plan, size_t sub_bytes)
{
    hipStream_t st0 = ex.stream;
    const size_t nb = plan.size();
    PrepareArgs pre = prepare_args(ex, job, sub_bytes);
    pre.ref_off = job.ref_off;
    pre.qry_off = job.qry_off;
    pre.nqueue = (int32_t)(kXcds * nb);
    for (const BucketPlan& b : plan)
        if (plan_is_split(b)) pre.nsplit = std::max(pre.nsplit, (int64_t)(b.split_at + split_words_of(b)));
    // the work order: up to kSmallSort pairs by one workgroup of the preparing launch
    // (10k pairs: 57 us less than keys and radix sort from launch to launch); more by a
    // radix sort on the whole GPU
    if (job.n <= kSmallSort) {
        pre.order = job.order;
    } else {
        pre.keys = job.keys;
        pre.vals = job.vals;
        pre.fine = plan_is_fine(plan) ? 1 : 0;
    }
    GBSW_HIP_TRY(prepare_job(pre, st0));
    if (pre.keys) {
        size_t tb = job.sort_temp_bytes;
        GBSW_HIP_TRY(sort_pairs(job.sort_temp, tb, job.keys, job.keys_sorted, job.vals, job.order, (int)job.n, kSortBits,
                                st0));
    }
    const int ns = std::max(1, std::min({kAuxStreams + 1, ex.streams, (int)nb}));
    if (ns > 1) GBSW_HIP_TRY(hipEventRecord(ex.ev_fork, st0));
    for (int i = 0; i < ns - 1; ++i) GBSW_HIP_TRY(hipStreamWaitEvent(ex.aux[i], ex.ev_fork, 0));
    // each launch (in the plan's order) goes to the stream with the least estimated
    // work queued so far (its share of the whole GPU, or its longest item): a short
    // bucket then does not wait behind a long one and run alone at the end
    std::vector<double> load((size_t)ns, 0.0);
    for (size_t i = 0; i < plan.size(); ++i) {
        size_t si = 0;
        for (size_t q = 1; q < load.size(); ++q)
            if (load[q] < load[si]) si = q;
        const BucketPlan& b = plan[i];
        const Bucket& bk = b.bk;
        load[si] += std::max(b.work, b.unit);
        a.order = job.order + bk.begin;
        a.order_n = bk.count;
        a.queue = ex.queue.as<uint32_t>() + kXcds * i;
        a.bnd_rows = std::max(1, bk.max_rows);
        a.kmax = b.K;
        a.nranges = (int32_t)b.ranges.size(); // (plan_batched: at most kMaxRanges)
        for (int32_t r = 0; r < a.nranges; ++r) a.ranges[r] = b.ranges[(size_t)r];
        a.sat_limit = b.sat_limit;
        std::memset(&a.split, 0, sizeof(a.split));
        if (plan_is_split(b))
            if (int rc = set_split_args(ex, b, a)) return rc;
        hipStream_t st = si == 0 ? st0 : ex.aux[si - 1];
        int rc = launch_timed(ex, st, b.kind, b.K, b.grid, b.lds, a, ex.bnd.as<uint32_t>() + b.bnd_at);
        if (rc) return rc;
        ex.launches.back().pairs = bk.count;
        ex.launches.back().cells = bk.cells;
    }
    for (int i = 0; i < ns - 1; ++i) {
        GBSW_HIP_TRY(hipEventRecord(ex.ev_join[i], ex.aux[i]));
        GBSW_HIP_TRY(hipStreamWaitEvent(st0, ex.ev_join[i], 0));
    }
    GBSW_HIP_TRY(hipMemcpyAsync(ex.status_host.ptr, ex.status.ptr, sizeof(int32_t) * kStatusWords,
                                hipMemcpyDeviceToHost, st0));
    return GBSW_OK;
}

// Every launch of a plan, as bytes.
std::string plan_text(const std::vector<BucketPlan>& plan)
{
    std::string k;
    for (const BucketPlan& b : plan) {
        const Bucket& bk = b.bk;
        const int64_t f[] = {b.kind, b.K, b.grid, b.lds, b.strips, (int64_t)b.bnd_at, (int64_t)b.split_at,
                             bk.begin, bk.count, bk.max_cols, bk.max_rows};
        k.append((const char*)f, sizeof(f));
        k.append((const char*)b.ranges.data(), sizeof(SetRange) * b.ranges.size());
    }
    return k;
}

// What a captured graph depends on besides the batch's bytes: the scoring, the
// options, the addresses of the context buffers it writes, and each bucket's
// slice of the sort order (baked into the captured launch arguments; another
// length -> geometry map of the same batch moves the slices while the plans may
// stay alike).
std::string graph_key(const Exec& ex, const Job& job, const gbsw_scoring* sc, const std::vector<BucketPlan>& plan)
{
    // DNA reads the first four scores only
    const size_t sc_bytes = sc->alphabet == GBSW_DNA ? offsetof(gbsw_scoring, matrix) : sizeof(*sc);
    std::string k((const char*)sc, sc_bytes);
    const void* ptrs[] = {ex.bnd.ptr,   ex.queue.ptr,          ex.split_buf.ptr, ex.redo.ptr,       ex.status.ptr,
                          ex.sub.ptr,   ex.lut.ptr,            ex.colmax.ptr,    ex.tables_host.ptr, ex.status_host.ptr,
                          ex.stream};
    k.append((const char*)ptrs, sizeof(ptrs));
    const int opts[] = {ex.streams, ex.f16 ? 1 : 0, (ex.split && !ex.split_misplaced) ? 1 : 0, (int)plan.size()};
    k.append((const char*)opts, sizeof(opts));
    const int64_t jf[] = {job.kmodel, job.n, (int64_t)(uintptr_t)job.order};
    k.append((const char*)jf, sizeof(jf));
    return k + plan_text(plan);
}

// Geometries are chosen for the byte profile of a large alphabet; scores outside int8
// take the int16 profile, in the widest geometry that fits.
int widest_k(const Job& job, bool p8)
{
    return (byte_profile_alphabet(job.alpha) && !p8) ? max_k_for(job.alpha, false) : 1 << 30;
}

// The plan of the batched form for a job and the tables of a scoring (prepare_scoring).
int plan_scored(Exec& ex, const Job& job, const gbsw_scoring* sc, const std::vector<int16_t>& sub, int max_sub, bool p8,
                bool f16p8, SweepChoice& sw, std::vector<BucketPlan>& plan)
{
    // scores of the sweep kernels: bytes where they fit an int8 profile (large alphabets)
    // or have at most three significant bits (small ones), and span 255; else 16 bits
    sw = sweep_choice(sub, job.alpha, sc->gap_open, sc->gap_extend, max_sub,
                      byte_profile_alphabet(job.alpha) ? p8 : f16p8, job.max_cols);
    sw.ok = sw.ok && ex.f16;
    return plan_batched(ex, job, max_sub, p8, sw, table_is_asymmetric(sc, job), widest_k(job, p8), plan);
}

} // namespace

int batched_plan_text(Exec& ex, const Job& job, const gbsw_scoring* sc, std::string* text)
{
    std::vector<int16_t> sub;
    std::vector<BucketPlan> plan;
    int max_sub = 0;
    bool p8 = false, f16p8 = false;
    SweepChoice sw;
    int rc = prepare_scoring(job, sc, sub, &max_sub, &p8, &f16p8);
    if (!rc) rc = plan_scored(ex, job, sc, sub, max_sub, p8, f16p8, sw, plan);
    if (!rc) *text = plan_text(plan);
    return rc;
}

int enqueue_job(Exec& ex, const Job& job, const gbsw_scoring* sc, int mode)
{
    ex.launches.clear();
    ex.graph_state = 0;
    std::vector<int16_t> sub;
    int max_sub = 0;
    bool p8 = false, f16p8 = false;
    int rc = prepare_scoring(job, sc, sub, &max_sub, &p8, &f16p8);
    if (rc) return rc;
    ex.max_sub = max_sub;
    ex.p8 = p8;
    const int kclamp = widest_k(job, p8);
    hipStream_t st0 = ex.stream;
    if (job.n == 0) {
        GBSW_HIP_TRY(hipEventRecord(ex.ev_start, st0));
        GBSW_HIP_TRY(hipEventRecord(ex.ev_stop, st0));
        std::memset(ex.status_host.ptr, 0, sizeof(int32_t) * kStatusWords);
        return GBSW_OK;
    }
    std::vector<int16_t> colmax((size_t)job.alpha, 0);
    for (int c = 0; c < job.alpha; ++c)
        for (int r = 0; r < job.alpha; ++r)
            colmax[(size_t)c] = std::max<int16_t>(colmax[(size_t)c], sub[(size_t)(r * job.alpha + c)]);
    // small tables in pinned memory, read by the preparing launch (the previous job of
    // this Exec has completed, so its staging is free)
    uint8_t* th = ex.tables_host.as<uint8_t>();
    std::memcpy(th, sub.data(), sizeof(int16_t) * sub.size());
    std::memcpy(th + 2048, job.lut_host, 256);
    std::memcpy(th + 2304, colmax.data(), sizeof(int16_t) * colmax.size());
    GBSW_HIP_TRY(ex.redo.reserve(sizeof(int32_t) * (size_t)std::max<int64_t>(1, job.n)));
    KernelArgs a = base_args(ex, job, sc);
    if (mode == GBSW_PLAIN) {
        GBSW_HIP_TRY(hipEventRecord(ex.ev_start, st0));
        GBSW_HIP_TRY(prepare_job(prepare_args(ex, job, sizeof(int16_t) * sub.size()), st0));
        // one geometry for the whole batch, sized by its longest shorter sequence;
        // with profiles (DNA) the occupancy model's narrower strips cost the long
        // pairs more than the extra waves gain (793 vs 593 GCUPS on the 1M-pair
        // DNA mix), so it applies to profile-free alphabets only
        const int K = std::min(kclamp, k_for_cols(job.max_cols, job.alpha,
                                                  byte_profile_alphabet(job.alpha) ? job.kmodel : kModelClassic));
        const int lds = lds_for(K, job.alpha, p8);
        const int64_t nquads = (job.n + kPairsPerWave - 1) / kPairsPerWave;
        a.order = nullptr;
        a.order_n = job.n;
        const int kf = with_profile(kPlainForward, p8), kr = with_profile(kPlainReverse, p8);
        int gf = grid_for(ex, kf, K, lds, nquads);
        int gr = grid_for(ex, kr, K, lds, nquads);
        const size_t per_wg = kPairsPerWave * (size_t)a.bnd_rows * sizeof(uint32_t);
        if (ex.fixed && (size_t)std::max(gf, gr) * per_wg > ex.bnd.bytes) {
            // preallocated scratch: fewer workgroups stride over the quads
            const int cap = (int)std::min<size_t>(ex.bnd.bytes / per_wg, INT_MAX);
            if (cap < 1) return fail(GBSW_E_RANGE, "strip boundary rows exceed the preallocated scratch");
            gf = std::min(gf, cap);
            gr = std::min(gr, cap);
        }
        GBSW_HIP_TRY(ex.bnd.reserve((size_t)std::max(gf, gr) * per_wg));
        rc = launch_timed(ex, st0, kf, K, gf, lds, a, ex.bnd.ptr);
        if (rc) return rc;
        ex.launches.back().pairs = job.n;
        ex.launches.back().cells = job.cells;
        rc = launch_timed(ex, st0, kr, K, gr, lds, a, ex.bnd.ptr);
        if (rc) return rc;
        ex.launches.back().pairs = job.n;
        GBSW_HIP_TRY(hipMemcpyAsync(ex.status_host.ptr, ex.status.ptr, sizeof(int32_t) * kStatusWords,
                                    hipMemcpyDeviceToHost, st0));
        GBSW_HIP_TRY(hipEventRecord(ex.ev_stop, st0));
        return GBSW_OK;
    }
    std::vector<BucketPlan> plan;
    SweepChoice sw;
    rc = plan_scored(ex, job, sc, sub, max_sub, p8, f16p8, sw, plan);
    if (rc) return rc;
    a.base = sw.base;
    a.bias = sw.bias;
    a.shift = sw.shift;
    const size_t sub_bytes = sizeof(int16_t) * sub.size();
    if (!ex.graphs || ex.fixed || !job.graph) {
        GBSW_HIP_TRY(hipEventRecord(ex.ev_start, st0));
        rc = record_batched(ex, job, a, plan, sub_bytes);
        if (rc) return rc;
        GBSW_HIP_TRY(hipEventRecord(ex.ev_stop, st0));
        return GBSW_OK;
    }
    // hipGraph: the stream work of this batch, scoring and options is captured
    // once and replayed (one launch instead of ~20 API calls); the per-launch
    // records of the capture stand for every replay
    JobGraph& G = *job.graph;
    const std::string key = graph_key(ex, job, sc, plan);
    if (!G.exec || G.key != key) {
        G.reset();
        GBSW_HIP_TRY(hipStreamBeginCapture(st0, hipStreamCaptureModeRelaxed));
        rc = record_batched(ex, job, a, plan, sub_bytes);
        hipGraph_t graph = nullptr;
        const hipError_t ce = hipStreamEndCapture(st0, &graph);
        if (rc) {
            if (graph) (void)hipGraphDestroy(graph);
            return rc;
        }
        if (ce != hipSuccess) return fail(GBSW_E_DEVICE, std::string("graph capture: ") + hipGetErrorString(ce));
        const hipError_t ie = hipGraphInstantiate(&G.exec, graph, nullptr, nullptr, 0);
        (void)hipGraphDestroy(graph);
        if (ie != hipSuccess) {
            G.exec = nullptr;
            return fail(GBSW_E_DEVICE, std::string("graph instantiate: ") + hipGetErrorString(ie));
        }
        G.key = key;
        G.launches = ex.launches;
        G.captures += 1;
        ex.graph_state = 1;
    } else {
        ex.graph_state = 2;
    }
    ex.launches = G.launches;
    GBSW_HIP_TRY(hipEventRecord(ex.ev_start, st0));
    GBSW_HIP_TRY(hipGraphLaunch(G.exec, st0));
    GBSW_HIP_TRY(hipEventRecord(ex.ev_stop, st0));
    G.replays += 1;
    return GBSW_OK;
}

namespace {

// The pairs in ex.redo again with int32 cells; blocks, and leaves the status words
// in ex.status_host.
int redo_int32(Exec& ex, const Job& job, const gbsw_scoring* sc, int64_t count)
{
    KernelArgs a = base_args(ex, job, sc);
    a.order = ex.redo.as<int32_t>();
    a.order_n = count;
    a.sat_limit = INT_MAX;
    BucketPlan b;
    b.bk.count = count;
    b.bk.max_cols = job.max_cols;
    b.bk.max_rows = job.max_rows;
    std::vector<int16_t> sub;
    int max_sub = 0;
    bool p8 = false, f16p8 = false;
    int rc = prepare_scoring(job, sc, sub, &max_sub, &p8, &f16p8);
    if (rc) return rc;
    const SweepChoice sw = sweep_choice(sub, job.alpha, sc->gap_open, sc->gap_extend, max_sub, false, job.max_cols);
    if (sw.wide_ok) {
        // One pair per wave; few pairs (up to a wave per SIMD) as strips of the split
        // form: 400 long reads, a few of them past the range, 773 -> 21.5 ms with
        // the few no longer on one 16-lane group each.
        a.base = sw.base;
        int32_geometry(job, kMostInt32, false, b);
        const bool few = count <= 4 * (int64_t)ex.num_cu;
        if (few && b.strips > 1 && ex.split && !ex.split_misplaced && !a.asym) int32_split_geometry(job, b);
    } else {
        int nk = 0;
        const int* wk = wide_k_list(&nk);
        b.K = wk[nk - 1];
        for (int i = 0; i < nk; ++i)
            if (kVirtPerPair * wk[i] >= job.max_cols) { b.K = wk[i]; break; }
        b.kind = with_profile(kBatchedWide, ex.p8);
        b.lds = lds_for(b.K, job.alpha, ex.p8, 8);
    }
    const size_t per_wg = (size_t)b.pairs_per_wave() * (size_t)a.bnd_rows * 8;
    auto set_grid = [&]() {
        if (b.kind & kSplitStrips) {
            const int occ = std::max(1, kernel_occupancy(b.kind, b.K, b.lds));
            const int64_t busy = (b.sets() + kXcds - 1) / kXcds * b.strips * kXcds;
            b.grid = (int)std::max<int64_t>(kXcds, std::min<int64_t>((int64_t)occ * ex.num_cu / kXcds * kXcds, busy));
        } else {
            b.grid = grid_for(ex, b.kind, b.K, b.lds, b.sets());
        }
    };
    set_grid();
    if (ex.fixed && (b.kind & kSplitStrips) &&
        (2 * (size_t)b.grid * per_wg > ex.bnd.bytes || split_words_of(b) * 4 > ex.split_buf.bytes)) {
        b.kind &= ~kSplitStrips;
        set_grid();
    }
    const bool split = (b.kind & kSplitStrips) != 0;
    if (ex.fixed && !split && (size_t)b.grid * per_wg > ex.bnd.bytes) {
        const int cap = (int)std::min<size_t>(ex.bnd.bytes / per_wg, INT_MAX);
        if (cap < 1) return fail(GBSW_E_RANGE, "int32 boundary rows exceed the preallocated scratch");
        b.grid = std::min(b.grid, cap);
    }
    GBSW_HIP_TRY(ex.bnd.reserve((size_t)(split ? 2 : 1) * b.grid * per_wg));
    a.queue = ex.queue.as<uint32_t>();
    GBSW_HIP_TRY(zero_u32(a.queue, kXcds, ex.stream));
    a.kmax = b.K;
    a.nranges = 1;
    a.ranges[0] = {(int32_t)count, b.K};
    if (split) {
        GBSW_HIP_TRY(ex.split_buf.reserve(split_words_of(b) * sizeof(uint32_t)));
        GBSW_HIP_TRY(zero_u32(ex.split_buf.as<uint32_t>(), (int)split_words_of(b), ex.stream));
        if ((rc = set_split_args(ex, b, a))) return rc;
    }
    rc = launch_timed(ex, ex.stream, b.kind, b.K, b.grid, b.lds, a, ex.bnd.ptr);
    if (rc) return rc;
    ex.launches.back().pairs = count;
    GBSW_HIP_TRY(hipMemcpyAsync(ex.status_host.ptr, ex.status.ptr, sizeof(int32_t) * kStatusWords,
                                hipMemcpyDeviceToHost, ex.stream));
    GBSW_HIP_TRY(hipEventRecord(ex.ev_stop, ex.stream));
    GBSW_HIP_TRY(hipEventSynchronize(ex.ev_stop));
    return GBSW_OK;
}

} // namespace

int complete_job(Exec& ex, const Job& job, const gbsw_scoring* sc, double* device_ms)
{
    GBSW_HIP_TRY(hipEventSynchronize(ex.ev_stop));
    ex.late_results = false;
    int32_t* status = ex.status_host.as<int32_t>();
    if (split_rerun_needed(status) && !ex.split_misplaced) {
        // a split launch found workgroups of one XCD counter on different XCCs,
        // so its boundary rows may have been read stale: the whole job again,
        // with the split form off from now on (it is only used in the batched form)
        ex.split_misplaced = true;
        set_error("split form disabled: workgroups of one XCD counter ran on different XCCs");
        int rc = enqueue_job(ex, job, sc, GBSW_BATCHED);
        if (!rc) rc = complete_job(ex, job, sc, device_ms);
        ex.late_results = true;
        return rc;
    }
    if (status[kStatusSaturated] > 0) {
        // pairs whose 16-bit score reached the saturation limit: recompute them
        // (forward + reverse) with int32 cells
        int rc = redo_int32(ex, job, sc, status[kStatusSaturated]);
        if (!rc && split_rerun_needed(status)) {
            // (as above: unsplit from now on; the status words of the first try go)
            ex.split_misplaced = true;
            GBSW_HIP_TRY(zero_u32(ex.status.as<uint32_t>(), kStatusWords, ex.stream));
            const int32_t count = status[kStatusSaturated];
            rc = redo_int32(ex, job, sc, count);
        }
        if (rc) return rc;
        ex.late_results = true;
    }
    float ms = 0.f;
    GBSW_HIP_TRY(hipEventElapsedTime(&ms, ex.ev_start, ex.ev_stop));
    if (device_ms) *device_ms = ms;
    for (size_t i = 0; i < ex.launches.size(); ++i) {
        // events recorded by a graph replay may not carry times: 0 then
        float t = 0.f;
        if (hipEventElapsedTime(&t, ex.kev[2 * i], ex.kev[2 * i + 1]) != hipSuccess) {
            t = 0.f;
            (void)hipGetLastError();
        }
        ex.launches[i].ms = t;
    }
    if (status[kStatusMisplaced]) return fail(GBSW_E_INTERNAL, "split-form placement check failed after an unsplit rerun");
    // a timed-out wait lets every later wait return at once, after which passes
    // may read boundary rows that are not there: report the timeout, not what
    // follows from it
    if (status[kStatusTimeout]) return fail(GBSW_E_INTERNAL, "a split-form wait timed out");
    if (status[kStatusRevMiss]) return fail(GBSW_E_INTERNAL, "reverse pass did not reach the forward score");
    return GBSW_OK;
}

} // namespace gbsw
