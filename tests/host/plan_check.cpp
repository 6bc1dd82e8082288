// plan_check.cpp -- CPU check of the batched form's plan (gbsw_exec.cpp, built into this
// program with stand-ins for the kernels): every set of pairs of every launch has a
// geometry that its kernel holds and that its pairs fit, and the launches cover every
// pair once.  Over the lengths of `kManyRanges`, whose geometries change from class to
// class, and over random mixes of lengths.  Prints "ok", or the first fault.
#include "../../gpu-bsw_amd/csrc/gbsw_exec.cpp"

#include <cstdio>
#include <random>

namespace gbsw {

// stand-ins: one occupancy for every kernel that fits a workgroup's LDS
static int g_occupancy = 16;
int kernel_occupancy(int, int, int lds) { return lds > 65536 ? 0 : std::min(g_occupancy, 163840 / lds); }
bool kernel_has(int kind, int) { return kind != 0; }
static const int kList16[] = {2, 3, 4, 5, 6, 7, 8, 10, 12, 14, 16, 20, 24, 28, 32}, kList32[] = {4, 8, 16};
const int* kernel_k_list(int* n) { *n = 15; return kList16; }
const int* wide_k_list(int* n) { *n = 3; return kList32; }
hipError_t kernel_launch(int, int, int, int, hipStream_t, const KernelArgs&) { return hipErrorUnknown; }
hipError_t prepare_job(const PrepareArgs&, hipStream_t) { return hipErrorUnknown; }
hipError_t zero_u32(uint32_t*, int, hipStream_t) { return hipErrorUnknown; }
hipError_t sort_pairs(void*, size_t&, const uint32_t*, uint32_t*, const int32_t*, int32_t*, int, int, hipStream_t)
{
    return hipErrorUnknown;
}

namespace {

struct Len {
    int32_t rows, cols;
};
const Len kManyRanges[] = {
    {11171, 4248}, {65000, 62287}, {1868, 656}, {5542, 3714}, {6968, 6534}, {60557, 52444}, {8825, 5187},
    {753, 536}, {65000, 30811}, {35047, 31495}, {6676, 4853}, {65000, 30489}, {6014, 2903}, {65000, 59887},
    {4081, 2383}, {39370, 16423}, {65000, 33239}, {1066, 474}, {8633, 3135}, {3277, 1242}, {3802, 1689},
    {64, 23}, {65000, 43207}, {2284, 833}, {531, 296}, {301, 144}};
// Seventeen ranges without the split form (also the pairs of test_gpu_ranges.py).
const Len kUnsplitRanges[] = {
    {5642, 5151}, {5633, 5633}, {4631, 4631}, {4151, 4151}, {3680, 3680}, {3087, 3087}, {2574, 2574}, {2049, 2049},
    {1543, 1543}, {1033, 1033}, {778, 778}, {647, 647}, {514, 514}, {386, 386}, {257, 257}, {130, 130}, {20, 20}};

// A job of these pairs, as batch_fill counts them.
Job job_of(const std::vector<Len>& v, int alphabet, int alpha)
{
    Job j;
    j.alphabet = alphabet;
    j.alpha = alpha;
    j.n = (int64_t)v.size();
    Bucket classes[kClasses], fine[kFineClasses];
    for (const Len& x : v) {
        classes[length_class(x.cols)].add(x.cols, x.rows);
        fine[fine_class(x.cols)].add(x.cols, x.rows);
        j.max_rows = std::max(j.max_rows, x.rows);
        j.max_cols = std::max(j.max_cols, x.cols);
    }
    place_buckets(j.buckets, classes, kClasses);
    place_buckets(j.fine, fine, kFineClasses);
    return j;
}

bool in(int K, const int* a, size_t n) { return std::find(a, a + n, K) != a + n; }

// nullptr, or what is wrong
const char* check(std::vector<Len> v, int alphabet, bool split, bool fixed, int* most_ranges)
{
    const bool dna = alphabet == GBSW_DNA;
    const int alpha = dna ? 4 : 20;
    Job j = job_of(v, alphabet, alpha);
    std::vector<int16_t> sub((size_t)(alpha * alpha), (int16_t)(dna ? -3 : -4));
    for (int c = 0; c < alpha; ++c) sub[(size_t)(c * alpha + c)] = dna ? 3 : 6;
    const int max_sub = dna ? 3 : 6;
    const SweepChoice sw = sweep_choice(sub, alpha, -6, -1, max_sub, true, j.max_cols);
    Exec ex;
    ex.num_cu = 256;
    ex.fixed = fixed;
    std::vector<BucketPlan> plan;
    plan_sweeps(ex, j, sw, split, false, plan);
    // the work order (k_prepare): classes of longer pairs first, then rows
    const bool fine = plan_is_fine(plan);
    std::sort(v.begin(), v.end(), [&](const Len& x, const Len& y) {
        const int a = fine ? fine_class(x.cols) : length_class(x.cols), b = fine ? fine_class(y.cols) : length_class(y.cols);
        return a != b ? a > b : x.rows > y.rows;
    });
    std::vector<int> taken(v.size(), 0);
    for (const BucketPlan& b : plan) {
        *most_ranges = std::max(*most_ranges, (int)b.ranges.size());
        if (b.ranges.empty() || b.ranges.size() > (size_t)kMaxRanges) return "a launch has more ranges than its arguments hold";
        const bool pairs = (b.kind & kHalfPairs) != 0, strips = plan_is_split(b), wide32 = (b.kind & 0xFF) == kBatchedWide;
        const int PW = pairs ? 8 : b.pairs_per_wave();
        for (int64_t q = 0; q * PW < b.bk.count; ++q) {
            // as the kernels choose (a split launch has one geometry)
            int K = 0;
            for (size_t r = b.ranges.size(); r-- > 0;)
                if (q * PW < b.ranges[r].end) K = b.ranges[r].K;
            if (strips && K != b.K) return "a split launch has two geometries";
            const int k32[] = {2, 4}, kp[] = {2, 3, 4, 5, 6, 7, 8, 9, 10, 11, 12, 13, 14, 15, 16};
            const bool held = wide32 ? in(K, k32, 2)
                              : strips ? in(K, kSweepSplitK, std::size(kSweepSplitK))
                              : pairs  ? in(K, kp, std::size(kp)) && (K > kPairsNarrowMax) == ((b.kind & kWideLanes) != 0)
                              : b.G == kWave ? in(K, kSweepK64, std::size(kSweepK64))
                                             : in(K, kSweepK16, std::size(kSweepK16)) &&
                                                   (K > kSweepNarrowMax) == ((b.kind & kWideLanes) != 0);
            if (!held) return "a set without a geometry of its kernel";
            if (K > b.K) return "a geometry wider than the launch's LDS";
            for (int64_t x = q * PW; x < std::min((q + 1) * PW, b.bk.count); ++x) {
                const Len& l = v[(size_t)(b.bk.begin + x)];
                const int lanes = pairs ? kLanesPerPair : 2 * b.G;
                if (l.rows > b.bk.max_rows) return "a pair of more rows than the launch has boundary rows for";
                if ((pairs || b.G != kWave) && l.cols > lanes * K) return "a pair wider than its one strip";
                if (b.G == kWave && (l.cols + lanes * K - 1) / (lanes * K) > std::max(1, b.strips))
                    return "a pair of more strips than the launch has boundary rows for";
                ++taken[(size_t)(b.bk.begin + x)];
            }
        }
    }
    for (int t : taken)
        if (t != 1) return "a pair in no launch, or in two";
    return nullptr;
}

// Pairs that a plan puts on int32 cells at once: a table's mean identical and mean other
// score, the rest of the diagonal alike but for one code of `rare`.
int64_t int32_pairs(const std::vector<Len>& v, int alphabet, int alpha, int16_t same, int16_t other, int16_t rare)
{
    Job j = job_of(v, alphabet, alpha);
    std::vector<int16_t> sub((size_t)(alpha * alpha), other);
    for (int c = 0; c < alpha; ++c) sub[(size_t)(c * alpha + c)] = same;
    sub[0] = rare;
    Exec ex;
    ex.num_cu = 256;
    std::vector<BucketPlan> plan;
    plan_sweeps(ex, j, sweep_choice(sub, alpha, -6, -1, std::max(same, rare), true, j.max_cols), true, false, plan);
    int64_t n = 0;
    for (const BucketPlan& b : plan)
        if ((b.kind & 0xFF) == kBatchedWide) n += b.bk.count;
    return n;
}

// A serving slot of `bnd_bytes` of boundary rows and a scoring of the int16 kernels:
// the job is planned, not refused.
const char* check_slot(const std::vector<Len>& v, int alphabet, size_t bnd_bytes)
{
    const int alpha = alphabet == GBSW_DNA ? 5 : 24;
    Job j = job_of(v, alphabet, alpha);
    Exec ex;
    ex.num_cu = 256;
    ex.fixed = true;
    // (views: sizes count, nothing is read or written)
    ex.bnd.view((void*)256, bnd_bytes);
    ex.queue.view((void*)256, 4 * kXcds * 64);
    ex.split_buf.view((void*)256, (size_t)1 << 30);
    SweepChoice sw;
    sw.ok = false;
    std::vector<BucketPlan> plan;
    if (plan_batched(ex, j, 3, alphabet == GBSW_PROTEIN, sw, false, 1 << 30, plan)) return last_error_text();
    size_t end = 0;
    int64_t pairs = 0;
    for (const BucketPlan& b : plan) {
        const size_t rows = 4 * (size_t)kPairsPerWave * (size_t)b.bk.max_rows * (size_t)b.grid * (plan_is_split(b) ? 2 : 1);
        if (b.grid < 1) return "an empty grid";
        if (b.strips > 1) end = std::max(end, 4 * b.bnd_at + rows);
        if ((b.bk.max_cols + kVirtPerPair * b.K - 1) / (kVirtPerPair * b.K) > b.strips) return "more strips than planned";
        pairs += b.bk.count;
    }
    if (end > bnd_bytes) return "boundary rows past the slot's";
    if (pairs != j.n) return "not every pair in a launch";
    return nullptr;
}

} // namespace
} // namespace gbsw

int main()
{
    using namespace gbsw;
    int most = 0;
    auto run = [&](const std::vector<Len>& v, int alphabet, const char* what) {
        for (int split = 0; split < 2; ++split)
            for (int fixed = 0; fixed < 2; ++fixed) {
                const char* e = check(v, alphabet, split != 0, fixed != 0, &most);
                if (e) {
                    std::printf("%s: alphabet %d split %d fixed %d pairs %zu: %s\n", what, alphabet, split, fixed, v.size(), e);
                    return false;
                }
            }
        return true;
    };
    for (int occ : {12, 16, 32}) {
        g_occupancy = occ;
        if (!run({std::begin(kManyRanges), std::end(kManyRanges)}, GBSW_DNA, "many ranges")) return 1;
        if (!run({std::begin(kUnsplitRanges), std::end(kUnsplitRanges)}, GBSW_DNA, "many ranges, unsplit")) return 1;
    }
    if (most < 17) {
        std::printf("the lists no longer take more than 16 ranges in one launch (%d)\n", most);
        return 1;
    }
    g_occupancy = 16;
    // 20 to 300 proteins of up to 4,096 columns stay in 16 bits though one residue scores 11
    // with itself (identical ones of 4,096 score about 22,000); ten of 8,000 do not, nor do
    // ten reads of 16,000 at +3/-3
    for (int n : {20, 100, 300}) {
        std::vector<Len> v;
        for (int x = 0; x < n; ++x) v.push_back({8000, 1024 + 3072 * x / (n - 1)});
        if (const int64_t k = int32_pairs(v, GBSW_PROTEIN, 20, 5, -1, 11)) {
            std::printf("%d of %d proteins on int32 cells\n", (int)k, n);
            return 1;
        }
    }
    {
        std::vector<Len> aa(10, Len{9000, 8000}), reads(10, Len{20000, 16000});
        for (int x = 0; x < 50; ++x) {
            aa.push_back({3000, 2000});
            reads.push_back({6000, 4000});
        }
        if (int32_pairs(aa, GBSW_PROTEIN, 20, 5, -1, 11) != 10 || int32_pairs(reads, GBSW_DNA, 4, 3, -3, 3) != 10) {
            std::printf("pairs that pass the 16-bit range not on int32 cells\n");
            return 1;
        }
    }
    std::mt19937 rng(5);
    auto real = [&]() { return std::uniform_real_distribution<double>(0.0, 1.0)(rng); };
    for (int mix = 0; mix < 3000; ++mix) {
        const int n = mix % 300 == 0 ? 20000 : (int)std::exp(std::log(300.0) * real());
        const double lo = std::log(1 + 100 * real()), hi = std::log(200 + 64800 * real() * real());
        std::vector<Len> v;
        for (int x = 0; x < n; ++x) {
            const int c = (int)std::exp(lo + (hi - lo) * real());
            v.push_back({std::min(65000, (int)(c * (1 + 3 * real() * real()))), std::max(0, c - (mix % 7 == 0 && x == 0 ? c : 0))});
        }
        // (4 x 65,000 x 4: the least a server takes)
        if (const char* e = check_slot(v, mix & 1, (size_t)4 * 65000 * 4)) {
            std::printf("a slot of the least boundary rows, pairs %zu: %s\n", v.size(), e);
            return 1;
        }
        if (!run(v, mix & 1 ? GBSW_PROTEIN : GBSW_DNA, "random mix")) return 1;
    }
    std::printf("ok\n");
    return 0;
}
