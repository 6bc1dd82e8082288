// gbsw_kernels.hpp -- host-visible entry points of gbsw_kernels.hip.
#pragma once
#include <hip/hip_runtime.h>

#include "gbsw_kernel_args.hpp"

namespace gbsw {

enum KernelKind {
    kPlainForward = 0,
    kPlainReverse = 1,
    kBatched = 2,
    kBatchedWide = 3,
    kBatchedF16 = 4, // k_sweep: 16-bit cells, f16 maxima
    kSplit = 5,    // k_split, int16 cells
    kSplitF16 = 6, // k_sweep_split
};
// Flag on a kind: the scores are held as bytes (profile or register tables).
constexpr int kByteProfile = 0x100;
inline int with_profile(int kind, bool bytes8) { return bytes8 ? (kind | kByteProfile) : kind; }

// The sweep kernels (gbsw_sweep.hpp) are kBatchedF16 and kSplitF16 with these
// flags.  kRegTables: the scores of a lane's columns in registers (at most
// kRegAlpha residue codes) instead of a profile in LDS.  kWideGroup: one pair per
// wave (64 lanes) instead of four (16 lanes each).  kWideLanes: the four-pair
// kernel of the wide geometries (K from 10).  A kernel without kSplitF16 holds
// every geometry of its list; a split one is compiled per K.
constexpr int kWideGroup = 0x200;
constexpr int kRegTables = 0x400;
constexpr int kWideLanes = 0x800;
constexpr int kHalfPairs = 0x2000; // eight pairs per wave, one in each half of 16 lanes' registers
constexpr int kShifted = 0x4000;   // byte tables hold the scores from the smallest one up
constexpr int kReportedKind = 0x1FF; // the part of a kind that launch statistics report
constexpr int kReportedPairs = 7;     // and for eight pairs per wave
inline int sweep_kind(int kind, int form, int flags)
{
    kind |= flags;
    return form == kProfRegs ? kind | kByteProfile | kRegTables : form == kProfBytes ? kind | kByteProfile : kind;
}
// Geometries of the sweep kernels.
#define GBSW_SWEEP_K16(X) X(2) X(3) X(4) X(5) X(6) X(7) X(8)
#define GBSW_SWEEP_K16_WIDE(X) X(10) X(12) X(14) X(16)
#define GBSW_SWEEP_PAIRS(X) X(2) X(3) X(4) X(5) X(6) X(7) X(8) X(9) X(10)
#define GBSW_SWEEP_PAIRS_WIDE(X) X(11) X(12) X(13) X(14) X(15) X(16)
constexpr int kPairsNarrowMax = 10;
#define GBSW_SWEEP_K64(X) X(1) X(2) X(3) X(4) X(5) X(6) X(8)
#define GBSW_SWEEP_K64_SPLIT(X) X(1) X(2) X(3) X(4) X(6) X(8)
// kernel of a form, nullptr where it is not compiled (gbsw_sweep_*.hip)
const void* sweep_kernel_regs(int kind, int K);
const void* sweep_kernel_bytes(int kind, int K);
const void* sweep_kernel_words(int kind, int K);
const void* sweep_kernel_regs_wide(int kind, int K);
const void* sweep_kernel_bytes_wide(int kind, int K);
const void* sweep_kernel_words_wide(int kind, int K);
const void* sweep_kernel_pairs(int kind);
const void* sweep_kernel_shifted(int kind);
const void* sweep_kernel_shifted_wide(int kind, int K);
// int32 cells (kBatchedWide | kWideGroup, with kSplitStrips the split form)
constexpr int kSplitStrips = 0x1000;
#define GBSW_SWEEP_K32(X) X(2) X(4)
const void* sweep_kernel_int32(int kind, int K);

bool kernel_has(int kind, int K);
const int* kernel_k_list(int* count); // K values with compiled kernels, ascending
const int* wide_k_list(int* count);   // K values of the int32 (kBatchedWide) kernel
int kernel_occupancy(int kind, int K, int lds_bytes);
hipError_t kernel_launch(int kind, int K, int grid, int lds_bytes, hipStream_t stream, const KernelArgs& args);
hipError_t zero_u32(uint32_t* p, int n, hipStream_t stream);

// gbsw_binning.hip
// Work of the launch that precedes a job's kernels.
constexpr int kSmallSort = 16384; // pairs sorted by one workgroup
struct PrepareArgs {
    const uint64_t* ref_off;
    const uint64_t* qry_off;
    int64_t n;
    int32_t* order;          // not null: the work order of n <= kSmallSort pairs
    uint32_t* keys;          // else, not null: sort keys and
    int32_t* vals;           // pair indices of the n pairs
    const int16_t* h_sub;    // tables in pinned host memory, and their device copies
    const uint8_t* h_lut;
    const int16_t* h_colmax;
    int16_t* sub;
    uint8_t* lut;
    int16_t* colmax;
    uint32_t* status;        // cleared: status, queues, split bookkeeping
    uint32_t* queue;
    uint32_t* split;
    int64_t nsplit;
    int32_t nsub, alpha, nstatus, nqueue;
    int32_t fine;            // keys by fine classes (not with `order`)
    int32_t helpers;         // workgroups for tables and clearing (set by prepare_job)
};
hipError_t prepare_job(const PrepareArgs& a, hipStream_t stream);
// Sets of byte values in p[0, n) and p2[0, n2) (16-byte aligned): eight mask words per
// workgroup of up to kPresenceBlocks, in pinned host memory.
constexpr int kPresenceBlocks = 128;
hipError_t byte_presence(const uint8_t* p, uint64_t n, const uint8_t* p2, uint64_t n2, uint32_t* masks,
                         hipStream_t stream);
hipError_t sort_pairs(void* temp, size_t& temp_bytes, const uint32_t* kin, uint32_t* kout, const int32_t* vin,
                      int32_t* vout, int n, int end_bit, hipStream_t stream);

// gbsw_gather.hip: one tile = 1..kGatherTileBytes bytes of one request part,
// copied from src to dst; part_flags[part] |= 1 when a byte has accept[byte] == 0.
constexpr uint32_t kGatherTileBytes = 32768;
struct GatherTile {
    const uint8_t* src; // device-readable pinned host memory
    uint8_t* dst;       // device memory
    uint32_t len;
    int32_t part;
};
hipError_t gather(const GatherTile* tiles, int ntiles, const uint8_t* accept, int32_t* part_flags,
                  hipStream_t stream);


// gbsw_traceback.hip: alignment paths of aligned pairs.
struct TbArgs {
    const uint8_t* ref;
    const uint8_t* qry;
    const uint64_t* ref_off;
    const uint64_t* qry_off;
    const int32_t* out;     // results, 5 x n (score, ref_begin, ref_end, query_begin, query_end)
    int64_t n;
    const uint8_t* lut;     // byte -> residue code
    const int16_t* sub;     // alpha x alpha, s(row code, column code)
    int32_t alpha;
    int32_t gap_open, gap_extend;
    int32_t max_sub;        // largest substitution score, at least 0
    int32_t base;           // added to every 16-bit cell value (none is negative then)
    int32_t kmax;           // most columns per lane (tb_kmax)
    const int32_t* order;   // pairs by position, largest first
    int64_t p0, count;      // the launch's positions
    uint32_t* queue;        // sets taken (0 at launch)
    uint8_t* dir;           // scratch of region_bytes per workgroup: path bits, boundary columns
    int64_t region_bytes;
    const int64_t* cap_off; // per pair: offset of its run capacity (rows + columns) in runs
    uint32_t* runs;         // run-length ops, last run first
    int32_t* nruns;         // per pair: runs written (n + 1 entries, the last 0)
    int32_t* path_score;    // per pair: score of the path
};
// Classes of pairs by rows x columns (two per factor of two), and what k_tb_keys finds
// in each; counters of the launches.
constexpr int kTbAreas = 128, kTbKeyBits = 21, kTbLaunches = 64;
struct TbCounts {
    uint32_t pairs[kTbAreas], value[kTbAreas], rows[kTbAreas], cols[kTbAreas];
    uint32_t scratch[2][kTbAreas]; // of one pair, in 256 bytes (16 and 64 lanes)
    uint32_t span, bad;            // largest rows + columns; a pair with an empty rectangle
    uint32_t queue[kTbLaunches];
};
// Cells: 16 bits with values below 7,936 (maxima through f16 patterns) or 16,384, 32 bits.
enum { kTbCells16 = 0, kTbCells16Wide = 1, kTbCells32 = 2 };
constexpr int64_t kTbTop16 = 7936, kTbTop16Wide = 16384;
// Columns per lane at most.
int tb_kmax(int cells, int form);
// Scratch of a set of `groups` pairs of pairs with rectangles up to rows x cols, in any
// geometry it may take; the set's work; LDS and resident workgroups of a kernel.
int64_t tb_region_bytes(int32_t rows, int32_t cols, int G, int kmax, int cells, int groups);
double tb_set_cost(int32_t rows, int32_t cols, int G, int kmax);
int tb_lds_bytes(int cells, int G, int form, int kmax, int alpha);
int tb_occupancy(int cells, int G, int form, int lds);
// Per pair its order key, index and run capacity; class counts (counts: zero before).
hipError_t tb_keys(const TbArgs& a, uint32_t* keys, int32_t* vals, int64_t* cap, TbCounts* counts, hipStream_t stream);
// Paths of the pairs at positions p0 .. p0 + count - 1 of `order`.
hipError_t tb_launch(const TbArgs& a, int cells, int G, int form, int grid, int lds, hipStream_t stream);
// Exclusive sums of n entries (temp == nullptr: only the scratch size).
hipError_t tb_scan(void* temp, size_t& temp_bytes, const int64_t* in, int64_t* out, int64_t n, hipStream_t stream);
hipError_t tb_scan(void* temp, size_t& temp_bytes, const int32_t* in, int64_t* out, int64_t n, hipStream_t stream);
// dst[dst_off[p] ...] = runs of pair p in path order.
hipError_t tb_compact(const uint32_t* runs, const int64_t* cap_off, const int32_t* nruns, const int64_t* dst_off,
                      uint32_t* dst, int64_t n, hipStream_t stream);

} // namespace gbsw
