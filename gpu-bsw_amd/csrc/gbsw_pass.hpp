// gbsw_pass.hpp -- device code shared by the alignment kernels: the tasks of the
// forward and reverse passes, the decoding of their winner keys, and the waits of
// the split forms.  G is the number of lanes that align one pair (a "group").
#pragma once
#include "gbsw_device.hpp"
#include "gbsw_kernel_args.hpp"

namespace gbsw {

// One pass (forward or reverse) of one pair, identical in the lanes of a group.
struct Task {
    const uint8_t* rows;      // row sequence (the longer one of this pass)
    const uint8_t* cols;      // column sequence
    int32_t nr, nc;           // rows / columns computed
    int32_t nr_full, nc_full; // extents the reversed indices count back from
    int32_t rev;              // 1: both sequences are read backwards (reverse pass)
    int32_t ubound;           // reverse pass: upper bound of the columns' substitution scores together
};

__device__ __forceinline__ uint32_t inv_prio(uint32_t p)
{
    // tie_prio is a per-1024-block bit-reversal of two 5-bit fields: its own inverse.
    return tie_prio(p);
}

// Max over K registers with ceil((K - 1) / 2) three-input maxima: a queue, each
// maximum takes the three oldest entries and appends its result (depth about
// log3 K).  Op j reads entries 3j .. 3j + 2 of the queue, which then holds
// K - 2j entries; only a last op with two entries left is a two-input maximum.
template <class A, int K>
__device__ __forceinline__ typename A::V tree_max(const typename A::V (&h)[K])
{
    constexpr int NOPS = (K - 1 + 1) / 2;
    typename A::V q[K + NOPS];
#pragma unroll
    for (int k = 0; k < K; ++k) q[k] = h[k];
#pragma unroll
    for (int j = 0; j < NOPS; ++j)
        q[K + j] = (K - 2 * j >= 3) ? A::vmax3(q[3 * j], q[3 * j + 1], q[3 * j + 2]) : A::vmax(q[3 * j], q[3 * j + 1]);
    return q[K + NOPS - 1];
}

// Bits 0 .. n-1 set (n clamped to [0, 16]): the columns of a block inside the pair.
__device__ __forceinline__ uint32_t cols_mask(int n)
{
    return n <= 0 ? 0u : n >= 16 ? 0xFFFFu : (1u << n) - 1u;
}

struct PassResult {
    uint64_t key; // 0: no cell reached a positive score (forward) / the target (reverse)
};

// A pass runs for every group of the wave at once.  All loops are wave-uniform;
// a group whose pair is shorter keeps computing on padding rows and columns,
// which can neither exceed nor (by row/column order) win over its real cells.
//
// Forward key: (score << 40) | ((2^20-1-row) << 20) | (2^20-1-prio(col)), max wins.
// Reverse key: ((2^20-1-col) << 20) | (2^20-1-row), max wins (target = score).
// One strip of the split form: its boundary input (the previous strip's rows,
// with that slot's progress word) and output.
struct StripIO {
    int strip;
    const void* bnd_in;
    void* bnd_out;
    const uint64_t* prog_in;
    uint64_t* prog_out;
    uint64_t epoch_in, epoch_out; // epoch << 32
};

// Wave-uniform wait until *w >= target.  Bounded: after kSpinTicks the timeout
// status word is set and the wave goes on (the host then reports the batch as
// failed), and once that word is set every wait returns at once, so a stalled
// pipeline drains instead of timing out wait by wait.
template <class T>
__device__ __forceinline__ void wait_at_least(const T* w, T target, int32_t* status)
{
    const uint64_t t0 = __builtin_amdgcn_s_memrealtime();
    for (;;) {
        uint64_t v = 0;
        int32_t stop = 0;
        if (threadIdx.x == 0) {
            v = (uint64_t)__hip_atomic_load(w, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            stop = __hip_atomic_load(status + kStatusTimeout, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        const uint32_t lo = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)v);
        const uint32_t hi = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(v >> 32));
        if ((((uint64_t)hi << 32) | lo) >= (uint64_t)target) break;
        if (__builtin_amdgcn_readfirstlane(stop) != 0) break;
        if (__builtin_amdgcn_s_memrealtime() - t0 > kSpinTicks) {
            if (threadIdx.x == 0) atomicOr(status + kStatusTimeout, 1);
            break;
        }
        __builtin_amdgcn_s_sleep(2);
    }
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
}
// Per 16-lane group: wait until the group's word *w >= target (no wait where w
// is null) and return it (target where w is null).  Bounded like wait_at_least.
__device__ __forceinline__ uint32_t wait_group_u32(const uint32_t* w, uint32_t target, int32_t* status)
{
    const uint64_t t0 = __builtin_amdgcn_s_memrealtime();
    uint32_t v = target;
    for (;;) {
        if (w) v = __hip_atomic_load(w, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (__ballot(v < target) == 0) break;
        int32_t stop = 0;
        if (threadIdx.x == 0) stop = __hip_atomic_load(status + kStatusTimeout, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (__builtin_amdgcn_readfirstlane(stop) != 0) break;
        if (__builtin_amdgcn_s_memrealtime() - t0 > kSpinTicks) {
            if (threadIdx.x == 0) atomicOr(status + kStatusTimeout, 1);
            break;
        }
        __builtin_amdgcn_s_sleep(2);
    }
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
    return v;
}
__device__ __forceinline__ void wait_word(const uint64_t* w, uint64_t target, int32_t* status)
{
    wait_at_least<uint64_t>(w, target, status);
}
__device__ __forceinline__ void wait_u32(const uint32_t* w, uint32_t target, int32_t* status)
{
    wait_at_least<uint32_t>(w, target, status);
}

// The wave's earlier global stores and atomics have completed (reached L2),
// then *w = v.  Readers on the same XCD see the stores once they see v.
__device__ __forceinline__ void publish_word(uint64_t* w, uint64_t v)
{
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    if (threadIdx.x == 0) __hip_atomic_store(w, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Every workgroup of split counter x must share one XCC (its L2): record this
// one's, and flag the job for an unsplit rerun when they differ.
__device__ __forceinline__ void split_check_placement(const SplitArgs& sp, int x, int32_t* status)
{
    if (threadIdx.x == 0) {
        const uint32_t xcc = (uint32_t)__builtin_amdgcn_s_getreg(kXccIdReg) & 15u;
        const uint32_t prev = atomicCAS(sp.xcc + x, 0u, xcc + 1u);
        if (!placement_consistent(prev, xcc)) {
            // the results of this job are void: let every wait return at once
            atomicOr(status + kStatusMisplaced, 1);
            atomicOr(status + kStatusTimeout, 1);
        }
    }
}

struct FwdOut {
    int32_t score, ref_end, query_end;
};

__device__ __forceinline__ Task empty_task(const KernelArgs& a, int rev)
{
    Task t;
    t.rows = a.ref; t.cols = a.qry;
    t.nr = t.nc = t.nr_full = t.nc_full = 0;
    t.rev = rev;
    t.ubound = 0;
    return t;
}

__device__ __forceinline__ Task forward_task(const KernelArgs& a, int64_t p)
{
    if (p < 0) return empty_task(a, 0);
    Task t;
    t.rev = 0;
    t.ubound = 0;
    const uint8_t* A = a.ref + a.ref_off[p];
    const uint8_t* B = a.qry + a.qry_off[p];
    const int32_t la = (int32_t)(a.ref_off[p + 1] - a.ref_off[p]);
    const int32_t lb = (int32_t)(a.qry_off[p + 1] - a.qry_off[p]);
    if (la < lb) { t.rows = B; t.nr = lb; t.cols = A; t.nc = la; } // kernel.cpp:248-253
    else { t.rows = A; t.nr = la; t.cols = B; t.nc = lb; }
    t.nr_full = t.nr;
    t.nc_full = t.nc;
    return t;
}

// Decodes the forward key.  A score at or above sat_limit may have saturated the
// int16 cells: the pair is queued for the int32 kernel (when record_redo) and
// reported as score -1.
template <int G = kLanesPerPair>
__device__ __forceinline__ FwdOut forward_result(const KernelArgs& a, int64_t p, uint64_t key, bool record_redo = true)
{
    FwdOut o{0, 0, 0};
    if (p < 0 || key == 0) return o;
    const int32_t la = (int32_t)(a.ref_off[p + 1] - a.ref_off[p]);
    const int32_t lb = (int32_t)(a.qry_off[p + 1] - a.qry_off[p]);
    const int32_t score = (int32_t)(key >> 40);
    const int32_t row = (int32_t)(0xFFFFFu - (uint32_t)((key >> 20) & 0xFFFFFu));
    const int32_t col = (int32_t)inv_prio(0xFFFFFu - (uint32_t)(key & 0xFFFFFu));
    if (score >= a.sat_limit) {
        if (record_redo && (threadIdx.x & (G - 1)) == 0) {
            const int32_t slot = atomicAdd(a.status + kStatusSaturated, 1);
            a.redo[slot] = (int32_t)p;
        }
        o.score = -1;
        return o;
    }
    o.score = score;
    if (la < lb) { o.query_end = row + 1; o.ref_end = col + 1; } // kernel.cpp:381-386
    else { o.ref_end = row + 1; o.query_end = col + 1; }        // kernel.cpp:387-392
    return o;
}

// Sum over the forward column prefix of each residue's best possible score: an
// upper bound of the substitution part of any alignment inside the prefix.
template <int G = kLanesPerPair, class S>
__device__ __forceinline__ int32_t column_bound(const KernelArgs& a, const S& sm, int64_t p, const FwdOut& f)
{
    const int l = threadIdx.x & (G - 1);
    int32_t u = 0;
    if (p >= 0 && f.score > 0) {
        const int32_t la = (int32_t)(a.ref_off[p + 1] - a.ref_off[p]);
        const int32_t lb = (int32_t)(a.qry_off[p + 1] - a.qry_off[p]);
        const bool ref_rows = !(la < lb);
        const uint8_t* C = ref_rows ? a.qry + a.qry_off[p] : a.ref + a.ref_off[p];
        const int32_t ec = ref_rows ? f.query_end : f.ref_end;
        const uint8_t* lut = sm.lut();
        const int16_t* cm = sm.colmax();
        for (int32_t j = l; j < ec; j += G) {
            const int code = lut[C[j]];
            u += code < a.alpha ? (int32_t)cm[code] : 0;
        }
    }
#pragma unroll
    for (int o = G / 2; o > 0; o >>= 1) u += __shfl_xor(u, o, G);
    return u;
}

// Reverse pass on the prefixes A[0:ref_end) x B[0:query_end), read backwards;
// orientation by the two end coordinates as in kernel.cpp:444-459.
//
// Exact extent bound: the forward winner has the smallest row R* among all cells
// scoring S, so every score-S alignment inside the prefixes ends on R*, i.e. at
// index 0 of the reversed forward-row sequence.  Such an alignment uses at most
// ec columns on the diagonal and its vertical gaps cost at least gap_min per
// position, so it spans at most ec + (U - S) / gap_min forward-row positions,
// with U = column_bound.  Cells farther along that axis cannot reach S, and
// cells nearer do not depend on them, so the pass stops there.
__device__ __forceinline__ Task reverse_task(const KernelArgs& a, int64_t p, const FwdOut& f, int32_t ubound)
{
    if (p < 0 || f.score <= 0) return empty_task(a, 1);
    Task t;
    t.rev = 1;
    t.ubound = ubound;
    const uint8_t* A = a.ref + a.ref_off[p];
    const uint8_t* B = a.qry + a.qry_off[p];
    const bool rev_rows_a = !(f.ref_end < f.query_end);
    if (!rev_rows_a) { t.rows = B; t.nr = f.query_end; t.cols = A; t.nc = f.ref_end; } // 444-451
    else { t.rows = A; t.nr = f.ref_end; t.cols = B; t.nc = f.query_end; }            // 452-459
    t.nr_full = t.nr;
    t.nc_full = t.nc;
    if (a.gap_min > 0) {
        const int32_t la = (int32_t)(a.ref_off[p + 1] - a.ref_off[p]);
        const int32_t lb = (int32_t)(a.qry_off[p + 1] - a.qry_off[p]);
        const bool fwd_rows_a = !(la < lb);
        const int32_t ec = fwd_rows_a ? f.query_end : f.ref_end;
        const int64_t span = (int64_t)ec + (int64_t)max(0, ubound - f.score) / a.gap_min;
        const int32_t lim = (int32_t)min<int64_t>(span, 0x7FFFFFFF);
        if (rev_rows_a == fwd_rows_a) t.nr = min(t.nr, lim);
        else t.nc = min(t.nc, lim);
    }
    return t;
}

// The reverse pass takes the other sequence as rows than the forward pass
// (kernel.cpp:248-259 decide by the full lengths, 444-459 by the end coordinates).
__device__ __forceinline__ bool reverse_swaps(const KernelArgs& a, int64_t p, const FwdOut& f)
{
    const int32_t la = (int32_t)(a.ref_off[p + 1] - a.ref_off[p]);
    const int32_t lb = (int32_t)(a.qry_off[p + 1] - a.qry_off[p]);
    return !(la < lb) != !(f.ref_end < f.query_end);
}

// The whole reversed prefix box A[0:ref_end) x B[0:query_end), no extent bound.
__device__ __forceinline__ Task reverse_task_full(const KernelArgs& a, int64_t p, const FwdOut& f)
{
    Task t;
    t.rev = 1;
    t.ubound = 0;
    const uint8_t* A = a.ref + a.ref_off[p];
    const uint8_t* B = a.qry + a.qry_off[p];
    if (f.ref_end < f.query_end) { t.rows = B; t.nr = f.query_end; t.cols = A; t.nc = f.ref_end; } // 444-451
    else { t.rows = A; t.nr = f.ref_end; t.cols = B; t.nc = f.query_end; }                        // 452-459
    t.nr_full = t.nr;
    t.nc_full = t.nc;
    return t;
}

// Reverse target of a pair.  With a symmetric table, or an asymmetric one whose
// reverse pass keeps the forward orientation, the reversed prefix box holds the
// same alignments with the same scores, so its maximum is the forward score S
// and the extent bound applies.  With an asymmetric table and the orientation
// swapped, the reverse DP scores the transposed table and its maximum (which
// decides the begins, kernel.cpp:1021-1030, 3-45) is found first, by a
// forward-style pass over the whole reversed box (run by the kernels through
// their one forward-pass call site, so that no second copy of the pass is
// inlined).  A target of 0 gives begins (0, 0), the reference's initial
// per-thread coordinates.
struct RevPlan {
    Task t;
    int32_t target;
    bool gen;       // this group's pair needs the maximum of its reversed box first
    bool saturated; // that maximum may have saturated int16: recomputed with int32
};
template <int G = kLanesPerPair, class S>
__device__ __forceinline__ RevPlan reverse_plan(const KernelArgs& a, const S& sm, int64_t p, const FwdOut& f)
{
    RevPlan r;
    r.t = reverse_task(a, p, f, column_bound<G>(a, sm, p, f));
    r.target = f.score;
    r.gen = a.asym && p >= 0 && f.score > 0 && reverse_swaps(a, p, f);
    r.saturated = false;
    if (r.gen) r.t = reverse_task_full(a, p, f);
    return r;
}
// The forward-style pass over the reversed box (r.t, or an empty task for
// groups that do not need it) returned `key`: its score is the target.
template <int G = kLanesPerPair>
__device__ __forceinline__ void reverse_plan_finish(const KernelArgs& a, int64_t p, uint64_t key, RevPlan& r)
{
    if (!r.gen) return;
    r.target = (int32_t)(key >> 40);
    if (r.target <= 0) r.t = empty_task(a, 1);
    if (r.target >= a.sat_limit) {
        r.saturated = true;
        r.target = 0; // (nothing to reach in this pass)
        r.t = empty_task(a, 1);
        if ((threadIdx.x & (G - 1)) == 0) {
            const int32_t slot = atomicAdd(a.status + kStatusSaturated, 1);
            a.redo[slot] = (int32_t)p;
        }
    }
}

__device__ __forceinline__ void reverse_result(const KernelArgs& a, int64_t p, const FwdOut& f, const Task& t,
                                               int32_t target, uint64_t key, int32_t* ref_begin, int32_t* query_begin)
{
    *ref_begin = 0;
    *query_begin = 0;
    if (p < 0 || f.score <= 0 || target <= 0) return;
    if (key == 0) { atomicOr(a.status + kStatusRevMiss, 1); return; }
    const int32_t col = (int32_t)(0xFFFFFu - (uint32_t)((key >> 20) & 0xFFFFFu));
    const int32_t row = (int32_t)(0xFFFFFu - (uint32_t)(key & 0xFFFFFu));
    const int32_t orow = t.nr_full - 1 - row; // kernel.cpp:579
    const int32_t ocol = t.nc_full - 1 - col; // kernel.cpp:580
    if (f.ref_end < f.query_end) { *query_begin = orow; *ref_begin = ocol; } // 591-595
    else { *ref_begin = orow; *query_begin = ocol; }                       // 596-600
}

// Byte->code table, substitution scores and column maxima into LDS.
template <class S>
__device__ __forceinline__ void stage_tables(const KernelArgs& a, const S& sm)
{
    for (int i = threadIdx.x; i < 256; i += kWave) sm.lut()[i] = a.lut[i];
    for (int i = threadIdx.x; i < a.alpha * a.alpha; i += kWave) sm.sub()[i] = a.sub[i];
    for (int i = threadIdx.x; i < a.alpha; i += kWave) sm.colmax()[i] = a.colmax[i];
    __syncthreads();
}

__device__ __forceinline__ int64_t slot_pair(const KernelArgs& a, int64_t slot)
{
    if (slot >= a.order_n) return -1;
    return a.order ? (int64_t)a.order[slot] : slot;
}

} // namespace gbsw
