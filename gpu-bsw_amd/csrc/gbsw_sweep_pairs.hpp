// gbsw_sweep_pairs.hpp -- the sweep kernel with eight pairs per wave: the recurrence,
// offsets, best-cell filter and strict reverse pass of gbsw_sweep.hpp, in another
// geometry.
//
// Sixteen lanes align two pairs, one in each 16-bit half of every state register.
// Lane l owns columns l K .. l K + K - 1 of both (one strip of 16 K columns, K <= 16)
// and works on row s - l at step s.  Against four pairs per wave, whose halves are two
// blocks of one pair's columns, a wavefront fills and drains in 15 steps instead of 31
// (the reverse pass of a 150-base read is 180 steps instead of 213), columns come in
// multiples of 16 instead of 32, and the instructions of a step that do not depend on
// K serve two pairs.  It takes as long per wave and holds twice the pairs, so small
// jobs keep the four-pair form.  Only for register tables (up to four residue codes):
// a profile per pair would leave LDS for few waves.
//
// The left boundary needs no selector: the DPP shift fills the first lane with zeros,
// which become negative, and a maximum with the boundary's value (the floor, which no
// other lane's value is below) replaces them.
//
// The row that holds a lane's best is kept in LDS, written under the mask of the
// lanes that improved: with eight pairs some pair improves in most steps (a read's
// best grows on nearly every row of its alignment), and selecting K registers is a
// third of such a step's extra instructions.  In 16-bit halves, so that 16 waves fit a
// CU at every K (dwords: 12, and 16.1 ms where this takes 14.4).
//
// Bound by VALU issue, 0.94 per CU-cycle.  The 858k pairs of up to 256 columns of the
// 1M-pair DNA mix (8.25e10 cells): 14.4 ms, 8.3e9 wave instructions; four pairs per wave
// took 16.3 ms and 9.9e9.  The whole mix 24.4 -> 22.0 ms.
#pragma once
#include "gbsw_sweep.hpp"

namespace gbsw {

constexpr int kNoStep = 0xFFFF; // (sequences end at 65,000)

struct PairsSmem {
    uint8_t* base;
    PairsLds L;
    __device__ uint8_t* lut() const { return base + L.lut_off; }
    __device__ int16_t* sub() const { return (int16_t*)(base + L.sub_off); }
    __device__ int16_t* colmax() const { return (int16_t*)(base + L.colmax_off); }
    __device__ uint16_t* row_tab() const { return (uint16_t*)(base + L.row_tab_off); }
    __device__ uint32_t* col_tab() const { return (uint32_t*)(base + L.col_tab_off); }
    __device__ uint32_t* ring(int g) const { return (uint32_t*)(base + L.ring_off) + g * (2 * kPairsRing); }
    __device__ uint16_t* snap() const { return (uint16_t*)(base + L.snap_off); }
};

// x and y of the lane to the left in the row, each less d; the first lane takes -d.
__device__ __forceinline__ void row_left(uint32_t x, uint32_t y, uint32_t d, uint32_t& xo, uint32_t& yo)
{
    asm volatile("s_nop 1\n\t"
                 "v_sub_u32_dpp %0, %2, %4 row_shr:1 row_mask:0xf bank_mask:0xf bound_ctrl:0\n\t"
                 "v_sub_u32_dpp %1, %3, %4 row_shr:1 row_mask:0xf bank_mask:0xf bound_ctrl:0"
                 : "=&v"(xo), "=v"(yo)
                 : "v"(x), "v"(y), "v"(d));
}

// One pass for the two pairs of every group of the wave (REV: the reverse one); key:
// their winner keys, as in gbsw_pass.hpp.
template <class A, int K, bool REV>
__device__ __forceinline__ void sweep_pairs(const KernelArgs& a, const PairsSmem& sm, const Task (&t)[2],
                                            const int32_t (&target)[2], bool strict, uint64_t (&key)[2])
{
    using V = uint32_t;
    constexpr int G = kLanesPerPair, R = kPairsRing, N = kChunk / G;
    constexpr int UN = K <= 8 ? kSweepUnroll : 2;
    const int lane = threadIdx.x, g = lane / G, l = lane & (G - 1);
    const int ge = -a.gap_extend, go = -a.gap_open;
    const int base = a.base, low = REV && strict ? kRevLow : 0, zero = base + low;
    uint32_t* ring = sm.ring(g);
    uint16_t* snap = sm.snap() + lane; // rows of the bests: word (half (K + 1) + k) x 64; k = K: the step

    bool live[2];
    int32_t tgt[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        live[h] = t[h].nr > 0 && t[h].nc > 0;
        tgt[h] = target[h] > 0 ? target[h] : kUnreached;
    }
    int steps_max = max(t[0].nr, t[1].nr) + G - 1;
    steps_max = max(steps_max, __shfl_xor(steps_max, 16));
    steps_max = max(steps_max, __shfl_xor(steps_max, 32));
    steps_max = __builtin_amdgcn_readfirstlane(steps_max);

    const uint32_t gs = A::uni(ge), cs = A::uni(ge - go), shift = A::uni(a.shift);
    // (opaque: kept in a vector register, where the DPP subtraction takes it)
    V hand = A::uni(ge * (K - 1));
    A::keep(hand);

    // ---- the four biased scores of each column, as bytes
    uint32_t tl[K], th[K];
    auto col_byte = [&](int h, int c) {
        return live[h] && c < t[h].nc ? (int)t[h].cols[t[h].rev ? t[h].nc_full - 1 - c : c] : kNoRow;
    };
    __syncthreads();
#pragma unroll
    for (int k = 0; k < K; ++k) {
        tl[k] = sm.col_tab()[col_byte(0, l * K + k)];
        th[k] = sm.col_tab()[col_byte(1, l * K + k)];
    }

    // forward: the lane's thresholds (true scores); reverse: the scores to reach less one
    V bt = REV ? A::pair(tgt[0] - 1, tgt[1] - 1) : A::pair(live[0] ? 0 : kUnreached, live[1] ? 0 : kUnreached);
    // reverse, strict: the least score (less one) from which a row of the lane may still
    // reach the target
    V dead = A::splat(kUnreached);
    if constexpr (REV) {
        if (strict) {
            int32_t d[2];
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                int own = 0;
#pragma unroll
                for (int k = 0; k < K; ++k) {
                    const int b = col_byte(h, l * K + k), c = b < kNoRow ? (int)sm.lut()[b] : a.alpha;
                    own += c < a.alpha ? (int)sm.colmax()[c] : 0;
                }
                int sum = own; // inclusive prefix sum over the lanes
#pragma unroll
                for (int x = 1; x < G; x <<= 1) {
                    const int u = __shfl_up(sum, x, G);
                    if (l >= x) sum += u;
                }
                d[h] = target[h] > 0 && live[h] ? max(0, tgt[h] - 1 - (t[h].ubound - (sum - own))) : kUnreached;
            }
            dead = A::pair(d[0], d[1]);
        }
    }

    // state before step 0: zero scores at the offsets of step -1
    V Ho[K], F[K];
#pragma unroll
    for (int k = 0; k < K; ++k) {
        Ho[k] = A::uni(zero + ge * k) + cs;
        F[k] = A::uni(zero);
    }
    V Eout = A::uni(zero + ge * K), Hd0 = A::uni(zero - go);
    int32_t rt[2] = {0x7FFFFFFF, 0x7FFFFFFF}, rr[2] = {0, 0}; // reverse hits
    bool dirty = false; // some lane's best moved since the groups' were last shared
    if constexpr (!REV) {
        snap[K * kWave] = snap[(2 * K + 1) * kWave] = kNoStep;
    }

    // row ring: a chunk of padding rows, then rows [s0, s0 + 32) as step s0 begins; the
    // next chunk's bytes are on their way
    struct Rows {
        int32_t b[2][N];
    };
    auto fetch_rows = [&](int chunk) {
        Rows f;
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int i = 0; i < N; ++i) {
                const int x = chunk * kChunk + l + G * i;
                f.b[h][i] = x < t[h].nr ? (int32_t)t[h].rows[t[h].rev ? t[h].nr_full - 1 - x : x] : kNoRow;
            }
        return f;
    };
    auto store_rows = [&](const Rows& f, int chunk) {
#pragma unroll
        for (int i = 0; i < N; ++i) {
            // a whole v_perm selector: a score byte of the low table, zero, one of the
            // high table, zero
            const uint32_t e0 = sm.row_tab()[f.b[0][i]], e1 = sm.row_tab()[f.b[1][i]];
            const uint32_t e = e0 | (e1 + (e1 == kPadSelector ? 0u : 4u)) << 16;
            const int at = (chunk * kChunk + l + G * i) & (R - 1);
            ring[at] = e;
            ring[at + R] = e; // again, so that a chunk's reads are contiguous
        }
    };
    {
        Rows none;
#pragma unroll
        for (int i = 0; i < N; ++i) none.b[0][i] = none.b[1][i] = kNoRow;
        store_rows(none, -1);
    }
    Rows pf = fetch_rows(0);
    for (int s0 = 0; s0 < steps_max; s0 += kChunk) {
        store_rows(pf, s0 / kChunk);
        pf = fetch_rows(s0 / kChunk + 1);
        __syncthreads();
        if (s0 > 0 && (s0 & (kRebase - 1)) == 0) {
            const uint32_t d = A::uni(ge * kRebase);
#pragma unroll
            for (int k = 0; k < K; ++k) { Ho[k] -= d; F[k] -= d; }
            Eout -= d;
            Hd0 -= d;
        }
        if (!REV && dirty) {
            V m = bt;
            m = pk_max(m, row_ror<1>(m));
            m = pk_max(m, row_ror<2>(m));
            m = pk_max(m, row_ror<4>(m));
            m = pk_max(m, row_ror<8>(m));
            bt = A::vmax(bt, A::less1(m));
            dirty = false;
        }
        // strict reverse pass: over once no value in flight can reach the target
        if (REV && strict && s0 >= G) {
            V m = A::vmax(Hd0, Ho[0]);
#pragma unroll
            for (int k = 1; k < K; ++k) m = A::vmax(m, Ho[k]);
            // (Hd0 has the smallest offset of them)
            const uint32_t zd = A::uni(zero + ge * ((s0 & (kRebase - 1)) - 1)) + cs;
            if (__ballot(A::exceeds(m, dead + zd)) == 0) break;
        }
        const int s_end = min(s0 + kChunk, steps_max);
        const uint32_t* rc = ring + ((s0 - l) & (R - 1));
        auto step = [&](const int s, const uint32_t code, const uint32_t z, const uint32_t zf, const V thr) {
            V xH, xE;
            row_left(Ho[K - 1], Eout, hand, xH, xE);
            xH = A::vmax(xH, zf - A::uni(go)); // zero scores left of the first column
            xE = A::vmax(xE, zf);
            V E = xE, Hd = Hd0;
#pragma unroll
            for (int k = 0; k < K; ++k) {
                const V D = A::template add<false>(Hd, __builtin_amdgcn_perm(th[k], tl[k], code), shift);
                Hd = Ho[k];
                const V H = A::max3(D, E, F[k]);
                const V ho = H + cs;
                E = A::max3u(E, ho, zf + (uint32_t)(k + 1) * gs);
                F[k] = A::vmax(F[k], ho);
                Ho[k] = ho;
            }
            Eout = E;
            Hd0 = xH;
            if (__ballot(A::exceeds(Eout, thr)) != 0) {
                const uint32_t zc = z + cs; // true scores of the row: Ho less its offset
                V h[K];
                if constexpr (!REV) {
#pragma unroll
                    for (int k = 0; k < K; ++k) h[k] = Ho[k] - (zc + (uint32_t)k * gs);
                    const V nb = tree_max<A, K>(h);
                    if ((nb & 0xFFFFu) > (bt & 0xFFFFu)) {
#pragma unroll
                        for (int k = 0; k < K; ++k) snap[k * kWave] = (uint16_t)h[k];
                        snap[K * kWave] = (uint16_t)s;
                    }
                    if ((nb >> 16) > (bt >> 16)) {
#pragma unroll
                        for (int k = 0; k < K; ++k) snap[(K + 1 + k) * kWave] = (uint16_t)(h[k] >> 16);
                        snap[(2 * K + 1) * kWave] = (uint16_t)s;
                    }
                    bt = A::vmax(bt, nb);
                    dirty = true;
                } else {
                    // first (smallest) column of this row that reaches the target
                    const int row = s - l;
                    uint32_t m0 = 0, m1 = 0;
#pragma unroll
                    for (int k = K - 1; k >= 0; --k) {
                        h[k] = A::sub_each(Ho[k], zc + (uint32_t)k * gs); // (may be negative)
                        m0 = 2 * m0 + (A::lo(h[k]) == tgt[0] ? 1u : 0u);
                        m1 = 2 * m1 + (A::hi(h[k]) == tgt[1] ? 1u : 0u);
                    }
#pragma unroll
                    for (int q = 0; q < 2; ++q) {
                        const uint32_t m = (q ? m1 : m0) & sweep_cols(t[q].nc - l * K);
                        const int c = l * K + (m ? __builtin_ctz(m) : K);
                        if (m && row >= 0 && row < t[q].nr && c < rt[q]) {
                            rt[q] = c;
                            rr[q] = row;
                        }
                    }
                }
            }
        };
        // offset of column 0 at step s0; steps past steps_max only meet padding rows
        uint32_t z = A::uni(zero + ge * ((s0 & (kRebase - 1)) + 1));
        // and that of the floor: zero scores while lanes may still be above row 0
        const uint32_t down = A::uni(REV && s0 >= G ? low : 0);
        uint32_t ca = rc[0], cb = rc[1];
        for (int s = s0; s < s_end; s += UN) {
            // a row of the iteration may improve the best (reach the target) only if E
            // leaving the lane exceeds this: best - o - g (K - 1) at the first step's offset
            const V thr = bt + (z + cs);
#pragma unroll
            for (int u = 0; u < UN; u += 2) {
                const uint32_t c0 = ca, c1 = cb;
                ca = rc[2];
                cb = rc[3];
                step(s + u, c0, z, z - down, thr);
                z += gs;
                step(s + u + 1, c1, z, z - down, thr);
                z += gs;
                rc += 2;
            }
        }
    }

    // ---- candidates, reduced over each group
    V most = bt; // forward: the groups' highest thresholds (see sweep)
    if constexpr (!REV) {
        most = pk_max(most, row_ror<1>(most));
        most = pk_max(most, row_ror<2>(most));
        most = pk_max(most, row_ror<4>(most));
        most = pk_max(most, row_ror<8>(most));
    }
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        uint64_t k64 = 0;
        if constexpr (!REV) {
            const int32_t s = snap[(h * (K + 1) + K) * kWave];
            uint32_t v[K];
            uint32_t b = 0;
#pragma unroll
            for (int k = 0; k < K; ++k) {
                v[k] = snap[(h * (K + 1) + k) * kWave];
                b = max(b, v[k]);
            }
            if (live[h] && s != kNoStep && b > 0) {
                uint32_t pbest = 0xFFFFFFFFu;
#pragma unroll
                for (int k = 0; k < K; ++k) {
                    const int col = l * K + k;
                    if (v[k] == b && col < t[h].nc) pbest = min(pbest, tie_prio((uint32_t)col));
                }
                const int row = s - l;
                if (pbest != 0xFFFFFFFFu && row < t[h].nr)
                    k64 = ((uint64_t)b << 40) | ((uint64_t)(0xFFFFFu - (uint32_t)row) << 20) |
                          (uint64_t)(0xFFFFFu - pbest);
            }
        } else if (live[h] && rt[h] != 0x7FFFFFFF) {
            k64 = ((uint64_t)(0xFFFFFu - (uint32_t)rt[h]) << 20) | (uint64_t)(0xFFFFFu - (uint32_t)rr[h]);
        }
#pragma unroll
        for (int x = 1; x < G; x <<= 1) {
            const uint64_t o = ((uint64_t)(uint32_t)__shfl_xor((int)(uint32_t)(k64 >> 32), x) << 32) |
                               (uint32_t)__shfl_xor((int)(uint32_t)k64, x);
            k64 = o > k64 ? o : k64;
        }
        const int32_t top = h ? A::hi(most) : A::lo(most);
        if (!REV && live[h] && top >= a.sat_limit) k64 = max(k64, (uint64_t)top << 40);
        key[h] = k64;
    }
}

// Both passes of the wave's pairs, and their results.
template <class A, int K>
__device__ __forceinline__ void sweep_pairs_set(const KernelArgs& a, const PairsSmem& sm, const int64_t (&p)[2])
{
    const int l = threadIdx.x & (kLanesPerPair - 1);
    const int32_t none[2] = {0, 0};
    uint64_t key[2];
    FwdOut f[2];
    Task t[2];
    {
        const Task tf[2] = {forward_task(a, p[0]), forward_task(a, p[1])};
        sweep_pairs<A, K, false>(a, sm, tf, none, false, key);
    }
    int32_t target[2];
    bool swaps = false;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        f[h] = forward_result<kLanesPerPair>(a, p[h], key[h]);
        const RevPlan rp = reverse_plan<kLanesPerPair>(a, sm, p[h], f[h]); // (a symmetric table)
        t[h] = rp.t;
        target[h] = rp.target;
        swaps |= p[h] >= 0 && f[h].score > 0 && reverse_swaps(a, p[h], f[h]);
    }
    const bool strict = __ballot(swaps) == 0;
    sweep_pairs<A, K, true>(a, sm, t, target, strict, key);
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        int32_t rb, qb;
        reverse_result(a, p[h], f[h], t[h], target[h], key[h], &rb, &qb);
        if (p[h] >= 0 && l == 0 && f[h].score >= 0) {
            a.out[kOutScore * a.n + p[h]] = f[h].score;
            a.out[kOutRefEnd * a.n + p[h]] = f[h].ref_end;
            a.out[kOutQueryEnd * a.n + p[h]] = f[h].query_end;
            a.out[kOutRefBegin * a.n + p[h]] = rb;
            a.out[kOutQueryBegin * a.n + p[h]] = qb;
        }
    }
}

// Persistent workgroups (one wave) pull sets of eight pairs, longest first; a.ranges
// gives their geometries, as in k_sweep.
// WIDE: the geometries of K > kPairsNarrowMax; apart, since their registers spill more
// outside the loops (one kernel for all: 14.6 ms for the 858k pairs, two 14.4).
template <class A, bool WIDE>
__global__ __launch_bounds__(64, 4) void k_sweep_pairs(KernelArgs a)
{
    extern __shared__ __align__(16) uint8_t smem_raw[];
    constexpr int PW = 8;
    const PairsSmem sm{smem_raw, pairs_lds(a.kmax, a.alpha)};
    stage_tables(a, sm);
    stage_byte_tables<A, kProfRegs>(a, sm);
    const int g = threadIdx.x / kLanesPerPair;
    const int64_t nsets = (a.order_n + PW - 1) / PW;
    for (;;) {
        uint32_t q = 0;
        if (threadIdx.x == 0) q = atomicAdd(a.queue, 1u);
        q = (uint32_t)__builtin_amdgcn_readfirstlane((int)q);
        if ((int64_t)q >= nsets) break;
        const int64_t p[2] = {slot_pair(a, (int64_t)q * PW + 2 * g), slot_pair(a, (int64_t)q * PW + 2 * g + 1)};
        int K = a.ranges[a.nranges - 1].K;
        for (int r = a.nranges - 2; r >= 0; --r)
            if ((int64_t)q * PW < a.ranges[r].end) K = a.ranges[r].K;
#define GBSW_CASE(k) case k: sweep_pairs_set<A, k>(a, sm, p); break;
        if constexpr (WIDE) {
            switch (K) { GBSW_SWEEP_PAIRS_WIDE(GBSW_CASE) }
        } else {
            switch (K) { GBSW_SWEEP_PAIRS(GBSW_CASE) }
        }
#undef GBSW_CASE
    }
}

} // namespace gbsw
