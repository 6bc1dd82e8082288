// gbsw_traceback.hip -- alignment paths (CIGAR) of aligned pairs on gfx950.
//
// The reference declares a traceback (traceBack, kernel.hpp:36-39) but never
// defines it.  Here the path of a pair with score > 0 is the best GLOBAL
// alignment of ref[ref_begin, ref_end) against query[query_begin, query_end)
// (the rectangle the forward and reverse passes report), scored like the forward
// pass: a run of L gap positions scores open + (L-1) extend, and the substitution
// is s(row residue, column residue) with rows = the longer full sequence (ref on
// ties, kernel.cpp:248-259).  Among optimal alignments the path is the one whose
// op sequence, read from its end, is lexicographically smallest with M < D < I.
//
// k_tb_keys orders the pairs (classes of like rectangles, largest first) and counts
// them; k_tb_path computes and walks the paths; k_tb_compact copies each pair's
// runs, reversed, to their final place.
//
// k_tb_path: one wave takes a set of 2 x 64/G pairs: G lanes per two pairs, one pair
// in each 16-bit half of every state register (or in two int32 registers).  Lane l
// owns K columns of a stripe of G x K and walks the rectangle's rows along
// anti-diagonals (row t - l + 1 at step t); the left neighbour's values arrive by a
// one-lane DPP shift, whose first lane takes the stripe's left boundary.  The
// rectangle is global, so every value can carry the offset g (row + column), with g
// the cost of extending a gap and o that of opening one; extending then costs nothing:
//   e  = max(E, Ho left)    f = max(F, Ho above)     Ho = H + g - o
//   D  = Ho diagonal + s + o + g                     H  = max3(D, F', E')
// Values are scaled by four; the low two bits name the op that made them, M (3) over
// D (2) over I (1), so that the maxima themselves prefer the smaller op:
//   H's tag is the op at the cell; F is extended under tag 2, so f's tag is the op
//   before a D there (a tie prefers opening from an M to extending, and extending to
//   an I); E is extended under tag 1, so e's tag is the op before an I there.
// The walk needs "extends" of f and e (one bit each, placed where one bit-select
// joins them) and H's tag: four bits per cell, four cells per 16-bit half.
//
// The same wave then walks its pairs back from the bits; its lanes look at
// consecutive cells of a run at once, so a run of matches costs one step per 64/pairs
// cells.  The bits live in a scratch region per workgroup that the next set overwrites.
//
// Bound by VALU issue: 13.5 packed instructions per two cells and about 16 per step
// (0.77 per CU-cycle on the DNA mix, 300k pairs); half a byte per cell is written.
// Before, with flags from compares (23 packed instructions per two cells), a byte per
// cell kept for a separate kernel that walked one pair per lane: 8.5 ms for those 300k
// pairs and 28 ms for a million, now 4.4 and 14.3; 5,000 proteins 7.4 ms, now 1.4.
#include <hip/hip_runtime.h>
#include <hipcub/hipcub.hpp>

#include "gbsw_device.hpp"
#include "gbsw_kernels.hpp"

namespace gbsw {

namespace {

enum : uint32_t { kOpM = 0, kOpI = 1, kOpD = 2 };        // BAM CIGAR op codes
constexpr uint32_t kTagM = 3, kTagD = 2, kTagI = 1;       // tags of scaled values

struct PairRect {
    int32_t m, n;    // rectangle rows (ref side) and columns (query side)
    bool swap;       // rows of the forward pass are the query (|ref| < |query|)
    const uint8_t* A;
    const uint8_t* B;
};

__device__ __forceinline__ PairRect pair_rect(const TbArgs& a, int64_t p)
{
    PairRect r;
    const int32_t rb = a.out[a.n + p], re = a.out[2 * a.n + p];
    const int32_t qb = a.out[3 * a.n + p], qe = a.out[4 * a.n + p];
    r.m = re - rb;
    r.n = qe - qb;
    r.swap = (a.ref_off[p + 1] - a.ref_off[p]) < (a.qry_off[p + 1] - a.qry_off[p]);
    r.A = a.ref + a.ref_off[p] + rb;
    r.B = a.qry + a.qry_off[p] + qb;
    return r;
}

constexpr int kTbBlock = 64;  // steps between refills of a group's row ring
constexpr int kTbRing = 128;  // rows per group: a block's and the G - 1 before

// half-octave of x > 0: floor(2 log2 x)
__host__ __device__ __forceinline__ int half_octave(uint32_t x)
{
#ifdef __HIP_DEVICE_COMPILE__
    const int b = 31 - __clz((int)x);
#else
    const int b = 31 - __builtin_clz(x);
#endif
    // x >= 2^(b + 1/2)  <=>  x^2 >= 2^(2b + 1)
    return 2 * b + (((uint64_t)x * x) >> (2 * b + 1) ? 1 : 0);
}

// ---------------------------------------------------------------- cell policies

// the same 16 bits in both halves (x may be negative: the halves then add like one
// 32-bit number as long as neither result is)
__device__ constexpr uint32_t both(uint32_t x) { return x * 0x00010001u; }

// Two pairs in the 16-bit halves of a register.  WIDE: maxima of unsigned 16-bit
// integers; else of integers up to 0x7C00 through their f16 patterns (three operands
// in one instruction).
template <bool WIDE>
struct Tag16 {
    using V = uint32_t;
    using B = uint2; // boundary entry: Ho and E of both pairs
    static constexpr bool kInt32 = false;
    __device__ static V splat(int32_t x) { return both((uint32_t)x); }
    __device__ static V lowest() { return 0; }
    __device__ static V add(V a, V b) { return a + b; }
    __device__ static V vmax(V a, V b) { return raw(__builtin_elementwise_max(as_u(a), as_u(b))); }
    __device__ static V max3(V a, V b, V c)
    {
        if constexpr (WIDE) return vmax(vmax(a, b), c);
        else return pk_max3_f16(a, b, c);
    }
    __device__ static V retag(V x, uint32_t tag) { return (x & both(0xFFFCu)) | both(tag); }
    __device__ static V tag_m(V x) { return x | both(kTagM); }
    // diagonal value + scaled score (biased; a word may be negative)
    template <int PF>
    __device__ static V score(V x, uint32_t S, int32_t)
    {
        if constexpr (PF == kProfWords) return raw((u16x2)(as_u(x) + as_u(S)));
        else return x + S;
    }
    // four bits of a cell pushed into the halves of acc (what a shift moves past a
    // half's top lands in bits that the next field covers)
    __device__ static V bits(V acc, bool first, V e, V f, V H)
    {
        V y = (both(2) & e) | (~both(2) & f);
        y = (both(3) & y) | (~both(3) & (H << 2));
        if (first) return y;
        return (both(15) & y) | (~both(15) & (acc << 4));
    }
    __device__ static uint32_t packed(V acc) { return acc; }
    __device__ static int32_t half(V x, int h) { return (int32_t)(h ? x >> 16 : x & 0xFFFFu); }
    template <int G>
    __device__ static void shift(V& xh, V& xe, V h, V e)
    {
        static_assert(G == 16 || G == 64, "lanes per group");
        if constexpr (G == 16)
            asm volatile("s_nop 1\n\t"
                         "v_mov_b32_dpp %0, %2 row_shr:1 row_mask:0xf bank_mask:0xf\n\t"
                         "v_mov_b32_dpp %1, %3 row_shr:1 row_mask:0xf bank_mask:0xf"
                         : "+&v"(xh), "+&v"(xe)
                         : "v"(h), "v"(e));
        else
            asm volatile("s_nop 1\n\t"
                         "v_mov_b32_dpp %0, %2 wave_shr:1 row_mask:0xf bank_mask:0xf\n\t"
                         "v_mov_b32_dpp %1, %3 wave_shr:1 row_mask:0xf bank_mask:0xf"
                         : "+&v"(xh), "+&v"(xe)
                         : "v"(h), "v"(e));
    }
    __device__ static B entry(V h, V e) { return make_uint2(h, e); }
    __device__ static void take(B b, V& h, V& e) { h = b.x; e = b.y; }
    __device__ static B load(const B* p)
    {
        const uint64_t v = __hip_atomic_load((const uint64_t*)p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        return make_uint2((uint32_t)v, (uint32_t)(v >> 32));
    }
};

// Two pairs in two int32 registers (16-bit profile of plain scores).
struct Tag32 {
    struct V {
        int32_t a, b;
    };
    using B = int4;
    static constexpr bool kInt32 = true;
    // cells outside a rectangle may run out of range: they only reach each other
    __device__ static int32_t plus(int32_t x, int32_t y) { return (int32_t)((uint32_t)x + (uint32_t)y); }
    __device__ static V splat(int32_t x) { return V{x, x}; }
    __device__ static V lowest() { return splat((int32_t)0x80000000); }
    __device__ static V add(V x, V y) { return V{plus(x.a, y.a), plus(x.b, y.b)}; }
    __device__ static V vmax(V x, V y) { return V{max(x.a, y.a), max(x.b, y.b)}; }
    __device__ static V max3(V x, V y, V z) { return vmax(vmax(x, y), z); }
    __device__ static V retag(V x, uint32_t tag) { return V{(x.a & ~3) | (int32_t)tag, (x.b & ~3) | (int32_t)tag}; }
    __device__ static V tag_m(V x) { return V{x.a | (int32_t)kTagM, x.b | (int32_t)kTagM}; }
    template <int PF>
    __device__ static V score(V x, uint32_t S, int32_t bias4)
    {
        static_assert(PF == kProfWords, "int32 cells take a 16-bit profile");
        return V{plus(x.a, (int32_t)(int16_t)S * 4 + bias4), plus(x.b, ((int32_t)S >> 16) * 4 + bias4)};
    }
    __device__ static int32_t bits1(int32_t acc, bool first, int32_t e, int32_t f, int32_t H)
    {
        int32_t y = (2 & e) | (~2 & f);
        y = (3 & y) | (~3 & (int32_t)((uint32_t)H << 2));
        return first ? y : (15 & y) | (~15 & (int32_t)((uint32_t)acc << 4));
    }
    __device__ static V bits(V acc, bool first, V e, V f, V H)
    {
        return V{bits1(acc.a, first, e.a, f.a, H.a), bits1(acc.b, first, e.b, f.b, H.b)};
    }
    __device__ static uint32_t packed(V acc) { return ((uint32_t)acc.a & 0xFFFFu) | ((uint32_t)acc.b << 16); }
    __device__ static int32_t half(V x, int h) { return h ? x.b : x.a; }
    template <int G>
    __device__ static void shift(V& xh, V& xe, V h, V e)
    {
        uint32_t a0 = (uint32_t)xh.a, a1 = (uint32_t)xe.a, b0 = (uint32_t)xh.b, b1 = (uint32_t)xe.b;
        Tag16<false>::shift<G>(a0, a1, (uint32_t)h.a, (uint32_t)e.a);
        Tag16<false>::shift<G>(b0, b1, (uint32_t)h.b, (uint32_t)e.b);
        xh = V{(int32_t)a0, (int32_t)b0};
        xe = V{(int32_t)a1, (int32_t)b1};
    }
    __device__ static B entry(V h, V e) { return make_int4(h.a, h.b, e.a, e.b); }
    __device__ static void take(B b, V& h, V& e) { h = V{b.x, b.y}; e = V{b.z, b.w}; }
    __device__ static B load(const B* p)
    {
        const uint64_t u = __hip_atomic_load((const uint64_t*)p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        const uint64_t w = __hip_atomic_load((const uint64_t*)p + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        return make_int4((int32_t)(uint32_t)u, (int32_t)(u >> 32), (int32_t)(uint32_t)w, (int32_t)(w >> 32));
    }
};

// ---------------------------------------------------------------- geometry

// Bytes of one profile row (one residue code of one pair, a stripe's columns).
__host__ __device__ constexpr int tb_lane_bytes(int K, int form)
{
    return form == kProfRegs ? 0 : form == kProfBytes ? (K <= 4 ? 4 : 8) : (K <= 4 ? 8 : 16);
}
struct TbLds {
    int32_t sub_off, lut_off, group_off, prof_bytes, ring_off, bnd_off, bout_off, group_bytes, total;
};
__host__ __device__ inline TbLds tb_lds(int G, int kmax, int form, int alpha, int entry_bytes)
{
    TbLds L;
    L.lut_off = 0; // 257 codes (256: outside the rectangle)
    L.sub_off = 272;
    L.group_off = (L.sub_off + 2 * alpha * alpha + 15) & ~15;
    L.prof_bytes = (alpha + 1) * G * tb_lane_bytes(kmax, form);
    L.ring_off = 2 * L.prof_bytes;
    L.bnd_off = L.ring_off + 4 * (kTbRing + 16);
    L.bout_off = L.bnd_off + entry_bytes * (kTbBlock + 4);
    L.group_bytes = (L.bout_off + entry_bytes * kTbBlock + 15) & ~15;
    L.total = L.group_off + (64 / G) * L.group_bytes;
    return L;
}
__host__ __device__ constexpr int tb_accs(int K) { return K > 4 ? 2 : 1; } // four cells per half

// Instructions of a step (two pairs): 13.5 per column and the rest.
__host__ __device__ constexpr int tb_step_cost(int K) { return (27 * K + 1) / 2 + 16; }

// Geometry of a set by its widest rectangle: the K (at most kmax) of least work.
__host__ __device__ __forceinline__ int tb_best_k(int32_t n, int G, int kmax)
{
    int best = 2;
    int64_t cost = (int64_t)1 << 62;
    for (int K = 2; K <= kmax; ++K) {
        if (K == 7) continue;
        const int64_t c = (int64_t)((n + G * K - 1) / (G * K)) * tb_step_cost(K);
        if (c < cost) { cost = c; best = K; }
    }
    return best;
}
// Scratch of a set of ng groups whose widest rectangle is rows x n.
__host__ __device__ __forceinline__ int64_t tb_set_bytes(int32_t rows, int32_t n, int G, int K, int ng, int entry_bytes)
{
    const int64_t stripes = (n + G * K - 1) / (G * K);
    const int64_t dir = stripes * (int64_t)(rows + G - 1) * ng * G * 4 * tb_accs(K);
    const int64_t bnd = stripes > 1 ? (int64_t)(rows + 1) * ng * entry_bytes : 0;
    return ((dir + 15) & ~(int64_t)15) + bnd;
}

// Order keys, largest class first; per class of the product its pairs and the largest
// value bound, rows, columns and scratch of one pair.
__global__ __launch_bounds__(256) void k_tb_keys(TbArgs a, uint32_t* keys, int32_t* vals, int64_t* cap, TbCounts* counts)
{
    __shared__ TbCounts c;
    constexpr int kWords = (int)(sizeof(TbCounts) / sizeof(uint32_t));
    for (int x = threadIdx.x; x < kWords; x += 256) ((uint32_t*)&c)[x] = 0;
    __syncthreads();
    const int64_t p = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (p < a.n) {
        const int32_t s = a.out[p];
        int32_t m = 0, n = 0;
        if (s > 0) {
            m = a.out[2 * a.n + p] - a.out[a.n + p];
            n = a.out[4 * a.n + p] - a.out[3 * a.n + p];
            if (m <= 0 || n <= 0) {
                atomicOr(&c.bad, 1u);
                m = n = 0;
            }
        }
        cap[p] = (int64_t)m + n;
        vals[p] = (int32_t)p;
        uint32_t key = (1u << kTbKeyBits) - 1u; // no path: last
        if (m > 0) {
            const int area = min(kTbAreas - 2, half_octave((uint32_t)m) + half_octave((uint32_t)n));
            // inside a class by columns (steps of 8), then rows (of 32): the pairs of a
            // set run the largest stripe and row counts among them
            const uint32_t c9 = min((uint32_t)n >> 3, 511u), r5 = min((uint32_t)m >> 5, 31u);
            key = ((uint32_t)(kTbAreas - 2 - area) << 14) | ((511u - c9) << 5) | (31u - r5);
            const int64_t value = (int64_t)a.max_sub * min(m, n) - (int64_t)a.gap_extend * ((int64_t)m + n);
            atomicAdd(&c.pairs[area], 1u);
            atomicMax(&c.value[area], (uint32_t)min(value, (int64_t)0x7FFFFFFF));
            atomicMax(&c.rows[area], (uint32_t)m);
            atomicMax(&c.cols[area], (uint32_t)n);
            atomicMax(&c.span, (uint32_t)(m + n));
#pragma unroll
            for (int w = 0; w < 2; ++w) {
                const int G = w ? 64 : 16;
                const int64_t bytes = max(tb_set_bytes(m, n, G, tb_best_k(n, G, 4), 1, 16),
                                          tb_set_bytes(m, n, G, tb_best_k(n, G, 8), 1, 16));
                atomicMax(&c.scratch[w][area], (uint32_t)min((bytes + 255) >> 8, (int64_t)0xFFFFFFFF));
            }
        } else {
            a.nruns[p] = 0;
            a.path_score[p] = 0;
        }
        keys[p] = key;
    } else if (p == a.n) {
        cap[p] = 0;
        a.nruns[p] = 0;
    }
    __syncthreads();
    for (int x = threadIdx.x; x < kTbAreas; x += 256)
        if (c.pairs[x]) {
            atomicAdd(&counts->pairs[x], c.pairs[x]);
            atomicMax(&counts->value[x], c.value[x]);
            atomicMax(&counts->rows[x], c.rows[x]);
            atomicMax(&counts->cols[x], c.cols[x]);
            atomicMax(&counts->scratch[0][x], c.scratch[0][x]);
            atomicMax(&counts->scratch[1][x], c.scratch[1][x]);
        }
    if (threadIdx.x == 0) {
        if (c.bad) atomicOr(&counts->bad, 1u);
        atomicMax(&counts->span, c.span);
    }
}

struct TbSmem {
    uint8_t* base;
    TbLds L;
};

// The two pairs of this lane's group.
struct TbPairs {
    int64_t p[2];
    PairRect r[2];
};

// DP and walk of a set in geometry K.  rows, n: the largest of its rectangles; ng
// groups of it are in use.
template <class A, int G, int K, int PF>
__device__ __forceinline__ void tb_set(const TbArgs& a, const TbSmem& sm, const TbPairs& pr, int32_t rows, int32_t n, int ng,
                                       uint8_t* region)
{
    using V = typename A::V;
    using B = typename A::B;
    constexpr int W = G * K, NA = tb_accs(K), LB = tb_lane_bytes(K, PF);
    const int lane = threadIdx.x, g = lane / G, l = lane & (G - 1);
    const int alpha = a.alpha, go = -a.gap_open, ge = -a.gap_extend, base = A::kInt32 ? 0 : a.base;
    const uint8_t* lut = sm.base + sm.L.lut_off;
    const int16_t* sub = (const int16_t*)(sm.base + sm.L.sub_off);
    uint8_t* gb = sm.base + sm.L.group_off + g * sm.L.group_bytes;
    uint32_t* ring = (uint32_t*)(gb + sm.L.ring_off);
    B* bndbuf = (B*)(gb + sm.L.bnd_off);
    B* bout = (B*)(gb + sm.L.bout_off);
    const int stripes = (n + W - 1) / W;
    const int32_t steps = rows + G - 1;
    const bool active = g < ng;
    const int64_t stripe_bytes = (int64_t)steps * ng * (G * 4 * NA);
    B* bnd = (B*)(region + ((stripes * stripe_bytes + 15) & ~(int64_t)15)) + (int64_t)(active ? g : 0) * (rows + 1);
    const uint32_t lane_off = (uint32_t)(g * G + l) * (4 * NA);
    const int bias4 = 4 * (go + ge);

    // scaled boundary values (in Ho form): the corner's H = 0; on row 0 and column 0
    // H = -o - (d - 1) g, at the offset g d
    const V corner = A::splat(4 * (base + ge - go)), edge = A::splat(4 * (base + 2 * ge - 2 * go));
    const V low = A::lowest(), cs = A::splat(4 * (ge - go));

    for (int s = 0; s < stripes; ++s) {
        const int32_t c0 = W * s + K * l; // the lane's first column (0-based)
        // ---- scores of the stripe's columns
        __syncthreads();
        uint32_t tb[2][PF == kProfRegs ? K : 1];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const PairRect& r = pr.r[h];
            int cb[K];
#pragma unroll
            for (int q = 0; q < K; ++q) {
                const int c = lut[c0 + q < r.n ? (int)r.B[c0 + q] : 256];
                cb[q] = c < alpha ? c : -1;
            }
            auto sc = [&](int row, int c) { return (int)(r.swap ? sub[c * alpha + row] : sub[row * alpha + c]); };
            if constexpr (PF == kProfRegs) {
#pragma unroll
                for (int q = 0; q < K; ++q) {
                    uint32_t w = 0;
#pragma unroll
                    for (int row = 0; row < kRegAlpha; ++row)
                        if (cb[q] >= 0 && row < alpha) w |= (uint32_t)(uint8_t)(4 * sc(row, cb[q]) + bias4) << (8 * row);
                    tb[h][q] = w;
                }
            } else {
                uint8_t* prof = gb + h * sm.L.prof_bytes + l * LB;
                for (int row = 0; row <= alpha; ++row) {
                    uint32_t w[LB / 4];
#pragma unroll
                    for (int d = 0; d < LB / 4; ++d) w[d] = 0;
#pragma unroll
                    for (int q = 0; q < K; ++q) {
                        const bool in = row < alpha && cb[q] >= 0;
                        if constexpr (PF == kProfBytes)
                            w[q / 4] |= (in ? (uint32_t)(uint8_t)(4 * sc(row, cb[q]) + bias4) : 0u) << (8 * (q & 3));
                        else
                            w[q / 2] |= (uint32_t)(uint16_t)(A::kInt32 ? (in ? sc(row, cb[q]) : -32000)
                                                                       : (in ? 4 * sc(row, cb[q]) + bias4 : 0))
                                        << (16 * (q & 1));
                    }
#pragma unroll
                    for (int d = 0; d < LB / 4; ++d) ((uint32_t*)(prof + row * (G * LB)))[d] = w[d];
                }
            }
        }
        V Ho[K], F[K];
#pragma unroll
        for (int q = 0; q < K; ++q) {
            Ho[q] = edge;
            F[q] = low;
        }
        V Hout = edge, Eout = low;
        // two sets of incoming values in turn: one is the other step's diagonal
        V xh[2] = {edge, s == 0 && l == 0 ? corner : edge}, xe[2] = {low, low};
        // the step at which this lane meets a pair's end corner
        int32_t tend[2];
#pragma unroll
        for (int h = 0; h < 2; ++h)
            tend[h] = (pr.p[h] >= 0 && pr.r[h].n > c0 && pr.r[h].n <= c0 + K) ? pr.r[h].m - 1 + l : -1;

        {
            for (int32_t t0 = 0; t0 < steps; t0 += kTbBlock) {
                // rows t0 .. t0 + 63 of both pairs enter the ring (table selectors or
                // profile offsets), and the boundary entries of those rows
                __syncthreads();
#pragma unroll
                for (int e = 0; e < kTbBlock / G; ++e) {
                    const int32_t x = t0 + e * G + l;
                    uint32_t v = 0;
#pragma unroll
                    for (int h = 0; h < 2; ++h) {
                        int c = lut[x < pr.r[h].m ? (int)pr.r[h].A[x] : 256];
                        c = c > alpha ? alpha : c;
                        if constexpr (PF == kProfRegs)
                            v |= (c == alpha ? 0x0C0Cu : 0x0C00u + (uint32_t)c + 4u * h) << (16 * h);
                        else
                            v |= (uint32_t)(c * (G * LB)) << (16 * h);
                    }
                    ring[x & (kTbRing - 1)] = v;
                    B in = A::entry(edge, low);
                    if (s > 0 && active && x < rows) in = A::load(bnd + x);
                    bndbuf[e * G + l] = in;
                }
                __syncthreads();
                const int32_t t1 = min(t0 + kTbBlock, steps);
                const bool ends = __ballot((tend[0] >= t0 && tend[0] < t1) || (tend[1] >= t0 && tend[1] < t1)) != 0;
                struct In {
                    B b; // left boundary (first lane)
                    uint32_t w[PF == kProfRegs ? 1 : 2 * (LB / 4)];
                };
                auto code = [&](int32_t t) { return ring[(t - l) & (kTbRing - 1)]; };
                auto fetch = [&](In& in, uint32_t c, int32_t t) {
                    in.b = bndbuf[t - t0];
                    if constexpr (PF == kProfRegs) {
                        in.w[0] = c;
                    } else {
                        const uint32_t* wa = (const uint32_t*)(gb + (c & 0xFFFFu) + l * LB);
                        const uint32_t* wb = (const uint32_t*)(gb + sm.L.prof_bytes + (c >> 16) + l * LB);
#pragma unroll
                        for (int d = 0; d < LB / 4; ++d) { in.w[d] = wa[d]; in.w[LB / 4 + d] = wb[d]; }
                    }
                };
                auto step = [&](const int32_t t, const In& in, V& xH, V& xE, const V& Hd0, auto masked) {
                    A::take(in.b, xH, xE);
                    A::template shift<G>(xH, xE, Hout, Eout);
                    // a lane starts on row 0 (in the first G - 1 steps)
                    if (!decltype(masked)::value || t >= l) {
                        V E = xE, Hl = xH, Hd = Hd0, acc[2] = {low, low};
#pragma unroll
                        for (int q = 0; q < K; ++q) {
                            uint32_t S;
                            if constexpr (PF == kProfRegs) {
                                S = __builtin_amdgcn_perm(tb[1][q], tb[0][q], in.w[0]);
                            } else if constexpr (PF == kProfBytes) {
                                const uint32_t b = (uint32_t)(q & 3);
                                S = __builtin_amdgcn_perm(in.w[LB / 4 + q / 4], in.w[q / 4], 0x0C040C00u + b + (b << 16));
                            } else {
                                S = (q & 1) ? __builtin_amdgcn_perm(in.w[LB / 4 + q / 2], in.w[q / 2], 0x07060302u)
                                            : __builtin_amdgcn_perm(in.w[LB / 4 + q / 2], in.w[q / 2], 0x05040100u);
                            }
                            const V e = A::vmax(E, Hl);
                            const V f = A::vmax(F[q], Ho[q]);
                            E = A::retag(e, kTagI);
                            F[q] = A::retag(f, kTagD);
                            const V D = A::tag_m(A::template score<PF>(Hd, S, bias4));
                            const V H = A::max3(D, F[q], E);
                            Hd = Ho[q];
                            Hl = A::add(H, cs);
                            Ho[q] = Hl;
                            acc[q / 4] = A::bits(acc[q / 4], q % 4 == 0, e, f, H);
                        }
                        Hout = Hl;
                        Eout = E;
                        if (active) {
                            uint8_t* d = region + s * stripe_bytes + (int64_t)t * (ng * (G * 4 * NA));
                            if constexpr (NA == 2) *(uint2*)(d + lane_off) = make_uint2(A::packed(acc[0]), A::packed(acc[1]));
                            else *(uint32_t*)(d + lane_off) = A::packed(acc[0]);
                        }
                        if (s + 1 < stripes && l == G - 1) bout[t - t0] = A::entry(Hout, Eout);
                        if (ends) {
#pragma unroll
                            for (int h = 0; h < 2; ++h)
                                if (t == tend[h]) {
                                    int32_t v = 0;
#pragma unroll
                                    for (int q = 0; q < K; ++q)
                                        if (c0 + q + 1 == pr.r[h].n) v = A::half(Ho[q], h);
                                    a.path_score[pr.p[h]] = (v >> 2) - (ge - go) - base - ge * (pr.r[h].m + pr.r[h].n);
                                }
                        }
                    }
                };
                In ia, ib;
                fetch(ia, code(t0), t0);
                uint32_t cn = code(t0 + 1);
                auto run = [&](int32_t from, int32_t to, auto masked) { // from: even
                    for (int32_t t = from; t < to; t += 2) {
                        fetch(ib, cn, t + 1);
                        cn = code(t + 2);
                        step(t, ia, xh[0], xe[0], xh[1], masked);
                        if (t + 1 < to) {
                            fetch(ia, cn, t + 2);
                            cn = code(t + 3);
                            step(t + 1, ib, xh[1], xe[1], xh[0], masked);
                        }
                    }
                };
                if (t0 == 0) {
                    const int32_t tm = min(t1, G);
                    run(0, tm, std::true_type{});
                    run(tm, t1, std::false_type{});
                } else {
                    run(t0, t1, std::false_type{});
                }
                // the block's outgoing boundary entries: step t0 + e holds row t0 + e -
                // (G - 1) of the last lane
                if (s + 1 < stripes) {
                    __syncthreads();
                    for (int32_t e = l; e < t1 - t0; e += G) {
                        const int32_t row = t0 + e - (G - 1);
                        if (active && row >= 0) bnd[row] = bout[e];
                    }
                }
            }
        }
        // the boundary column is in memory before the next stripe's loads
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    }

    // ---- walk: LW lanes per pair; pair wp of the set is in half wp & 1 of group wp / 2
    constexpr int PAIRS = 2 * (64 / G), LW = 64 / PAIRS;
    const int wp = lane / LW, wl = lane & (LW - 1), wb = wp * LW, src = (wp >> 1) * G;
    const int64_t p0 = __shfl((long long)pr.p[0], src), p1 = __shfl((long long)pr.p[1], src);
    const int32_t m0 = __shfl(pr.r[0].m, src), m1 = __shfl(pr.r[1].m, src);
    const int32_t n0 = __shfl(pr.r[0].n, src), n1 = __shfl(pr.r[1].n, src);
    const int64_t p = (wp & 1) ? p1 : p0;
    int32_t i = (wp & 1) ? m1 : m0, j = (wp & 1) ? n1 : n0;
    uint32_t* runs = p >= 0 ? a.runs + a.cap_off[p] : nullptr;
    int32_t nr = 0;
    uint32_t run_op = 0, run_len = 0;
    auto emit = [&](uint32_t op, uint32_t len) {
        if (len == 0) return;
        if (run_len && op == run_op) {
            run_len += len;
        } else {
            if (run_len && wl == 0) runs[nr] = run_len << 4 | run_op;
            nr += run_len ? 1 : 0;
            run_op = op;
            run_len = len;
        }
    };
    // the four bits of cell (ci, cj), 1-based
    auto cell = [&](int32_t ci, int32_t cj) {
        const uint32_t c = (uint32_t)(cj - 1), st = c / W, cr = c % W, cl = cr / K, q = cr % K;
        const int64_t at = (int64_t)st * stripe_bytes + (int64_t)(ci - 1 + (int32_t)cl) * (ng * (G * 4 * NA)) +
                           ((wp >> 1) * G + (int32_t)cl) * (4 * NA) + (NA == 2 && q >= 4 ? 4 : 0);
        const uint32_t w =
            __hip_atomic_load((const uint32_t*)(region + at), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        const uint32_t last = q >= 4 ? K - 1 : (K < 4 ? K : 4) - 1; // column in the lowest bits of that dword
        return (w >> (16 * (wp & 1) + 4 * (last - q))) & 15u;
    };
    int st = 0; // 0: H, 1: in a D run (F), 2: in an I run (E)
    bool more = p >= 0 && i > 0 && j > 0;
    while (__ballot(more) != 0) {
        // lane wl looks wl cells down the diagonal, or along the run of gap positions
        const int32_t ci = i - (st != 2 ? wl : 0), cj = j - (st != 1 ? wl : 0);
        const bool in = more && ci >= 1 && cj >= 1;
        uint32_t b = 0;
        if (in) b = cell(ci, cj);
        // the run goes on past this cell
        const bool on = in && (st == 0 ? (b >> 2) == kTagM : st == 1 ? (b & 1u) == 0 : (b & 2u) == 0);
        const uint32_t mask = LW == 64 ? 0u : (uint32_t)(__ballot(on) >> wb) & (uint32_t)((1ull << LW) - 1);
        int c = mask == 0xFFFFFFFFu ? 32 : __builtin_ctz(~mask); // <= LW
        const uint32_t bc = (uint32_t)__shfl((int)b, wb + (c < LW ? c : 0)); // the first cell past it
        if (more) {
            if (st == 0) {
                emit(kOpM, (uint32_t)c);
                i -= c;
                j -= c;
                if (c < LW && i > 0 && j > 0) {
                    // a gap opens at that cell
                    if ((bc >> 2) == kTagD) {
                        emit(kOpD, 1);
                        --i;
                        st = (bc & 1u) ? 0 : 1;
                    } else {
                        emit(kOpI, 1);
                        --j;
                        st = (bc & 2u) ? 0 : 2;
                    }
                }
            } else {
                const int32_t room = st == 1 ? i : j;
                const bool ends = c < LW;
                if (ends && c < room) ++c; // the run's first position (read from its end: the last)
                emit(st == 1 ? kOpD : kOpI, (uint32_t)c);
                if (st == 1) i -= c;
                else j -= c;
                if (ends) st = 0;
            }
            more = i > 0 && j > 0;
        }
    }
    if (p >= 0) {
        emit(kOpI, (uint32_t)j); // a border reached: the rest is one gap
        emit(kOpD, (uint32_t)i);
        if (run_len && wl == 0) runs[nr] = run_len << 4 | run_op;
        nr += run_len ? 1 : 0;
        if (wl == 0) a.nruns[p] = nr;
    }
}

// Persistent workgroups (one wave) pull sets in order, largest first.  A set whose
// rectangles do not fit the workgroup's region together (unlike neighbours in the
// order) is done in parts, in the end pair by pair: the region holds any one pair.
template <class A, int G, int PF>
__global__ __launch_bounds__(64, A::kInt32 ? 2 : 4) void k_tb_path(TbArgs a)
{
    extern __shared__ __align__(16) uint8_t tb_smem[];
    constexpr int NP = 2 * (64 / G);
    constexpr int EB = (int)sizeof(typename A::B);
    const TbSmem sm{tb_smem, tb_lds(G, a.kmax, PF, a.alpha, EB)};
    for (int x = threadIdx.x; x <= 256; x += 64) tb_smem[sm.L.lut_off + x] = x < 256 ? a.lut[x] : 0xFF;
    for (int x = threadIdx.x; x < a.alpha * a.alpha; x += 64) ((int16_t*)(tb_smem + sm.L.sub_off))[x] = a.sub[x];
    const int g = threadIdx.x / G;
    for (int x = threadIdx.x & (G - 1); x < kTbRing; x += G)
        ((uint32_t*)(tb_smem + sm.L.group_off + g * sm.L.group_bytes + sm.L.ring_off))[x] =
            PF == kProfRegs ? 0x0C0C0C0Cu : 0u;
    __syncthreads();
    uint8_t* region = a.dir + (int64_t)blockIdx.x * a.region_bytes;
    const int64_t nsets = (a.count + NP - 1) / NP;
    for (;;) {
        uint32_t q = 0;
        if (threadIdx.x == 0) q = atomicAdd(a.queue, 1u);
        q = (uint32_t)__builtin_amdgcn_readfirstlane((int)q);
        if ((int64_t)q >= nsets) break;
        for (int from = 0, np = NP; from < NP;) {
            // pairs [from, from + np) of the set, in the first groups
            TbPairs pr;
            int32_t rows = 0, n = 0;
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const int64_t k = (int64_t)q * NP + from + 2 * g + h;
                pr.p[h] = 2 * g + h < np && k < a.count ? (int64_t)a.order[a.p0 + k] : -1;
                pr.r[h] = PairRect{0, 0, false, a.ref, a.qry};
                if (pr.p[h] >= 0) pr.r[h] = pair_rect(a, pr.p[h]);
                rows = max(rows, pr.r[h].m);
                n = max(n, pr.r[h].n);
            }
#pragma unroll
            for (int o = G; o < 64; o <<= 1) {
                rows = max(rows, __shfl_xor(rows, o));
                n = max(n, __shfl_xor(n, o));
            }
            rows = __builtin_amdgcn_readfirstlane(rows);
            n = __builtin_amdgcn_readfirstlane(n);
            const int ng = np > 1 ? np / 2 : 1;
            const int K = n > 0 ? tb_best_k(n, G, a.kmax) : 0;
            if (np > 1 && K && tb_set_bytes(rows, n, G, K, ng, EB) > a.region_bytes) {
                np /= 2;
                continue;
            }
            switch (K) {
            case 0: break; // past the last pair
            case 2: tb_set<A, G, 2, PF>(a, sm, pr, rows, n, ng, region); break;
            case 3: tb_set<A, G, 3, PF>(a, sm, pr, rows, n, ng, region); break;
            case 4: tb_set<A, G, 4, PF>(a, sm, pr, rows, n, ng, region); break;
            default:
                if constexpr (PF != kProfWords) { // (words: at most 4)
                    if (K == 5) tb_set<A, G, 5, PF>(a, sm, pr, rows, n, ng, region);
                    else if (K == 6) tb_set<A, G, 6, PF>(a, sm, pr, rows, n, ng, region);
                    else tb_set<A, G, 8, PF>(a, sm, pr, rows, n, ng, region);
                }
            }
            // the next set's stores stay behind this one's loads
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            from += np;
        }
    }
}

__global__ __launch_bounds__(256) void k_tb_compact(const uint32_t* runs, const int64_t* cap_off,
                                                    const int32_t* nruns, const int64_t* dst_off, uint32_t* dst,
                                                    int64_t n)
{
    const int64_t p = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (p >= n) return;
    const int32_t c = nruns[p];
    const uint32_t* src = runs + cap_off[p];
    uint32_t* d = dst + dst_off[p];
    for (int32_t x = 0; x < c; ++x) d[x] = src[c - 1 - x];
}

template <class A, int G>
const void* tb_kernel_form(int form)
{
    if constexpr (A::kInt32) return (const void*)&k_tb_path<A, G, kProfWords>;
    else
        return form == kProfRegs    ? (const void*)&k_tb_path<A, G, kProfRegs>
               : form == kProfBytes ? (const void*)&k_tb_path<A, G, kProfBytes>
                                    : (const void*)&k_tb_path<A, G, kProfWords>;
}

const void* tb_kernel(int cells, int G, int form)
{
    switch (cells) {
    case kTbCells16: return G == 16 ? tb_kernel_form<Tag16<false>, 16>(form) : tb_kernel_form<Tag16<false>, 64>(form);
    case kTbCells16Wide: return G == 16 ? tb_kernel_form<Tag16<true>, 16>(form) : tb_kernel_form<Tag16<true>, 64>(form);
    default: return G == 16 ? tb_kernel_form<Tag32, 16>(form) : tb_kernel_form<Tag32, 64>(form);
    }
}

int tb_entry_bytes(int cells) { return cells == kTbCells32 ? 16 : 8; }

struct Widen {
    __device__ __host__ int64_t operator()(int32_t x) const { return x; }
};

} // namespace

int tb_kmax(int cells, int form) { return cells == kTbCells32 || form == kProfWords ? 4 : 8; }

int64_t tb_region_bytes(int32_t rows, int32_t cols, int G, int kmax, int cells, int groups)
{
    int64_t most = 0; // a set takes the K that fits its own widest rectangle
    for (int K = 2; K <= kmax; ++K)
        most = std::max(most, tb_set_bytes(rows, cols, G, K, groups, tb_entry_bytes(cells)));
    return most;
}

// Instructions of a set's steps: the yardstick of the choice between 16 and 64 lanes.
double tb_set_cost(int32_t rows, int32_t cols, int G, int kmax)
{
    const int K = tb_best_k(cols, G, kmax);
    return (double)((cols + G * K - 1) / (G * K)) * (rows + G - 1) * tb_step_cost(K);
}

int tb_lds_bytes(int cells, int G, int form, int kmax, int alpha)
{
    return tb_lds(G, kmax, cells == kTbCells32 ? kProfWords : form, alpha, tb_entry_bytes(cells)).total;
}

int tb_occupancy(int cells, int G, int form, int lds)
{
    int nb = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, tb_kernel(cells, G, form), 64, (size_t)lds) != hipSuccess) {
        (void)hipGetLastError();
        return 1;
    }
    return std::max(1, nb);
}

hipError_t tb_keys(const TbArgs& a, uint32_t* keys, int32_t* vals, int64_t* cap, TbCounts* counts, hipStream_t stream)
{
    hipLaunchKernelGGL(k_tb_keys, dim3((unsigned)((a.n + 1 + 255) / 256)), dim3(256), 0, stream, a, keys, vals, cap, counts);
    return hipGetLastError();
}

hipError_t tb_launch(const TbArgs& args, int cells, int G, int form, int grid, int lds, hipStream_t stream)
{
    TbArgs a = args;
    void* params[] = {&a};
    return hipLaunchKernel(tb_kernel(cells, G, form), dim3((unsigned)grid), dim3(64), params, (size_t)lds, stream);
}

hipError_t tb_scan(void* temp, size_t& temp_bytes, const int64_t* in, int64_t* out, int64_t n, hipStream_t stream)
{
    return hipcub::DeviceScan::ExclusiveSum(temp, temp_bytes, in, out, (int)n, stream);
}

hipError_t tb_scan(void* temp, size_t& temp_bytes, const int32_t* in, int64_t* out, int64_t n, hipStream_t stream)
{
    hipcub::TransformInputIterator<int64_t, Widen, const int32_t*> it(in, Widen());
    return hipcub::DeviceScan::ExclusiveSum(temp, temp_bytes, it, out, (int)n, stream);
}

hipError_t tb_compact(const uint32_t* runs, const int64_t* cap_off, const int32_t* nruns, const int64_t* dst_off,
                      uint32_t* dst, int64_t n, hipStream_t stream)
{
    if (n <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_tb_compact, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, stream, runs, cap_off, nruns,
                       dst_off, dst, n);
    return hipGetLastError();
}

} // namespace gbsw
