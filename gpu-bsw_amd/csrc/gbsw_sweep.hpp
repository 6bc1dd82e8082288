// gbsw_sweep.hpp -- the alignment kernels of the batched form: six packed
// instructions per two DP cells.
//
// Geometry.  G lanes (a "group": 16, one DPP row, or the whole wave) align one
// pair.  Each lane owns two blocks of K columns of the shorter sequence: the low
// 16-bit half of every state register holds block l (virtual lane v = l), the high
// half block l + G.  Virtual lane v works on row s - v at step s, so the 2G virtual
// lanes form an anti-diagonal wavefront over a strip of 2G x K columns, and the
// halves of a register are independent cells.  Longer column sequences run strip
// by strip; strip t + 1 reads the last column of strip t (H and E per row) from
// global memory.
//
// Recurrence.  With g the cost of extending a gap, o that of opening one, every
// value is held with the offset phi(s, k) = base + g (t + k), t = 1 + s mod
// kRebase, k the column within the lane:
//   D  = Ho(s-1, k-1) + S''            S'' = s(row, col) + o + g (in the tables; where
//                                      bytes do not hold it, less a constant: Sweep16Shifted)
//   H  = max3(D, E, F)
//   Ho = H + (g - o)                   the state, in place of H
//   E' = max3(E, Ho, floor(s, k+1))    (next column)
//   F' = max(F, Ho)                    (next row)
// The offset grows by g along both gap directions, so extending a gap costs no
// instruction, and the floor at zero of H = max(D, E, F, 0) is the third operand
// of E' (every H is at least the floored E of its column).  Between lanes a value
// moves from column K - 1 to the next lane's column -1 one step later, which takes
// g (K - 1) off its offset: the subtraction is the DPP move itself.  Every kRebase
// steps the state drops the g x kRebase it has accumulated.
//
// The maxima are v_pk_maximum3_f16 on integers: the bit patterns of non-negative
// f16 values up to infinity (0x7C00) order as integers do, denormals (below 0x400,
// where most values of short pairs lie) included: the instruction keeps them.  base
// keeps every value non-negative, and a pair whose score comes near the top of
// that range is recomputed with int32 cells: cell values grow by at most one
// substitution per cell, so some lane's threshold passes sat_limit before any value
// passes 0x7C00, and whatever the halves hold after that, thresholds only rise.
//
// Scores: with at most four residue codes a lane keeps, per column, the four
// scores S'' as the bytes of one register, and one v_perm picks the scores of both
// halves by the row codes (read from an LDS ring in the selector's own form);
// larger alphabets read a byte or 16-bit profile of the strip from LDS.
//
// Best cell (forward).  E' leaving a lane is at least every Ho of its row less the
// extensions in between, so one comparison of it with the lane's threshold decides
// whether the row can hold a new best; only then the row's H values are formed,
// their maximum taken and the row kept.  The threshold is the lane's best, raised
// every 32 steps to one below the best of its whole group (a smaller value cannot
// win; an equal one still can, by a smaller row).
//
// Reverse pass.  Where both passes have the same sequence as rows, every alignment
// that reaches the target starts on row 0 of the reversed box (the forward winner is
// the first row with that score) and its partial scores stay positive.  The strict
// form therefore floors values at -kRevLow instead of zero once all lanes have left
// the rows before row 0: alignments that start on later rows stay far below, no
// hit is lost, and none appears (such an alignment is worth at most the target
// less kRevLow).  Every 32 steps the pass ends if no value in flight is positive and
// within reach of the target, given what the columns after it can add at most.  (The
// static row bound of reverse_task alone: 1M-pair DNA mix 25.6 -> 24.4 ms, 10k long
// proteins, whose box is three times as high as the alignment, 71.9 -> 64.3 ms.)
//
// What bounds it: VALU issue (one instruction per SIMD and four cycles, packed or
// not).  A step of K columns takes 6 K + about 8 instructions and, in the forward
// pass, 2.5 K + 6 more in the steps that may improve the best.  Measured against the
// kernels it replaced (f16 cells with the gap steps as instructions and a byte
// profile, int16 cells; 8 and 9 instructions per two cells and a maximum tree per
// row): the 1M-pair DNA mix 32.3 -> 26.3 ms per batch, its K = 5 bucket alone
// 4.42 -> 3.62 ms (1.70e10 cells), 20k proteins 2.72 -> 2.47 ms, 10k long proteins
// 150.2 -> 124.9 ms.
#pragma once
#include <type_traits>

#include "gbsw_device.hpp"
#include "gbsw_kernel_args.hpp"
#include "gbsw_kernels.hpp"
#include "gbsw_pass.hpp"

namespace gbsw {

// A score no cell reaches (above every sat_limit's pairs that are not recomputed
// only in groups without a pair, whose cells stay zero).
constexpr int kUnreached = 0x7000;

struct SweepSmem {
    uint8_t* base;
    SweepLds L;
    __device__ uint8_t* lut() const { return base + L.lut_off; }
    __device__ int16_t* sub() const { return (int16_t*)(base + L.sub_off); }
    __device__ int16_t* colmax() const { return (int16_t*)(base + L.colmax_off); }
    __device__ uint16_t* row_tab() const { return (uint16_t*)(base + L.row_tab_off); }
    __device__ uint32_t* col_tab() const { return (uint32_t*)(base + L.col_tab_off); }
    __device__ uint8_t* group(int g) const { return base + L.group_off + g * L.group_bytes; }
};
constexpr uint16_t kPadSelector = 0x0C0C; // two zero bytes

// x and y rotated right by one lane inside the group, each less d: the DPP operand
// of the subtraction.  (Written as asm, with the two wait states a DPP read of a
// fresh VALU result needs: the compiler kept the moves apart from the subtractions.)
template <int G>
__device__ __forceinline__ void group_left(uint32_t x, uint32_t y, uint32_t d, uint32_t& xo, uint32_t& yo)
{
    static_assert(G == 16 || G == 64, "group");
    if constexpr (G == 16)
        asm volatile("s_nop 1\n\t"
                     "v_sub_u32_dpp %0, %2, %4 row_ror:1 row_mask:0xf bank_mask:0xf\n\t"
                     "v_sub_u32_dpp %1, %3, %4 row_ror:1 row_mask:0xf bank_mask:0xf"
                     : "=&v"(xo), "=v"(yo)
                     : "v"(x), "v"(y), "v"(d));
    else
        asm volatile("s_nop 1\n\t"
                     "v_sub_u32_dpp %0, %2, %4 wave_ror:1 row_mask:0xf bank_mask:0xf\n\t"
                     "v_sub_u32_dpp %1, %3, %4 wave_ror:1 row_mask:0xf bank_mask:0xf"
                     : "=&v"(xo), "=v"(yo)
                     : "v"(x), "v"(y), "v"(d));
}
template <int N>
__device__ __forceinline__ uint32_t row_ror(uint32_t v)
{
    return (uint32_t)__builtin_amdgcn_mov_dpp((int)v, 0x120 + N, 0xf, 0xf, false);
}

// Per-lane constants of the fix-up after the rotation: in a group's first lane the
// low virtual lane (0) takes the strip boundary and the high one (G) the rotated
// low half (virtual lane G - 1); other lanes keep the rotated value.
struct GroupFix {
    bool first;
    uint32_t selh, sele; // v_perm selectors with the boundary's H (low) or E (high) half
};
__device__ __forceinline__ GroupFix group_fix(int l)
{
    GroupFix f;
    f.first = l == 0;
    f.selh = l == 0 ? 0x05040100u : 0x07060504u;
    f.sele = l == 0 ? 0x05040302u : 0x07060504u;
    return f;
}

// Sweep16: the cells of a lane's two virtual lanes in the 16-bit halves of one
// register.  U: a wave-uniform value, in both halves.  Sums and differences are
// 32-bit operations (four-byte encodings that take a scalar operand): no half
// carries or borrows while values stay in range.
struct Sweep16 {
    using V = uint32_t;
    using U = uint32_t;
    using B = uint32_t; // strip boundary entry: H | E << 16
    static constexpr bool kWide = false, kShifts = false;
    __device__ static U uni(int32_t x) { return (uint32_t)x * 0x00010001u; }
    __device__ static V from(U u) { return u; }
    __device__ static V splat(int32_t x) { return uni(x); }
    __device__ static V pair(int32_t lo, int32_t hi) { return pack16(lo, hi); }
    __device__ static V bytes(uint32_t w) { return w; } // scores picked by v_perm, one per half
    __device__ static V addu(V a, U u) { return a + u; }
    __device__ static V subu(V a, U u) { return a - u; }
    __device__ static V sub_each(V a, U u) { return raw(as_u(a) - as_u(u)); } // no borrow between the halves
    // + scores: 32-bit while they are non-negative, else per half
    template <bool SIGNED>
    __device__ static V add(V a, V b, U)
    {
        if constexpr (SIGNED) return raw(as_u(a) + as_u(b));
        else return a + b;
    }
    __device__ static V max3(V a, V b, V c) { return pk_max3_f16(a, b, c); }
    __device__ static V max3u(V a, V b, U c) { return pk_max3_f16(a, b, c); }
    __device__ static V vmax(V a, V b) { return pk_max(a, b); }
    __device__ static V vmax3(V a, V b, V c) { return pk_max3_f16(a, b, c); }
    // the left neighbour's values, less the offset between the two lanes
    template <int G>
    __device__ static void left(V x, V y, V d, V& xo, V& yo) { group_left<G>(x, y, d, xo, yo); }
    __device__ static void keep(V& x) { asm volatile("" : "+v"(x)); }
    __device__ static V fix_h(V x, B bnd, const GroupFix& f) { return __builtin_amdgcn_perm(x, bnd, f.selh); }
    __device__ static V fix_e(V x, B bnd, const GroupFix& f) { return __builtin_amdgcn_perm(x, bnd, f.sele); }
    // zero-score boundary at offsets zh (H) and ze (E); entries less / plus offsets
    __device__ static B bnd_zero(int32_t zh, int32_t ze) { return (uint32_t)zh | ((uint32_t)ze << 16); }
    __device__ static B first_bnd(U z, int32_t go) { return z - (uint32_t)go; } // zero scores, left of the first strip
    __device__ static B bnd_add(B b, int32_t zh, int32_t ze) { return b + bnd_zero(zh, ze); }
    __device__ static B bnd_sub(B b, int32_t zh, int32_t ze) { return b - bnd_zero(zh, ze); }
    __device__ static B bnd_out(V h, V e) { return __builtin_amdgcn_perm(e, h, 0x07060302u); } // high halves
    __device__ static V words(const uint32_t* plo, const uint32_t* phi, int k)
    {
        return (k & 1) ? __builtin_amdgcn_perm(phi[k / 2], plo[k / 2], 0x07060302u)
                       : __builtin_amdgcn_perm(phi[k / 2], plo[k / 2], 0x05040100u);
    }
    // x exceeds the threshold in some half
    __device__ static bool exceeds(V x, V thr) { return raw(__builtin_elementwise_sub_sat(as_u(x), as_u(thr))) != 0u; }
    __device__ static V ltmask(V a, V b) { return pk_lt_mask(a, b); }
    __device__ static V sel(V m, V a, V b) { return bfi(m, a, b); }
    __device__ static V sel_step(V m, int s, V b) { return bfi_s(m, (uint32_t)__builtin_amdgcn_readfirstlane((int)pack16(s, s)), b); }
    __device__ static V less1(V x) { return raw(__builtin_elementwise_sub_sat(as_u(x), (u16x2){1, 1})); }
    __device__ static int32_t lo(V x) { return (int32_t)(x & 0xFFFFu); }
    __device__ static int32_t hi(V x) { return (int32_t)(x >> 16); }
    // maximum over both halves of the group's lanes, in both halves of each lane
    template <int G>
    __device__ static V group_max(V x)
    {
        V m = pk_max(x, (x >> 16) | (x << 16));
        m = pk_max(m, row_ror<1>(m));
        m = pk_max(m, row_ror<2>(m));
        m = pk_max(m, row_ror<4>(m));
        m = pk_max(m, row_ror<8>(m));
        if constexpr (G == 64) {
            uint32_t r = 0;
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const uint32_t v = (uint32_t)__builtin_amdgcn_readlane((int)m, 16 * q) & 0xFFFFu;
                r = v > r ? v : r;
            }
            m = r * 0x00010001u;
        }
        return m;
    }
    __device__ static B load_bnd(const B* p) { return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
    __device__ static B zero_bnd() { return 0u; }
};

// The same where the byte tables hold the scores from the smallest one up: the rest of
// score + open + extend (KernelArgs::shift) is the third operand of the addition, whose
// halves do not carry or borrow either.  Apart from Sweep16, since the longer encoding
// costs every step (1M-pair DNA mix 21.9 -> 22.1 ms, 10k long proteins 64.0 -> 65.4).
struct Sweep16Shifted : Sweep16 {
    static constexpr bool kShifts = true;
    template <bool SIGNED>
    __device__ static V add(V a, V b, U shift)
    {
        static_assert(!SIGNED, "byte forms");
        return a + b + shift;
    }
};

// Sweep32: the same two virtual lanes as two int32 registers, for pairs whose score
// may exceed the 16-bit range.
struct Sweep32 {
    struct V {
        int32_t l, h;
    };
    using U = int32_t;
    using B = uint2; // (H, E)
    static constexpr bool kWide = true, kShifts = false;
    __device__ static U uni(int32_t x) { return x; }
    __device__ static V from(U u) { return V{u, u}; }
    __device__ static V splat(int32_t x) { return V{x, x}; }
    __device__ static V pair(int32_t lo, int32_t hi) { return V{lo, hi}; }
    __device__ static V addu(V a, U u) { return V{a.l + u, a.h + u}; }
    __device__ static V subu(V a, U u) { return V{a.l - u, a.h - u}; }
    __device__ static V sub_each(V a, U u) { return subu(a, u); }
    template <bool SIGNED>
    __device__ static V add(V a, V b, U) { return V{a.l + b.l, a.h + b.h}; }
    __device__ static V vmax(V a, V b) { return V{max(a.l, b.l), max(a.h, b.h)}; }
    __device__ static V max3(V a, V b, V c) { return V{max(max(a.l, b.l), c.l), max(max(a.h, b.h), c.h)}; }
    __device__ static V max3u(V a, V b, U c) { return V{max(max(a.l, b.l), c), max(max(a.h, b.h), c)}; }
    __device__ static V vmax3(V a, V b, V c) { return max3(a, b, c); }
    __device__ static void keep(V& x) { asm volatile("" : "+v"(x.l), "+v"(x.h)); }
    template <int G>
    __device__ static void left(V x, V y, V d, V& xo, V& yo)
    {
        uint32_t xl, xh, yl, yh;
        group_left<G>((uint32_t)x.l, (uint32_t)y.l, (uint32_t)d.l, xl, yl);
        group_left<G>((uint32_t)x.h, (uint32_t)y.h, (uint32_t)d.h, xh, yh);
        xo = V{(int32_t)xl, (int32_t)xh};
        yo = V{(int32_t)yl, (int32_t)yh};
    }
    __device__ static V fix_h(V x, B bnd, const GroupFix& f)
    {
        return V{f.first ? (int32_t)bnd.x : x.l, f.first ? x.l : x.h};
    }
    __device__ static V fix_e(V x, B bnd, const GroupFix& f)
    {
        return V{f.first ? (int32_t)bnd.y : x.l, f.first ? x.l : x.h};
    }
    __device__ static B bnd_zero(int32_t zh, int32_t ze) { return make_uint2((uint32_t)zh, (uint32_t)ze); }
    __device__ static B first_bnd(U z, int32_t go) { return bnd_zero(z - go, z); }
    __device__ static B bnd_add(B b, int32_t zh, int32_t ze) { return make_uint2(b.x + (uint32_t)zh, b.y + (uint32_t)ze); }
    __device__ static B bnd_sub(B b, int32_t zh, int32_t ze) { return make_uint2(b.x - (uint32_t)zh, b.y - (uint32_t)ze); }
    __device__ static B bnd_out(V h, V e) { return make_uint2((uint32_t)h.h, (uint32_t)e.h); }
    __device__ static V bytes(uint32_t w) { return V{(int32_t)(w & 0xFFFFu), (int32_t)(w >> 16)}; }
    __device__ static V words(const uint32_t* plo, const uint32_t* phi, int k)
    {
        const int sh = (k & 1) * 16;
        return V{(int32_t)(int16_t)(plo[k / 2] >> sh), (int32_t)(int16_t)(phi[k / 2] >> sh)};
    }
    __device__ static bool exceeds(V x, V thr) { return x.l > thr.l || x.h > thr.h; }
    __device__ static V ltmask(V a, V b) { return V{a.l < b.l ? -1 : 0, a.h < b.h ? -1 : 0}; }
    __device__ static V sel(V m, V a, V b) { return V{m.l ? a.l : b.l, m.h ? a.h : b.h}; }
    __device__ static V sel_step(V m, int s, V b) { return V{m.l ? s : b.l, m.h ? s : b.h}; }
    __device__ static V less1(V x) { return V{max(x.l - 1, 0), max(x.h - 1, 0)}; }
    __device__ static int32_t lo(V x) { return x.l; }
    __device__ static int32_t hi(V x) { return x.h; }
    template <int G>
    __device__ static V group_max(V x)
    {
        int32_t m = max(x.l, x.h);
        m = max(m, (int32_t)row_ror<1>((uint32_t)m));
        m = max(m, (int32_t)row_ror<2>((uint32_t)m));
        m = max(m, (int32_t)row_ror<4>((uint32_t)m));
        m = max(m, (int32_t)row_ror<8>((uint32_t)m));
        if constexpr (G == 64) {
            int32_t r = 0;
#pragma unroll
            for (int q = 0; q < 4; ++q) r = max(r, __builtin_amdgcn_readlane(m, 16 * q));
            m = r;
        }
        return V{m, m};
    }
    __device__ static B load_bnd(const B* p)
    {
        const uint64_t v = __hip_atomic_load((const uint64_t*)p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        return make_uint2((uint32_t)v, (uint32_t)(v >> 32));
    }
    __device__ static B zero_bnd() { return make_uint2(0u, 0u); }
};

// Bits 0 .. n - 1 (n clamped to [0, 32]): the columns of a block inside the pair.
__device__ __forceinline__ uint32_t sweep_cols(int n)
{
    return n <= 0 ? 0u : n >= 32 ? 0xFFFFFFFFu : (1u << n) - 1u;
}

// Raw row bytes and boundary entries of the next chunk, on their way to the ring.
template <class A, int N>
struct SweepFetch {
    int32_t b[N];       // residue byte, kNoRow outside [0, nr)
    typename A::B d[N]; // strip boundary (H, E)
};
constexpr int kNoRow = 256; // its entry of the row table is the padding row

// The rings.  ROWB: bytes of a profile row.  MS: the wave has pairs of several
// strips (boundary entries in use).
template <class A, int G, int PF, int ROWB, bool MS>
struct SweepRows {
    static constexpr int N = kChunk / G > 1 ? kChunk / G : 1; // rows per lane and chunk
    static constexpr int R = sweep_ring(G);
    using F = SweepFetch<A, N>;
    __device__ static F none()
    {
        F f;
#pragma unroll
        for (int i = 0; i < N; ++i) { f.b[i] = kNoRow; f.d[i] = A::zero_bnd(); }
        return f;
    }
    // nbnd: boundary rows to read; the others take (none, none)
    __device__ static F fetch(const Task& t, int chunk, int l, const typename A::B* bnd, int nbnd, int none)
    {
        F f;
#pragma unroll
        for (int i = 0; i < N; ++i) {
            const int x = chunk * kChunk + l + G * i;
            const bool v = l < kChunk && x < t.nr;
            f.b[i] = v ? (int32_t)t.rows[t.rev ? t.nr_full - 1 - x : x] : kNoRow;
            // the boundary rows were stored by this workgroup during the previous strip,
            // or by another one of its XCD: an agent-scope load hits no stale L1 line
            f.d[i] = (MS && l < kChunk && x < nbnd) ? A::load_bnd(bnd + x) : A::bnd_zero(none, none);
        }
        return f;
    }
    // codes in the form the step reads (row table), boundary entries with row x's
    // offset.  Every code entry is written twice, a ring length apart, so that a
    // chunk's reads are contiguous wherever it starts.
    __device__ static void store(const F& f, int chunk, int l, uint16_t* ring_code, typename A::B* ring_bnd,
                                 const uint16_t* row_tab, int base, int g, int o)
    {
        if (G > kChunk && l >= kChunk) return;
#pragma unroll
        for (int i = 0; i < N; ++i) {
            const int x = chunk * kChunk + l + G * i;
            const uint32_t c = row_tab[f.b[i]];
            const uint16_t e = (uint16_t)(PF == kProfRegs ? c : c * (uint32_t)ROWB);
            const int at = x & (R - 1);
            if constexpr (PF == kProfRegs) {
                // entry r is a whole v_perm selector, for a lane's rows r (low half) and
                // r - G (high half): each half a score byte (of the low table, of the
                // high one), then a zero byte
                const uint16_t eh = (uint16_t)(e + (e == kPadSelector ? 0 : 4));
                const int ah = (x + G) & (R - 1);
                ring_code[2 * at] = e;
                ring_code[2 * (at + R)] = e;
                ring_code[2 * ah + 1] = eh;
                ring_code[2 * (ah + R) + 1] = eh;
            } else {
                ring_code[at] = e;
                ring_code[at + R] = e;
            }
            if constexpr (MS) {
                const int z = base + g * ((x & (kRebase - 1)) + 1);
                ring_bnd[at] = A::bnd_add(f.d[i], z - o, z);
            }
        }
    }
};

// What the tables add to the scores.
template <class A>
__device__ __forceinline__ int table_bias(const KernelArgs& a)
{
    return A::kShifts ? a.bias : -(a.gap_open + a.gap_extend);
}

// Row table: byte -> code of its row (register form: its half of the selector).
// Column table (register form): byte -> the four biased scores of its column.
template <class A, int PF, class S>
__device__ __forceinline__ void stage_byte_tables(const KernelArgs& a, const S& sm)
{
    const int alpha = a.alpha, sbias = table_bias<A>(a);
    for (int i = threadIdx.x; i <= kNoRow; i += kWave) {
        int c = i < kNoRow ? (int)sm.lut()[i] : alpha;
        c = c > alpha ? alpha : c; // bytes outside the alphabet read the padding row
        sm.row_tab()[i] = PF == kProfRegs ? (uint16_t)(c == alpha ? kPadSelector : 0x0C00 | c) : (uint16_t)c;
        if constexpr (PF == kProfRegs) {
            uint32_t w = 0;
            for (int r = 0; r < alpha; ++r)
                if (c < alpha) w |= (uint32_t)(uint8_t)(sm.sub()[r * alpha + c] + sbias) << (8 * r);
            sm.col_tab()[i] = w;
        }
    }
    __syncthreads();
}

// Profile words of virtual lane v from profile row `row` (form PF): blocks of 16
// bytes for all virtual lanes, then the remainder.
template <int G, int K, int PF>
struct SweepProf {
    static constexpr int COLB = PF == kProfBytes ? 1 : 2;                       // bytes per column
    static constexpr int Q = K * COLB / 16;                                     // full 16-byte blocks
    static constexpr int RB = (PF == kProfBytes ? kstride8(K) : 2 * kstride(K)) - 16 * Q; // remainder bytes
    static constexpr int NW = (16 * Q + RB) / 4;                                // dwords
    static constexpr int VL = 2 * G;
    __device__ static void load(const uint8_t* row, int v, uint32_t (&d)[NW])
    {
#pragma unroll
        for (int q = 0; q < Q; ++q) {
            const uint4 x = *(const uint4*)(row + q * (16 * VL) + v * 16);
            d[4 * q + 0] = x.x; d[4 * q + 1] = x.y; d[4 * q + 2] = x.z; d[4 * q + 3] = x.w;
        }
        const uint8_t* r = row + Q * (16 * VL) + v * RB;
        if constexpr (RB == 16) {
            const uint4 x = *(const uint4*)r;
            d[4 * Q + 0] = x.x; d[4 * Q + 1] = x.y; d[4 * Q + 2] = x.z; d[4 * Q + 3] = x.w;
        } else if constexpr (RB == 12) {
            const uint3 x = *(const uint3*)r;
            d[4 * Q + 0] = x.x; d[4 * Q + 1] = x.y; d[4 * Q + 2] = x.z;
        } else if constexpr (RB == 8) {
            const uint2 x = *(const uint2*)r;
            d[4 * Q + 0] = x.x; d[4 * Q + 1] = x.y;
        } else if constexpr (RB == 4) {
            d[4 * Q] = *(const uint32_t*)r;
        }
    }
    // byte offset within a profile row -> (virtual lane, column of it)
    __device__ static void slot(int at, int& v, int& k)
    {
        if (at < Q * 16 * VL) {
            v = (at & (16 * VL - 1)) >> 4;
            k = ((at / (16 * VL)) * 16 + (at & 15)) / COLB;
        } else {
            const int r = at - Q * 16 * VL;
            v = RB ? r / (RB ? RB : 1) : 0;
            k = (Q * 16 + (r - v * RB)) / COLB;
        }
    }
};

// One pass (REV: the reverse one, target = the score to reach) for the groups of
// the wave; SPLIT: strip io.strip only, its boundary rows passed on through
// io.bnd_in / io.bnd_out as they are published, else every strip with the
// boundary rows in bnd_g.  Winner keys as in gbsw_pass.hpp.
template <class A, int G, int K, int PF, bool REV, bool SPLIT = false>
__device__ __forceinline__ PassResult sweep(const KernelArgs& a, const SweepSmem& sm, const Task& t, int32_t target,
                                            bool strict, typename A::B* bnd_g, const StripIO& io = StripIO{})
{
    using V = typename A::V;
    using U = typename A::U;
    using Bd = typename A::B;
    constexpr int VL = 2 * G, W = VL * K, R = sweep_ring(G);
    constexpr int rowstride = sweep_row_bytes(G, K, PF);
    constexpr int UN = K <= 8 ? kSweepUnroll : 2;
    const int lane = threadIdx.x, g = lane / G, l = lane & (G - 1);
    const int alpha = a.alpha;
    const int ge = -a.gap_extend, go = -a.gap_open, sbias = table_bias<A>(a);
    // offset of the floor (base) and of zero scores (zero)
    const int base = a.base, low = REV && strict ? kRevLow : 0, zero = base + low;
    const GroupFix fix = group_fix(l);
    uint8_t* gb = sm.group(g);
    uint16_t* ring_code = (uint16_t*)(gb + sm.L.ring_code_off);
    Bd* ring_bnd = (Bd*)(gb + sm.L.ring_bnd_off);
    const uint8_t* lut = sm.lut();
    const uint16_t* row_tab = sm.row_tab();
    const uint32_t* col_tab = sm.col_tab();
    const int16_t* sub = sm.sub();

    // wave-uniform extents
    const int strips_g = (t.nr > 0 && t.nc > 0) ? (t.nc + W - 1) / W : 0;
    int strips_max = strips_g, steps_max = t.nr + VL - 1;
#pragma unroll
    for (int x = G; x < kWave; x <<= 1) {
        strips_max = max(strips_max, __shfl_xor(strips_max, x));
        steps_max = max(steps_max, __shfl_xor(steps_max, x));
    }
    strips_max = __builtin_amdgcn_readfirstlane(strips_max);
    steps_max = __builtin_amdgcn_readfirstlane(steps_max);
    // (the host gives four-pair waves pairs of one strip only)
    const bool multi_strip = G == kWave && strips_max > 1;
    const int strip_lo = SPLIT ? io.strip : 0;

    const U gs = A::uni(ge), cs = A::uni(ge - go), hand_u = A::uni(ge * (K - 1)), shift = A::uni(a.shift);
    // (opaque: kept in vector registers, where the DPP subtraction takes it)
    V hand = A::from(hand_u);
    A::keep(hand);
    const int v_lo = l, v_hi = l + G;
    uint64_t cand_lo = 0, cand_hi = 0;
    // forward: the lane's threshold (true scores); reverse: the score to reach.
    // Groups without a pair take one that no cell reaches.
    V bt = A::splat(strips_g > strip_lo ? 0 : kUnreached);
    int ahead = t.ubound;      // reverse: what the columns from the strip's first on can still add
    int avail = 0x7FFFFFFF;    // boundary rows the strip before left (the rest are dead)
    const int tgt = target > 0 ? target : kUnreached;
    const V tgt1 = A::splat(tgt - 1);

    Bd* bnd_rd = SPLIT ? (Bd*)io.bnd_in : bnd_g;
    Bd* bnd_wr = SPLIT ? (Bd*)io.bnd_out : bnd_g;
    const int strip_hi = SPLIT ? min(io.strip + 1, strips_max) : strips_max;
    for (int strip = strip_lo; strip < strip_hi; ++strip) {
        // (opaque: the compiler would keep a pointer per column across the strips)
        int strip_base = __builtin_amdgcn_readfirstlane(strip * W);
        asm volatile("" : "+s"(strip_base));
        const bool live = strip < strips_g;
        const bool use_bnd = strip > 0;
        const bool write_bnd = live && strip + 1 < strips_g;
        // split form: boundary rows [0, n) of the previous strip are readable once
        // its progress word reaches epoch_in | n
        auto need_rows = [&](const int n) {
            if constexpr (SPLIT) {
                if (strip > 0) wait_word(io.prog_in, io.epoch_in | (uint64_t)(uint32_t)n, a.status);
            }
        };
        auto col_byte = [&](const int c) {
            return live && c < t.nc ? (int)t.cols[t.rev ? t.nc_full - 1 - c : c] : kNoRow;
        };
        auto col_code = [&](const int c) { // -1: padding
            const int b = col_byte(c), code = b < kNoRow ? (int)lut[b] : alpha;
            return code < alpha ? code : -1;
        };

        // ---- scores of the strip's columns (a score of 0 after the bias: padding; -1
        // where the bias is 0, so that padding scores are negative)
        const int pad = PF == kProfWords && sbias == 0 ? -1 : 0;
        __syncthreads();
        uint32_t tlo[PF == kProfRegs ? K : 1], thi[PF == kProfRegs ? K : 1];
        if constexpr (PF == kProfRegs) {
#pragma unroll
            for (int k = 0; k < K; ++k) {
                tlo[k] = col_tab[col_byte(strip_base + v_lo * K + k)];
                thi[k] = col_tab[col_byte(strip_base + v_hi * K + k)];
            }
        } else {
            using P = SweepProf<G, K, PF>;
            for (int j4 = l; j4 < rowstride / 4; j4 += G) {
                int code[4];
#pragma unroll
                for (int b = 0; b < 4; b += P::COLB) {
                    int vj, kj;
                    P::slot(j4 * 4 + b, vj, kj);
                    code[b] = kj < K ? col_code(strip_base + vj * K + kj) : -1;
                }
                for (int r = 0; r <= alpha; ++r) {
                    uint32_t w = 0;
#pragma unroll
                    for (int b = 0; b < 4; b += P::COLB) {
                        const int sc = (code[b] >= 0 && r < alpha) ? sub[r * alpha + code[b]] + sbias : pad;
                        w |= ((uint32_t)sc & (P::COLB == 1 ? 0xFFu : 0xFFFFu)) << (8 * b);
                    }
                    *(uint32_t*)(gb + r * rowstride + j4 * 4) = w;
                }
            }
        }
        need_rows(2 * kChunk);

        // reverse, strict: the least score (less one) from which a row of the lane may
        // still reach the target
        V dead = A::splat(kUnreached);
        if constexpr (REV) {
            if (strict) {
                int own[2] = {0, 0};
#pragma unroll
                for (int k = 0; k < K; ++k) {
                    const int cl = col_code(strip_base + v_lo * K + k), ch = col_code(strip_base + v_hi * K + k);
                    own[0] += cl >= 0 ? (int)sm.colmax()[cl] : 0;
                    own[1] += ch >= 0 ? (int)sm.colmax()[ch] : 0;
                }
                int sum[2] = {own[0], own[1]}; // inclusive prefix sums over the lanes
#pragma unroll
                for (int x = 1; x < G; x <<= 1) {
                    const int u0 = __shfl_up(sum[0], x, G), u1 = __shfl_up(sum[1], x, G);
                    if (l >= x) { sum[0] += u0; sum[1] += u1; }
                }
                const int all0 = __shfl(sum[0], G - 1, G), all1 = __shfl(sum[1], G - 1, G);
                if (target > 0 && live) {
                    const int r0 = ahead - (sum[0] - own[0]), r1 = ahead - all0 - (sum[1] - own[1]);
                    dead = A::pair(max(0, tgt - 1 - r0), max(0, tgt - 1 - r1));
                }
                ahead -= all0 + all1;
            }
        }

        // state before step 0: zero scores at the offsets of step -1
        V Ho[K], F[K];
        V snap[REV ? 1 : K];
#pragma unroll
        for (int k = 0; k < K; ++k) {
            Ho[k] = A::from(A::uni(zero + ge * k) + cs);
            F[k] = A::from(A::uni(zero));
        }
#pragma unroll
        for (int k = 0; k < (REV ? 1 : K); ++k) snap[k] = A::from(A::uni(0));
        V Eout = A::from(A::uni(zero + ge * K)), Hd0 = A::from(A::uni(zero - go));
        V bstep = A::from(A::uni(0)); // step of the first row reaching the lane's best
        int32_t rt_lo = 0x7FFFFFFF, rr_lo = 0, rt_hi = 0x7FFFFFFF, rr_hi = 0; // reverse hits
        bool dirty = false; // some lane's best moved since the group's was last shared

        // Rows [r0, r0 + 32) of the outgoing boundary, parked in their ring slots with
        // the offsets of the step that wrote them, go to global memory as true scores
        auto flush_bnd = [&](const int r0) {
            if (write_bnd) {
#pragma unroll
                for (int i = 0; i < (kChunk / G > 1 ? kChunk / G : 1); ++i) {
                    const int row = r0 + l + G * i;
                    if (l < kChunk && row >= 0 && row < t.nr) {
                        const int z = base + ge * (((row + VL - 1) & (kRebase - 1)) + 1 + K);
                        bnd_wr[row] = A::bnd_sub(ring_bnd[row & (R - 1)], z - go, z);
                    }
                }
            }
        };
        auto share_best = [&]() {
            if constexpr (!REV) bt = A::vmax(bt, A::less1(A::template group_max<G>(bt)));
        };

        // waves of single-strip pairs read no boundary column and hand none on; the
        // two forms are separate loops so that neither holds the other's registers
        auto chunks = [&](auto ms) {
            constexpr bool MS = decltype(ms)::value;
            using Rows = SweepRows<A, G, PF, rowstride, MS>;
            // row ring: 2G padding rows, rows [0, 32) now, [32, 64) in flight
            for (int c = -(VL / kChunk); c < 0; ++c)
                Rows::store(Rows::none(), c, l, ring_code, ring_bnd, row_tab, base, ge, go);
            // boundary rows to read, and the entry of the first strip's rows (zero
            // scores; strict: from row 2G on the floor)
            const int nbnd = use_bnd ? min(avail, t.nr) : 0;
            auto first_rows = [&](const int chunk) { return !use_bnd && chunk * kChunk < VL ? low : 0; };
            Rows::store(Rows::fetch(t, 0, l, bnd_rd, nbnd, first_rows(0)), 0, l, ring_code, ring_bnd, row_tab, base, ge, go);
            typename Rows::F pf = Rows::fetch(t, 1, l, bnd_rd, nbnd, first_rows(1));
            const int last_in = use_bnd ? min(avail, steps_max) : 0; // live boundary rows enter until then
            int s_stop = steps_max; // steps run
            for (int s0 = 0; s0 < steps_max; s0 += kChunk) {
                // refill: rows of chunk (s0/32 + 1) enter the ring, chunk + 2 is requested
                {
                    const int ck = s0 / kChunk + 1;
                    Rows::store(pf, ck, l, ring_code, ring_bnd, row_tab, base, ge, go);
                    if constexpr (MS) need_rows((ck + 2) * kChunk);
                    pf = Rows::fetch(t, ck + 1, l, bnd_rd, nbnd, first_rows(ck + 1));
                }
                __syncthreads();
                // rows leaving the last virtual lane during the previous chunk
                if (MS && s0 > 0) {
                    flush_bnd(s0 - kChunk - (VL - 1));
                    if constexpr (SPLIT) {
                        // rows below s0 - (2G - 1) are stored once the flush completes: the
                        // wait for it (publish_word) is hidden by the other waves of the SIMD
                        if (strip + 1 < strips_max && s0 >= VL)
                            publish_word(io.prog_out, io.epoch_out | (uint64_t)(uint32_t)(s0 - (VL - 1)));
                    }
                }
                if (s0 > 0 && (s0 & (kRebase - 1)) == 0) {
                    const U d = A::uni(ge * kRebase);
#pragma unroll
                    for (int k = 0; k < K; ++k) { Ho[k] = A::subu(Ho[k], d); F[k] = A::subu(F[k], d); }
                    Eout = A::subu(Eout, d);
                    Hd0 = A::subu(Hd0, d);
                }
                if (!REV && dirty) {
                    share_best();
                    dirty = false;
                }
                // strict reverse pass: over once no value in flight can reach the target (a
                // split strip with a successor runs on: its rows are announced one by one)
                if (REV && strict && s0 >= VL && s0 >= last_in && !(SPLIT && strip + 1 < strips_max)) {
                    V m = A::vmax(Hd0, Ho[0]);
#pragma unroll
                    for (int k = 1; k < K; ++k) m = A::vmax(m, Ho[k]);
                    // (Hd0 has the smallest offset of them)
                    const U zd = A::uni(zero + ge * ((s0 & (kRebase - 1)) - 1)) + cs;
                    if (__ballot(A::exceeds(m, A::addu(dead, zd))) == 0) {
                        s_stop = s0;
                        break;
                    }
                }
                const int s_end = min(s0 + kChunk, steps_max);
                struct StepIn {
                    uint32_t w[PF == kProfRegs ? 1 : 2 * SweepProf<G, K, PF>::NW];
                    Bd bnd;
                };
                // this chunk's entries are contiguous in the rings (profile forms: the rows of
                // virtual lane v_lo lie G entries on from those of v_hi)
                using Code = std::conditional_t<PF == kProfRegs, uint32_t, uint16_t>;
                const Code* rc0 = (const Code*)ring_code + ((s0 - (PF == kProfRegs ? v_lo : v_hi)) & (R - 1));
                const Bd* pb0 = ring_bnd + (s0 & (R - 1));
                // a step's row codes (profile forms: read two steps ahead, the profile
                // words they address one step ahead)
                struct Rc {
                    uint32_t lo, hi;
                };
                auto codes = [&](const Code* rc) {
                    if constexpr (PF == kProfRegs) return Rc{*rc, 0u};
                    else return Rc{rc[G], rc[0]};
                };
                auto fetch = [&](StepIn& in, const Rc c, const Bd* pb) {
                    if constexpr (PF == kProfRegs) {
                        in.w[0] = c.lo;
                    } else {
                        using P = SweepProf<G, K, PF>;
                        uint32_t wl[P::NW], wh[P::NW];
                        P::load(gb + c.lo, v_lo, wl);
                        P::load(gb + c.hi, v_hi, wh);
#pragma unroll
                        for (int q = 0; q < P::NW; ++q) { in.w[q] = wl[q]; in.w[P::NW + q] = wh[q]; }
                    }
                    if constexpr (MS) in.bnd = *pb;
                };
                auto step = [&](const int s, const StepIn& in, const U z, const U zf, const V thr) {
                    // left inputs at this lane's column -1 and, for E, column 0
                    const Bd bnd = MS ? in.bnd : A::first_bnd(zf, go);
                    V xH, xE;
                    A::template left<G>(Ho[K - 1], Eout, hand, xH, xE);
                    xH = A::fix_h(xH, bnd, fix);
                    xE = A::fix_e(xE, bnd, fix);
                    V E = xE, Hd = Hd0;
#pragma unroll
                    for (int k = 0; k < K; ++k) {
                        V S;
                        if constexpr (PF == kProfRegs) {
                            S = A::bytes(__builtin_amdgcn_perm(thi[k], tlo[k], in.w[0]));
                        } else if constexpr (PF == kProfBytes) {
                            constexpr uint32_t pick = 0x0C000C00u | (4u << 16);
                            const uint32_t b = (uint32_t)(k & 3);
                            S = A::bytes(__builtin_amdgcn_perm(in.w[SweepProf<G, K, PF>::NW + k / 4], in.w[k / 4],
                                                               pick + b + (b << 16)));
                        } else {
                            S = A::words(in.w, in.w + SweepProf<G, K, PF>::NW, k);
                        }
                        const V D = A::template add<PF == kProfWords>(Hd, S, shift);
                        Hd = Ho[k];
                        const V H = A::max3(D, E, F[k]);
                        const V ho = A::addu(H, cs);
                        E = A::max3u(E, ho, zf + (U)(k + 1) * gs);
                        F[k] = A::vmax(F[k], ho);
                        Ho[k] = ho;
                    }
                    Eout = E;
                    Hd0 = xH;
                    if constexpr (MS) {
                        if (write_bnd && l == G - 1) ring_bnd[(s - v_hi) & (R - 1)] = A::bnd_out(Ho[K - 1], Eout);
                    }
                    // true scores of the row: Ho less its offset
                    const U zc = z + cs;
                    if constexpr (!REV) {
                        if (__ballot(A::exceeds(Eout, thr)) != 0) {
                            V h[K];
#pragma unroll
                            for (int k = 0; k < K; ++k) h[k] = A::subu(Ho[k], zc + (U)k * gs);
                            const V nb = tree_max<A, K>(h);
                            const V m = A::ltmask(bt, nb);
                            bstep = A::sel_step(m, s, bstep);
#pragma unroll
                            for (int k = 0; k < K; ++k) snap[k] = A::sel(m, h[k], snap[k]);
                            bt = A::vmax(bt, nb);
                            dirty = true;
                        }
                    } else {
                        if (__ballot(A::exceeds(Eout, thr)) != 0) {
                            const int row_lo = s - v_lo, row_hi = s - v_hi;
                            // first (smallest) column of this row that reaches the target
                            uint32_t m_lo = 0, m_hi = 0;
#pragma unroll
                            for (int k = K - 1; k >= 0; --k) {
                                const V h = A::sub_each(Ho[k], zc + (U)k * gs); // (may be negative)
                                m_lo = 2 * m_lo + (A::lo(h) == tgt ? 1u : 0u);
                                m_hi = 2 * m_hi + (A::hi(h) == tgt ? 1u : 0u);
                            }
                            m_lo &= sweep_cols(t.nc - (strip_base + v_lo * K));
                            m_hi &= sweep_cols(t.nc - (strip_base + v_hi * K));
                            const int k_lo = m_lo ? __builtin_ctz(m_lo) : K, k_hi = m_hi ? __builtin_ctz(m_hi) : K;
                            if (k_lo < K && row_lo >= 0 && row_lo < t.nr && strip_base + v_lo * K + k_lo < rt_lo) {
                                rt_lo = strip_base + v_lo * K + k_lo;
                                rr_lo = row_lo;
                            }
                            if (k_hi < K && row_hi >= 0 && row_hi < t.nr && strip_base + v_hi * K + k_hi < rt_hi) {
                                rt_hi = strip_base + v_hi * K + k_hi;
                                rr_hi = row_hi;
                            }
                        }
                    }
                };
                {
                    const Code* rc = rc0;
                    const Bd* pb = pb0;
                    // offset of column 0 at step s0; steps past steps_max only meet padding rows
                    U z = A::uni(zero + ge * ((s0 & (kRebase - 1)) + 1));
                    // and that of the floor: zero scores while lanes may still be above row 0
                    const U down = A::uni(REV && s0 >= VL ? low : 0);
                    StepIn ia, ib;
                    fetch(ia, codes(rc), pb);
                    Rc cn = codes(rc + 1);
                    for (int s = s0; s < s_end; s += UN) {
                        // a row of the iteration may improve the best (reach the target) only if E
                        // leaving the lane exceeds this: best - o - g (K - 1) at the first step's offset
                        const V thr = A::addu(REV ? tgt1 : bt, z + cs);
#pragma unroll
                        for (int u = 0; u < UN; u += 2) {
                            fetch(ib, cn, pb + 1);
                            cn = codes(rc + 2);
                            step(s + u, ia, z, z - down, thr);
                            z += gs;
                            fetch(ia, cn, pb + 2);
                            cn = codes(rc + 3);
                            step(s + u + 1, ib, z, z - down, thr);
                            z += gs;
                            rc += 2;
                            pb += 2;
                        }
                    }
                }
            }
            return s_stop;
        };
        int s_stop;
        if constexpr (G == kWave) {
            if (multi_strip) s_stop = chunks(std::true_type{});
            else s_stop = chunks(std::false_type{});
        } else {
            s_stop = chunks(std::false_type{});
        }
        if (multi_strip) {
            // the last chunk's rows; complete before the next strip reads them (after an
            // early end the rows below s_stop - (2G - 1) are there, and no others count)
            __syncthreads();
            if (s_stop == steps_max) flush_bnd(((steps_max - 1) & ~(kChunk - 1)) - (VL - 1));
            avail = s_stop == steps_max ? 0x7FFFFFFF : max(0, s_stop - (VL - 1));
            if constexpr (SPLIT) {
                if (strip + 1 < strips_max) publish_word(io.prog_out, io.epoch_out | 0xFFFFFFFFull);
            } else {
                asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            }
        }

        // ---- candidates of this strip
        if constexpr (!REV) {
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                int32_t b = 0;
#pragma unroll
                for (int k = 0; k < K; ++k) b = max(b, h ? A::hi(snap[k]) : A::lo(snap[k]));
                if (live && b > 0) {
                    const int32_t row = (h ? A::hi(bstep) : A::lo(bstep)) - (h ? v_hi : v_lo);
                    const int col0 = strip_base + (h ? v_hi : v_lo) * K;
                    uint32_t pbest = 0xFFFFFFFFu;
#pragma unroll
                    for (int k = 0; k < K; ++k) {
                        const int32_t v = h ? A::hi(snap[k]) : A::lo(snap[k]);
                        const int col = col0 + k;
                        if (v == b && col < t.nc) pbest = min(pbest, tie_prio((uint32_t)col));
                    }
                    if (pbest != 0xFFFFFFFFu && row < t.nr) {
                        const uint64_t key = ((uint64_t)b << 40) | ((uint64_t)(0xFFFFFu - (uint32_t)row) << 20) |
                                             (uint64_t)(0xFFFFFu - pbest);
                        if (h) cand_hi = key > cand_hi ? key : cand_hi;
                        else cand_lo = key > cand_lo ? key : cand_lo;
                    }
                }
            }
            // a later strip's cells below the best so far cannot win
            if (strip + 1 < strip_hi) {
                const V m = A::less1(A::template group_max<G>(bt));
                bt = strip + 1 < strips_g ? m : A::splat(kUnreached);
            }
        } else {
            if (live && rt_lo != 0x7FFFFFFF) {
                const uint64_t key = ((uint64_t)(0xFFFFFu - (uint32_t)rt_lo) << 20) | (uint64_t)(0xFFFFFu - (uint32_t)rr_lo);
                cand_lo = key > cand_lo ? key : cand_lo;
            }
            if (live && rt_hi != 0x7FFFFFFF) {
                const uint64_t key = ((uint64_t)(0xFFFFFu - (uint32_t)rt_hi) << 20) | (uint64_t)(0xFFFFFu - (uint32_t)rr_hi);
                cand_hi = key > cand_hi ? key : cand_hi;
            }
            // a later strip only holds larger columns: stop once every group has a hit
            const uint64_t found = __ballot((cand_lo | cand_hi) != 0);
            const uint64_t mine = G == kWave ? ~0ull : (((1ull << (G & 63)) - 1) << (G * g));
            if (__ballot(strips_g > strip + 1 && (found & mine) == 0) == 0) break;
        }
    }

    // ---- reduce the candidates of each group
    uint64_t key = cand_lo > cand_hi ? cand_lo : cand_hi;
#pragma unroll
    for (int x = 1; x < G; x <<= 1) {
        const uint64_t o = ((uint64_t)(uint32_t)__shfl_xor((int)(uint32_t)(key >> 32), x) << 32) |
                           (uint32_t)__shfl_xor((int)(uint32_t)key, x);
        key = o > key ? o : key;
    }
    if constexpr (!REV && !A::kWide) {
        // The thresholds never fall (but by one from strip to strip).  A row that a lane
        // kept may have been replaced where the pair is past its range, by padding rows or
        // columns, whose values then mean nothing: such a pair is recomputed.
        const int32_t top = A::lo(A::template group_max<G>(bt)) + strips_g;
        if (strips_g > strip_lo && top >= a.sat_limit) key = max(key, (uint64_t)top << 40);
    }
    PassResult r;
    r.key = key;
    return r;
}

template <class A, int G, int PF>
__device__ __forceinline__ SweepSmem sweep_smem(uint8_t* mem, const KernelArgs& a)
{
    SweepLds L = sweep_lds(G, a.kmax, PF, a.alpha, (int)sizeof(typename A::B));
    // an opaque group offset keeps the compiler from splitting the layout's rounding
    // constants into the profile address (see make_smem of the int16 kernels)
    asm volatile("" : "+s"(L.group_off));
    return SweepSmem{mem, L};
}

// Both passes of one set of pairs, and its results.
template <class A, int G, int K, int PF>
__device__ __forceinline__ void sweep_set(const KernelArgs& a, const SweepSmem& sm, int64_t p, typename A::B* bnd_g)
{
    const int l = threadIdx.x & (G - 1);
    // the forward pass, then (asymmetric tables, wave-uniform) the forward-style
    // pass over the reversed boxes that need their own maximum: one call site
    Task tf = forward_task(a, p);
    FwdOut f{0, 0, 0};
    RevPlan rp;
#pragma nounroll
    for (int fp = 0;; ++fp) {
        const PassResult rf = sweep<A, G, K, PF, false>(a, sm, tf, 0, false, bnd_g);
        if (fp == 0) {
            f = forward_result<G>(a, p, rf.key);
            rp = reverse_plan<G>(a, sm, p, f);
            if (__ballot(rp.gen) == 0) break;
            tf = rp.gen ? rp.t : empty_task(a, 1);
        } else {
            reverse_plan_finish<G>(a, p, rf.key, rp);
            break;
        }
    }
    const bool strict = __ballot(rp.gen || (p >= 0 && f.score > 0 && reverse_swaps(a, p, f))) == 0;
    const PassResult rr = sweep<A, G, K, PF, true>(a, sm, rp.t, rp.target, strict, bnd_g);
    int32_t rb, qb;
    reverse_result(a, p, f, rp.t, rp.target, rr.key, &rb, &qb);
    if (p >= 0 && l == 0 && f.score >= 0 && !rp.saturated) {
        a.out[kOutScore * a.n + p] = f.score;
        a.out[kOutRefEnd * a.n + p] = f.ref_end;
        a.out[kOutQueryEnd * a.n + p] = f.query_end;
        a.out[kOutRefBegin * a.n + p] = rb;
        a.out[kOutQueryBegin * a.n + p] = qb;
    }
}

// Persistent workgroups (one wave) pull sets of 64/G pairs from a device work queue,
// longest first, and run forward then reverse back to back.  One launch holds every
// geometry of its list: the sets' geometries come from a.ranges, so the waves run
// through all of them without a gap and the launch has one tail.  (One launch per
// geometry, sixteen on the 1M-pair DNA mix, left each its own tail and the hardware
// queues unevenly loaded: 26.3-27.5 ms against 25.7 ms; 150k pairs 9.4 against 5.0.)
// WIDE: the four-pair geometries of K >= 10, whose registers leave room for fewer
// waves.
template <class A>
constexpr int sweep_group_waves(int G, bool WIDE) { return A::kWide ? 2 : G == 16 && WIDE ? 3 : 4; }
template <class A, int G, int PF, bool WIDE>
__global__ __launch_bounds__(64, sweep_group_waves<A>(G, WIDE)) void k_sweep(KernelArgs a)
{
    extern __shared__ __align__(16) uint8_t smem_raw[];
    constexpr int PW = kWave / G;
    const SweepSmem sm = sweep_smem<A, G, PF>(smem_raw, a);
    stage_tables(a, sm);
    stage_byte_tables<A, PF>(a, sm);
    const int g = threadIdx.x / G;
    typename A::B* bnd_g = (typename A::B*)a.bnd + ((int64_t)blockIdx.x * PW + g) * a.bnd_rows;
    const int64_t nsets = (a.order_n + PW - 1) / PW;
    for (;;) {
        uint32_t q = 0;
        if (threadIdx.x == 0) q = atomicAdd(a.queue, 1u);
        q = (uint32_t)__builtin_amdgcn_readfirstlane((int)q);
        if ((int64_t)q >= nsets) break;
        const int64_t p = slot_pair(a, (int64_t)q * PW + g);
        // (the host fails a plan whose ranges do not reach the last pair; starting from the
        // last range's K takes 266 to 271 us for the 300 reads that take 261 so)
        int K = 0;
        for (int r = a.nranges - 1; r >= 0; --r)
            if ((int64_t)q * PW < a.ranges[r].end) K = a.ranges[r].K;
#define GBSW_CASE(k) case k: sweep_set<A, G, k, PF>(a, sm, p, bnd_g); break;
        if constexpr (A::kWide) {
            switch (K) { GBSW_SWEEP_K32(GBSW_CASE) }
        } else if constexpr (G == kWave) {
            switch (K) { GBSW_SWEEP_K64(GBSW_CASE) }
        } else if constexpr (WIDE) {
            switch (K) { GBSW_SWEEP_K16_WIDE(GBSW_CASE) }
        } else {
            switch (K) { GBSW_SWEEP_K16(GBSW_CASE) }
        }
#undef GBSW_CASE
    }
}

// Split form: a set's strips run on different workgroups, pipelined on the boundary
// rows.  The protocol is that of k_split (gbsw_kernels.hip): one work counter and
// set of boundary slots per XCD, items in (pass, set, strip) order, each slot
// released once per epoch by the strip that read it; every wait is for an item
// taken from the counter earlier, which holds its workgroup until it finishes,
// and is bounded by kSpinTicks besides.
template <class A, int G, int K, int PF>
__global__ __launch_bounds__(64, A::kWide ? 2 : K <= 6 ? 4 : 3) void k_sweep_split(KernelArgs a)
{
    extern __shared__ __align__(16) uint8_t smem_raw[];
    constexpr int PW = kWave / G;
    const SweepSmem sm = sweep_smem<A, G, PF>(smem_raw, a);
    stage_tables(a, sm);
    stage_byte_tables<A, PF>(a, sm);
    const int l = threadIdx.x & (G - 1), g = threadIdx.x / G;
    const int x = (int)(blockIdx.x % kXcds);
    const SplitArgs& sp = a.split;
    split_check_placement(sp, x, a.status);
    // as in k_split: the chain of waits goes first
    if (sp.first) __builtin_amdgcn_s_setprio(3);
    else __builtin_amdgcn_s_setprio(2);
    const int64_t nsets = (a.order_n + PW - 1) / PW;
    const int64_t nsets_x = nsets > x ? (nsets - x + kXcds - 1) / kXcds : 0;
    const int64_t per_pass = nsets_x * sp.strips;
    typename A::B* bnd = (typename A::B*)a.bnd;
    const int64_t slot0 = (int64_t)x * sp.slots;
    auto slot_bnd = [&](int64_t i) { return bnd + ((slot0 + i % sp.slots) * PW + g) * a.bnd_rows; };
    // release epoch i / slots of slot i % slots, after the epoch before it
    auto release = [&](int64_t i) {
        uint32_t* r = sp.rel + slot0 + i % sp.slots;
        const uint32_t e = (uint32_t)(i / sp.slots);
        wait_u32(r, e, a.status);
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        if (threadIdx.x == 0) __hip_atomic_store(r, e + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    };
    for (;;) {
        uint32_t it = 0;
        if (threadIdx.x == 0) it = atomicAdd(a.queue + x, 1u);
        const int64_t i = (int64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)it);
        if (i >= 2 * per_pass) break;
        const int rev = i >= per_pass;
        const int64_t k = rev ? i - per_pass : i;
        const int64_t q = (int64_t)x + (int64_t)kXcds * (k / sp.strips);
        const int s = (int)(k % sp.strips);
        const int64_t ws = q * PW + g; // work slot of this group's pair
        const int64_t p = slot_pair(a, ws);
        uint64_t* fkey = sp.keys;
        uint64_t* rkey = sp.keys + a.order_n;

        Task t;
        FwdOut f{0, 0, 0};
        bool strict = false;
        if (!rev) {
            t = forward_task(a, p);
        } else {
            // the set's forward strips have all finished
            wait_u32(sp.done + q, (uint32_t)sp.strips, a.status);
            const uint64_t fk = p >= 0 ? __hip_atomic_load(fkey + ws, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) : 0;
            f = forward_result<G>(a, p, fk, s == 0);
            t = reverse_task(a, p, f, column_bound<G>(a, sm, p, f));
            // (from the ends alone: the same for every strip of the set)
            strict = __ballot(p >= 0 && f.score > 0 && reverse_swaps(a, p, f)) == 0;
            // a pair whose target an earlier strip reached drops out of the rest of its
            // strips, monotonically along them (k_split): strip s > 0 waits for strip
            // s - 1's decision and publishes its own
            uint32_t* gw = p >= 0 ? sp.gate + ws : nullptr;
            const uint32_t prev = wait_group_u32(s > 0 ? gw : nullptr, (uint32_t)s, a.status);
            bool keep = t.nr > 0 && t.nc > 0 && prev != kGateDropped;
            if (keep && s > 0 && __hip_atomic_load(rkey + ws, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0)
                keep = false;
            if (!keep) t.nr = 0;
            if (gw && l == 0)
                __hip_atomic_store(gw, keep ? (uint32_t)s + 1 : kGateDropped, __ATOMIC_RELAXED,
                                   __HIP_MEMORY_SCOPE_AGENT);
        }
        // strips of the set (wave maximum)
        int st = (t.nr > 0 && t.nc > 0) ? (t.nc + 2 * G * K - 1) / (2 * G * K) : 0;
#pragma unroll
        for (int o = G; o < kWave; o <<= 1) st = max(st, __shfl_xor(st, o));
        st = __builtin_amdgcn_readfirstlane(st);
        if (s < st) {
            wait_u32(sp.rel + slot0 + i % sp.slots, (uint32_t)(i / sp.slots), a.status); // slot free
            StripIO io;
            io.strip = s;
            io.bnd_in = s > 0 ? (const void*)slot_bnd(i - 1) : nullptr;
            io.bnd_out = (void*)slot_bnd(i);
            io.prog_in = s > 0 ? sp.prog + slot0 + (i - 1) % sp.slots : nullptr;
            io.prog_out = sp.prog + slot0 + i % sp.slots;
            io.epoch_in = s > 0 ? (uint64_t)((i - 1) / sp.slots) << 32 : 0;
            io.epoch_out = (uint64_t)(i / sp.slots) << 32;
            PassResult r;
            if (!rev) r = sweep<A, G, K, PF, false, true>(a, sm, t, 0, false, nullptr, io);
            else r = sweep<A, G, K, PF, true, true>(a, sm, t, f.score, strict, nullptr, io);
            if (p >= 0 && l == 0 && r.key != 0) atomicMax((unsigned long long*)((rev ? rkey : fkey) + ws), r.key);
        }
        if (s > 0) release(i - 1);          // done with the previous strip's rows
        if (s == sp.strips - 1) release(i); // no strip follows
        // count the item; the last reverse item of the set writes its results
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        uint32_t before = 0;
        if (threadIdx.x == 0) before = atomicAdd(sp.done + (rev ? nsets : 0) + q, 1u);
        before = (uint32_t)__builtin_amdgcn_readfirstlane((int)before);
        if (rev && before == (uint32_t)sp.strips - 1) {
            const uint64_t rk = p >= 0 ? __hip_atomic_load(rkey + ws, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) : 0;
            int32_t rb, qb;
            reverse_result(a, p, f, t, f.score, rk, &rb, &qb); // (the host never splits asymmetric tables)
            if (p >= 0 && l == 0 && f.score >= 0) {
                a.out[kOutScore * a.n + p] = f.score;
                a.out[kOutRefEnd * a.n + p] = f.ref_end;
                a.out[kOutQueryEnd * a.n + p] = f.query_end;
                a.out[kOutRefBegin * a.n + p] = rb;
                a.out[kOutQueryBegin * a.n + p] = qb;
            }
        }
    }
}

} // namespace gbsw
