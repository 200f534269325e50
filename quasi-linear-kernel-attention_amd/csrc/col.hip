// The forward sums column by column (segments with N + M <= COL_MAX elements).
//
//   abs      out[p,m,c] = sum_{d,n} |k[p,d,n] - q[p,d,m]| v[p,n,c]
//   Laplace  out[p,m,c] = sum_{d,n} e^{-|k[p,d,n] - q[p,d,m]|} v[p,n,c]
//
// One workgroup owns CH channels of one p: their columns of v (N words each) and their accumulators (M words each) stay
// in LDS while it runs over the features d. Per feature it walks the merged sorted sequence of keys and queries: each
// thread owns E consecutive elements, reads their words from LDS (a key's v, a query's accumulator; random access), the
// prefix states are combined over threads by a scan, and each query adds its feature's value to its accumulator. The D
// sum happens in LDS, so no per-feature contribution ever goes to memory, which is what a walk with one row per (p, d,
// query) has to write and a reduce to read back (6.6 of 10.4 GB per call at P = 12, D = 64, N = M = 16384, C = 64).
//
// The merged sequence of a segment does not depend on the channel: col_merge writes it once (6 bytes per element) and
// the C / CH workgroups of a p read it, neighbours on one XCD at about the same time, so from its L2.
//   val[s][E/4][T][4]   abs: the value less the thread's anchor, its value nearest the segment's median key; Laplace:
//                       e^-distance to the previous element
//   tag[s][E/4][T][4]   16-bit word index: query m at spread(m), key n at K0 + spread(n), padding at K0 + N (K0 = M,
//                       or M rounded up)
//   xe[s][T]            abs: each thread's anchor less the median key; Laplace: its Decays
//   eq[s][T]            (abs backward) bit e: element e of the thread has the value of the element before it
// With 4 elements per 16-byte (8-byte) load, a wave's loads are contiguous.
//
// What bounds col_sum: per element and channel one LDS read and, for a query, one masked write at random addresses
// (about 8 and 6 cycles a wave, bank conflicts of 64 random words), beside some 10 (abs) or 15 (Laplace) vector
// instructions. At N = M = 16384, one channel per workgroup, P = 12, D = C = 64, a kernel trace has 0.90 ms (abs; VALU
// 59%, LDS 61% of it by the counters) and 1.01 ms (Laplace; 76%, 55%). LDS float atomics in place of the read and the
// write ran at 100 cycles a wave (4.3 ms). Whole calls against the walk: abs 1.70 -> 1.35 ms, Laplace 1.69 -> 1.44 ms
// at that size, Laplace 0.81 -> 0.54 ms at N = M = 8192, add_riesz 0.97 -> 0.55 ms at 24 x 3111, add_bump 8.9 -> 5.4 ms
// at 48 x 8192, abs forward + backward 4.76 -> 3.61 ms at 12 x 16384.
#include <algorithm>
#include <cfloat>
#include <utility>

#include "per_device.h"
#include "qlka_common.h"
#include "qlka_internal.h"

namespace qlka {

#define LDS_AS __attribute__((address_space(3)))

typedef float f2_t __attribute__((ext_vector_type(2)));
typedef unsigned int u2_t __attribute__((ext_vector_type(2)));

enum ColKind : int { COL_ABS = 0, COL_LAPLACE = 1 };

// ---------------------------------------------------------------------------------------------------------------
// DPP helpers: the value of another lane, or `old` where the pattern has no source lane
// ---------------------------------------------------------------------------------------------------------------
template <int CTRL>
__device__ __forceinline__ float dpp(float old, float x) {
    return __int_as_float(__builtin_amdgcn_update_dpp(__float_as_int(old), __float_as_int(x), CTRL, 0xf, 0xf, false));
}
constexpr int WAVE_SHR1 = 0x138, WAVE_SHL1 = 0x130;

// Steps of the scans as one DPP instruction each (the compiler's form moves the other lane's value first): x += y of
// the lane the pattern names, x = a y + x and a *= that lane's a; lanes without a source keep x. A DPP read needs two
// wait states after the register's write (as a lane read does after the last step: settle), which the compiler does not
// know of around an asm statement.
#define QLKA_DPP_STEP(NAME, PATTERN)                                                                                  \
    struct NAME {                                                                                                     \
        __device__ static __forceinline__ void add(float& x) {                                                        \
            asm("s_nop 1\n\tv_add_f32_dpp %0, %0, %0 " PATTERN : "+v"(x));                                            \
        }                                                                                                             \
        __device__ static __forceinline__ void fma(float& x, float a) {                                               \
            asm("s_nop 1\n\tv_fmac_f32_dpp %0, %0, %1 " PATTERN : "+v"(x) : "v"(a));                                  \
        }                                                                                                             \
        __device__ static __forceinline__ void mul(float& x) {                                                        \
            asm("s_nop 1\n\tv_mul_f32_dpp %0, %0, %0 " PATTERN : "+v"(x));                                            \
        }                                                                                                             \
    }
QLKA_DPP_STEP(Up1, "row_shr:1 row_mask:0xf bank_mask:0xf");
QLKA_DPP_STEP(Up2, "row_shr:2 row_mask:0xf bank_mask:0xf");
QLKA_DPP_STEP(Up4, "row_shr:4 row_mask:0xf bank_mask:0xf");
QLKA_DPP_STEP(Up8, "row_shr:8 row_mask:0xf bank_mask:0xf");
QLKA_DPP_STEP(UpRow, "row_bcast:15 row_mask:0xa bank_mask:0xf");
QLKA_DPP_STEP(UpHalf, "row_bcast:31 row_mask:0xc bank_mask:0xf");
QLKA_DPP_STEP(Down1, "row_shl:1 row_mask:0xf bank_mask:0xf");
QLKA_DPP_STEP(Down2, "row_shl:2 row_mask:0xf bank_mask:0xf");
QLKA_DPP_STEP(Down4, "row_shl:4 row_mask:0xf bank_mask:0xf");
QLKA_DPP_STEP(Down8, "row_shl:8 row_mask:0xf bank_mask:0xf");
#undef QLKA_DPP_STEP

__device__ __forceinline__ void settle(float& x) { asm("s_nop 1" : "+v"(x)); }

// inclusive prefix sum over the wave's lanes
__device__ __forceinline__ float wave_scan_sum(float x) {
    Up1::add(x);
    Up2::add(x);
    Up4::add(x);
    Up8::add(x);
    UpRow::add(x);
    UpHalf::add(x);
    settle(x);
    return x;
}
// the same within rows of 16 lanes, over W <= 16 entries
template <int W>
__device__ __forceinline__ float row_scan_sum(float x) {
    if constexpr (W > 1) Up1::add(x);
    if constexpr (W > 2) Up2::add(x);
    if constexpr (W > 4) Up4::add(x);
    if constexpr (W > 8) Up8::add(x);
    settle(x);
    return x;
}
// one step of the inclusive scan of y <- a y' + b, y' from the lane the step names
template <int CH>
__device__ __forceinline__ void settle(float& a, float (&b)[CH]) {
    settle(a);
#pragma unroll
    for (int c = 0; c < CH; ++c) settle(b[c]);
}
template <class Step, int CH>
__device__ __forceinline__ void affine_step(float& a, float (&b)[CH]) {
#pragma unroll
    for (int c = 0; c < CH; ++c) Step::fma(b[c], a);
    Step::mul(a);
}
// lane_id() counted again, for a loop whose registers cannot hold it (spilled, its reload waits for every load in
// flight)
__device__ __forceinline__ int lane_now() {
    int r;
    asm volatile("v_mbcnt_lo_u32_b32 %0, -1, 0\n\tv_mbcnt_hi_u32_b32 %0, -1, %0" : "=v"(r));
    return r;
}

// The Laplace decays of a thread and around it in its wave, each formed from its own distance: a scan that multiplies
// the threads' decays up doubles their errors at every step, to thousands of times a rounding that repeats (a grid of
// keys).
struct Decays {
    float own;                       // over the thread
    float row, half;                 // from the start of its row of 16 lanes, and of lane 32, to the thread's end
    float before, after;             // from the wave's start to the thread, and from it to the wave's end
    float rest;                      // from the thread's start to its row's end
};
// inclusive scans of y <- a y' + b over the wave's threads
template <int CH>
__device__ __forceinline__ void wave_affine_up(const Decays& y, float (&b)[CH]) {       // lane order
    float a = y.own;
    affine_step<Up1>(a, b);
    affine_step<Up2>(a, b);
    affine_step<Up4>(a, b);
#pragma unroll
    for (int c = 0; c < CH; ++c) Up8::fma(b[c], a);
#pragma unroll
    for (int c = 0; c < CH; ++c) UpRow::fma(b[c], y.row);
#pragma unroll
    for (int c = 0; c < CH; ++c) {
        UpHalf::fma(b[c], y.half);
        settle(b[c]);
    }
}
template <int CH>
__device__ __forceinline__ void wave_affine_down(const Decays& y, float (&b)[CH]) {     // reverse lane order
    float a = y.own;
    affine_step<Down1>(a, b);
    affine_step<Down2>(a, b);
    affine_step<Down4>(a, b);
#pragma unroll
    for (int c = 0; c < CH; ++c) {
        Down8::fma(b[c], a);
        settle(b[c]);
    }
    // rows above, last first (no DPP pattern reads the next row): their totals are in their first lanes
    const int row = lane_now() >> 4;
    const float a1 = bcast(y.row, 31), a2 = bcast(y.row, 47);
#pragma unroll
    for (int c = 0; c < CH; ++c) {
        const float b3 = bcast(b[c], 48);
        const float b2 = fmaf(a2, b3, bcast(b[c], 32));
        const float b1 = fmaf(a1, b2, bcast(b[c], 16));
        const float bin = row == 0 ? b1 : row == 1 ? b2 : row == 2 ? b3 : 0.f;
        b[c] = fmaf(y.rest, bin, b[c]);
    }
}
// the same over W <= 16 entries of a row, the decays multiplied up
template <int W, int CH>
__device__ __forceinline__ void row_affine_up(float& a, float (&b)[CH]) {
    if constexpr (W > 1) affine_step<Up1>(a, b);
    if constexpr (W > 2) affine_step<Up2>(a, b);
    if constexpr (W > 4) affine_step<Up4>(a, b);
    if constexpr (W > 8) affine_step<Up8>(a, b);
    settle(a, b);
}
template <int W, int CH>
__device__ __forceinline__ void row_affine_down(float& a, float (&b)[CH]) {
    if constexpr (W > 1) affine_step<Down1>(a, b);
    if constexpr (W > 2) affine_step<Down2>(a, b);
    if constexpr (W > 4) affine_step<Down4>(a, b);
    if constexpr (W > 8) affine_step<Down8>(a, b);
    settle(a, b);
}

// words of CH channels at an LDS byte address
template <int CH>
__device__ __forceinline__ void lds_read(float (&x)[CH], uint32_t byte) {
    if constexpr (CH == 1) {
        x[0] = *(LDS_AS const float*)byte;
    } else {
        const f2_t v = *(LDS_AS const f2_t*)byte;
        x[0] = v.x;
        x[1] = v.y;
    }
}
// Store in the lanes of `mask` only, without a branch around it (the compiler's form of a masked store jumps over it
// when no lane stores, which costs more than the store: half of a wave's elements are queries). Every lane of the wave
// is active here. The compiler does not count this store: a wait for lgkmcnt(0) must come before the next barrier.
template <int CH>
__device__ __forceinline__ void lds_write_masked(const float (&x)[CH], uint32_t byte, uint64_t mask) {
    if constexpr (CH == 1) {
        asm volatile("s_mov_b64 exec, %2\n\tds_write_b32 %0, %1\n\ts_mov_b64 exec, -1" ::"v"(byte), "v"(x[0]), "s"(mask)
                     : "memory");
    } else {
        f2_t v;
        v.x = x[0];
        v.y = x[1];
        asm volatile("s_mov_b64 exec, %2\n\tds_write_b64 %0, %1\n\ts_mov_b64 exec, -1" ::"v"(byte), "v"(v), "s"(mask)
                     : "memory");
    }
}
// Byte address of the low / high 16-bit word index of a tag pair, words of B bytes (one instruction each; the compiler
// takes two for the low half).
template <int B>
__device__ __forceinline__ uint32_t tag_addr(uint32_t pair, bool high) {
    uint32_t r;
    const uint32_t sh = B == 4 ? 2 : 3;
    if (high)
        asm("v_lshlrev_b32_sdwa %0, %1, %2 dst_sel:DWORD dst_unused:UNUSED_PAD src0_sel:DWORD src1_sel:WORD_1"
            : "=v"(r) : "v"(sh), "v"(pair));
    else
        asm("v_lshlrev_b32_sdwa %0, %1, %2 dst_sel:DWORD dst_unused:UNUSED_PAD src0_sel:DWORD src1_sel:WORD_0"
            : "=v"(r) : "v"(sh), "v"(pair));
    return r;
}
// b where the lane's bit of mask is set, else a; the empty asm keeps it one select (the compiler otherwise branches
// around the arithmetic that follows)
__device__ __forceinline__ float pick(float a, float b, uint64_t mask) {
    float r = __builtin_amdgcn_inverse_ballot_w64(mask) ? b : a;
    asm("" : "+v"(r));
    return r;
}
__device__ __forceinline__ float unless(float a, uint64_t mask) { return pick(a, 0.f, mask); }
// All ones where bit e of x is set, else 0; and b where m is all ones, a where it is 0. As asm, or the compiler turns
// the bits of a loop into one lane mask each, more than there are scalar registers.
template <int e>
__device__ __forceinline__ uint32_t bit_mask(uint32_t x) {
    uint32_t r;
    asm("v_bfe_i32 %0, %1, %2, 1" : "=v"(r) : "v"(x), "n"(e));
    return r;
}
__device__ __forceinline__ float bit_pick(float a, float b, uint32_t m) {
    float r;
    asm("v_bfi_b32 %0, %1, %2, %3" : "=v"(r) : "v"(m), "v"(b), "v"(a));
    return r;
}
// f(integral_constant<int, 0>) ... f(integral_constant<int, E - 1>)
template <class F, int... I>
__device__ __forceinline__ void each_index(F f, std::integer_sequence<int, I...>) {
    (f(std::integral_constant<int, I>{}), ...);
}
template <int E, class F>
__device__ __forceinline__ void each(F f) { each_index(f, std::make_integer_sequence<int, E>{}); }

// ---------------------------------------------------------------------------------------------------------------
// col_merge: one workgroup per segment
// ---------------------------------------------------------------------------------------------------------------
// e^-x, x >= 0, for a chain of products. Below 1/2 as 1 - h with h = 1 - e^-x by its Taylor series (9 terms: to 2^-26
// of h), so that it rounds to nearest: near 1 the library's expf is off to one side by up to an ulp, which thousands of
// factors add up. And `rest`, what rounding the factors before has left to be taken off, is taken off here and left
// anew: where the distances repeat (a grid) or are all below half an ulp, factors rounded one by one err to one side as
// well. With this and Decays, Laplace at N = M = 8192, relative 2-norm against 64 bits, a grid over +-3 and uniform
// keys in +-2e-5: 5.1e-6 and 3.5e-6 -> 3.9e-7 and 1.5e-7 (walks: 5.7e-7 and 2.1e-7); N(0, 1) 1.4e-7 -> 7.6e-8 (2.9e-7).
__device__ __forceinline__ float decay(float x, float& rest) {
    if (x >= 0.5f) return expf(-x);
    float h = fmaf(x, -1.f / 362880.f, 1.f / 40320.f);
    h = fmaf(x, -h, 1.f / 5040.f);
    h = fmaf(x, -h, 1.f / 720.f);
    h = fmaf(x, -h, 1.f / 120.f);
    h = fmaf(x, -h, 1.f / 24.f);
    h = fmaf(x, -h, 1.f / 6.f);
    h = fmaf(x, -h, 0.5f);
    h = fmaf(x, -h, 1.f);
    h = fmaf(x, h, rest);
    const float r = 1.f - h;
    rest = h - (1.f - r);                                    // exact
    return r;
}

struct ColMergeArgs {
    const float* qs; const uint32_t* qp; const float* ks; const uint32_t* kp;   // sorted queries and keys
    const uint8_t* keep;             // (P, N) key mask or null: masked keys become padding
    float* val; uint16_t* tag; float* xe; float* xe2; uint32_t* eq;  // eq: null unless wanted; xe2: Laplace only
    float* u;                        // (S, M) v == 1 terms in the order of the words, or null
    float* bad;                      // (P, M), bwd: (P, N), in the order of the words: NaN at the rows whose own value
                                     // makes them NaN, 0 else; or null
    int D, N, M, K0;
    int sets;                        // 1, or 3: streams of q, q + 1 and q - 1 per segment (add_bump), their v == 1
                                     // terms weighted
};

// add_bump: max(0, 1 - |x|) = (|x + 1| + |x - 1|) / 2 - |x|, one feature's three abs sums after one another. The same
// sorted order serves all three: adding a constant in fp32 is monotone.
__device__ __forceinline__ float set_shift(int set) { return set == 0 ? 0.f : set == 1 ? 1.f : -1.f; }
__device__ __forceinline__ float set_weight(int sets, int set) { return sets == 1 ? 1.f : set == 0 ? -1.f : 0.5f; }

// A finite stand-in for an element that carries no weight: x, or the largest float on x's side. Its value enters the
// shared sums as value x 0, which an infinity or a NaN would turn into NaN for every row of the p.
__device__ __forceinline__ float bounded(float x) { return fabsf(x) <= FLT_MAX ? x : copysignf(FLT_MAX, x); }
// a NaN as the infinity on its side
__device__ __forceinline__ float no_nan(float x) { return x == x ? x : copysignf(__int_as_float(0x7f800000), x); }
// Values with which all below is finite without looking at each (abs: their differences are; Laplace: not a NaN); a
// segment with another one is `rare`
template <int KIND>
__device__ __forceinline__ bool ordinary(float x) { return KIND == COL_ABS ? fabsf(x) <= 1e37f : x == x; }
// true in the whole workgroup if x is in any of its threads; flags: W words of LDS, read before they may be written
// again
template <int W>
__device__ __forceinline__ bool any_of(bool x, uint32_t* flags) {
    const uint64_t b = __ballot(x);
    if (lane_id() == 0) flags[wave_in_block()] = b != 0;
    __syncthreads();
    return __ballot(flags[lane_id() % W] != 0) != 0;
}

// The word of row i among the L of a side (and the row of word i): within each whole block of 64, shuffled by the
// block's number. Where values tie, the sorts leave rows in order, and threads of E consecutive elements each would
// read words E apart, 16 and more of them from one bank (12 x 64 x 16384, half the keys 0 as by a mask multiplied in:
// abs 1.93 -> 1.35 ms, Laplace 2.11 -> 1.44, training 5.88 -> 3.81; walks 1.72, 1.71, 4.75).
__device__ __forceinline__ int spread(int i, int L) { return i < (L & ~63) ? i ^ ((i >> 6) & 63) : i; }

// 16-bit word indices, two in a register
template <int E>
struct Halves {
    uint32_t w[E / 2];
    __device__ __forceinline__ uint32_t get(int i) const { return (i & 1) ? w[i / 2] >> 16 : w[i / 2] & 0xffffu; }
    __device__ __forceinline__ void set(int i, uint32_t x) {         // in order: the low half first
        if (i & 1) w[i / 2] |= x << 16;
        else w[i / 2] = x;
    }
};

__device__ __forceinline__ bool is_key(int word, const ColMergeArgs& A) {
    return (uint32_t)(word - A.K0) < (uint32_t)A.N;
}

// The median of a segment's keys that are not padding, from its merged order (as emit_stream's), 0 without any;
// scratch: 1 + W words of LDS.
template <int T, int E>
__device__ __forceinline__ float median_key(const ColMergeArgs& A, const float (&val)[E], const Halves<E>& src,
                                            uint32_t* scratch)
{
    constexpr int W = T / WAVE;
    const int lane = lane_id(), wv = wave_in_block();
    int keys = 0;
#pragma unroll
    for (int e = 0; e < E; ++e) keys += is_key((int)src.get(e), A);
    int inc = keys;
#pragma unroll
    for (int off = 1; off < WAVE; off <<= 1) {
        const int y = __shfl_up(inc, off, WAVE);
        if (lane >= off) inc += y;
    }
    if (lane == WAVE - 1) scratch[1 + wv] = (uint32_t)inc;
    if (threadIdx.x == 0) scratch[0] = 0;
    __syncthreads();
    int at = keys - inc, total = 0;                          // the median's number among this thread's keys
    for (int w = 0; w < W; ++w) {
        if (w < wv) at -= (int)scratch[1 + w];
        total += (int)scratch[1 + w];
    }
    at += total / 2;
    if (at >= 0 && at < keys) {
#pragma unroll
        for (int e = 0; e < E; ++e)
            if (is_key((int)src.get(e), A) && at-- == 0) scratch[0] = __float_as_uint(val[e]);
    }
    __syncthreads();
    return __uint_as_float(scratch[0]);
}

// The stream and the v == 1 terms of one segment, from its merged order: thread t's elements as word indices src
// (padding, masked keys among it: K0 + N) and as values val (padding: the value before); x0 the median key, xs the
// value before the thread's first element. sm: N + M words and 3 words a wave, free to use.
//
// A query (bwd: a key) only receives sums, so whatever it holds stays in its own row. In a rare segment abs sums take
// its value bounded, Laplace sums a NaN as the infinity on its side, and the row is marked in A.bad, which the finish
// makes NaN: for abs where the value is infinite or NaN (as the walks' rows are), for Laplace where it is NaN (an
// infinite one is far from every finite key). poison: a NaN among the weights' values that val no longer shows; every
// row is NaN.
template <int KIND, int T, int E>
__device__ __forceinline__ void emit_stream(const ColMergeArgs& A, float* sm, int s, float x0, float xs,
                                            float (&val)[E], const Halves<E>& src, bool rare, bool poison)
{
    constexpr int W = T / WAVE;
    const int N = A.N, M = A.M, n = N + M, tid = threadIdx.x, seg = s / A.sets, p = seg / A.D;
    const int acc0 = A.eq ? A.K0 : 0, accs = A.eq ? N : M;       // the words that receive sums
    auto receives = [&](int e) { return src.get(e) - (uint32_t)acc0 < (uint32_t)accs; };
    auto weightless = [&](int e) { return receives(e) || (int)src.get(e) == A.K0 + N; };
    if (rare) {
        if constexpr (KIND == COL_LAPLACE) xs = no_nan(xs);
#pragma unroll
        for (int e = 0; e < E; ++e) {
            const bool row = receives(e) && (KIND == COL_ABS ? !(fabsf(val[e]) <= FLT_MAX) : val[e] != val[e]);
            if (row && A.bad) A.bad[(size_t)p * accs + ((int)src.get(e) - acc0)] = __int_as_float(0x7fc00000);
            if (weightless(e)) val[e] = KIND == COL_ABS ? bounded(val[e]) : no_nan(val[e]);
        }
    }
    float dist[E];
    // A thread's values are taken relative to its anchor, its value nearest the median, so that every value an
    // element's sums are formed from is bounded by distances to keys: on either side of the median the end towards it,
    // and the median itself in a thread on both sides
    float anchor = 0.f;
    Decays dec;
    if constexpr (KIND == COL_ABS) {
        const float xa = x0 <= val[0] ? val[0] : x0 >= val[E - 1] ? val[E - 1] : x0;
        anchor = xa - x0;
#pragma unroll
        for (int e = 0; e < E; ++e) dist[e] = val[e] - xa;
        if (rare) {
            anchor = poison ? __int_as_float(0x7fc00000) : bounded(anchor);
#pragma unroll
            for (int e = 0; e < E; ++e)
                if (weightless(e)) dist[e] = bounded(dist[e]);
        }
    } else {                                             // e^-distance once per element for all channels
        float prev = xs, rest = 0.f;
#pragma unroll
        for (int e = 0; e < E; ++e) {
            dist[e] = decay(val[e] != prev ? val[e] - prev : 0.f, rest);         // equal infinities: 0 apart
            prev = val[e];
        }
        const int lane = lane_id();
        auto over = [](float from, float to) {           // one distance's decay
            float none = 0.f;
            return decay(to != from ? to - from : 0.f, none);
        };
        dec.own = over(xs, prev);
        dec.row = over(__shfl(xs, lane & 48, WAVE), prev);
        dec.half = lane < 32 ? 1.f : over(__shfl(xs, 32, WAVE), prev);
        dec.before = over(__shfl(xs, 0, WAVE), xs);
        dec.after = over(prev, __shfl(prev, WAVE - 1, WAVE));
        dec.rest = over(xs, __shfl(prev, lane | 15, WAVE));
        if (rare && poison)
            dec.own = dec.row = dec.half = dec.before = dec.after = dec.rest = __int_as_float(0x7fc00000);
    }
    float* vo = A.val + (size_t)s * T * E;
    uint16_t* to = A.tag + (size_t)s * T * E;
#pragma unroll
    for (int g = 0; g < E / 4; ++g) {
        f4_t x;
        u2_t y;
#pragma unroll
        for (int e = 0; e < 4; ++e) x[e] = dist[4 * g + e];
        y.x = src.w[2 * g];
        y.y = src.w[2 * g + 1];
        *(f4_t*)(vo + ((size_t)g * T + tid) * 4) = x;
        *(u2_t*)(to + ((size_t)g * T + tid) * 4) = y;
    }
    if constexpr (KIND == COL_ABS) {
        A.xe[(size_t)s * T + tid] = anchor;
    } else {
        const f4_t x = {dec.own, dec.row, dec.half, dec.before};
        const f2_t y = {dec.after, dec.rest};
        ((f4_t*)A.xe)[(size_t)s * T + tid] = x;
        ((f2_t*)A.xe2)[(size_t)s * T + tid] = y;
    }
    if (A.u == nullptr) return;

    // v == 1: the same walk as col_sum's with every key's weight 1
    float wt[E];
#pragma unroll
    for (int e = 0; e < E; ++e) wt[e] = is_key((int)src.get(e), A) ? 1.f : 0.f;
    const int lane = lane_id(), wv = wave_in_block();
    float* agg = sm + n;
    float out[E];
    if constexpr (KIND == COL_ABS) {
        float sw = 0.f, sk_ = 0.f;
#pragma unroll
        for (int e = 0; e < E; ++e) {
            out[e] = fmaf(dist[e], sw, -sk_);
            sw += wt[e];
            sk_ = fmaf(dist[e], wt[e], sk_);
        }
        float we = sw, ke = fmaf(anchor, sw, sk_);
        const float wi = wave_scan_sum(we), ki = wave_scan_sum(ke);
        we = wi - we;
        ke = ki - ke;
        if (lane == WAVE - 1) { agg[2 * wv] = wi; agg[2 * wv + 1] = ki; }
        __syncthreads();
        float wp = 0.f, kp = 0.f, wtot = 0.f, ktot = 0.f;
        for (int x = 0; x < W; ++x) {
            const float a = agg[2 * x], b = agg[2 * x + 1];
            if (x < wv) { wp += a; kp += b; }
            wtot += a;
            ktot += b;
        }
        const float S = we + fmaf(-0.5f, wtot, wp);
        const float F = fmaf(anchor, S, -(ke + fmaf(-0.5f, ktot, kp)));
#pragma unroll
        for (int e = 0; e < E; ++e)
            out[e] = 2.f * set_weight(A.sets, s - seg * A.sets) * (out[e] + fmaf(dist[e], S, F));
    } else {
        float l = 0.f, r = 0.f, pr = 1.f;
#pragma unroll
        for (int e = 0; e < E; ++e) {
            l = fmaf(dist[e], l, wt[e]);
            pr *= dist[e];
            r = fmaf(pr, wt[e], r);
        }
        float up[1] = {l}, dn[1] = {r};
        wave_affine_up(dec, up);
        wave_affine_down(dec, dn);
        if (lane == WAVE - 1) { agg[3 * wv] = up[0]; agg[3 * wv + 2] = dec.before * dec.own; }
        if (lane == 0) agg[3 * wv + 1] = dn[0];
        float L = dpp<WAVE_SHR1>(0.f, up[0]), R = dpp<WAVE_SHL1>(0.f, dn[0]);
        __syncthreads();
        float lin = 0.f, rin = 0.f;
        for (int x = 0; x < wv; ++x) lin = fmaf(agg[3 * x + 2], lin, agg[3 * x]);
        for (int x = W - 1; x > wv; --x) rin = fmaf(agg[3 * x + 2], rin, agg[3 * x + 1]);
        L = fmaf(dec.before, lin, L);
        R = fmaf(dec.after, rin, R);
#pragma unroll
        for (int e = E - 1; e >= 0; --e) {               // R at the element (later keys), then at the one before
            R += wt[e];
            out[e] = R;                                  // a query's weight is 0
            R *= dist[e];
        }
#pragma unroll
        for (int e = 0; e < E; ++e) { L = fmaf(dist[e], L, wt[e]); out[e] += L; }
    }
    // in the order of the words through LDS (every thread has read its word indices before the scan's barrier)
#pragma unroll
    for (int e = 0; e < E; ++e)
        if ((int)src.get(e) < M) sm[src.get(e)] = out[e];
    __syncthreads();
    float* uo = A.u + (size_t)s * M;
    for (int x = tid; x < M; x += T) uo[x] = sm[x];
}

// f(i, x[i]) for the n elements of x, shared out over T threads; eight loads of each are in flight at a time
template <int T, class X, class F>
__device__ __forceinline__ void each_of(const X* __restrict__ x, int n, F f) {
    for (int i = threadIdx.x; i < n; i += 8 * T) {
        X r[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) r[j] = x[min(i + j * T, n - 1)];
#pragma unroll
        for (int j = 0; j < 8; ++j)
            if (i + j * T < n) f(i + j * T, r[j]);
    }
}

// dynamic LDS: N + M words (values, then word indices, then the v == 1 terms), then the scans' 3 words a wave
template <int KIND, int T, int E>
__global__ __launch_bounds__(T)
void col_merge(const ColMergeArgs A)
{
    extern __shared__ float sm[];
    const int s = blockIdx.x, seg = s / A.sets, tid = threadIdx.x;     // stream, segment
    const int N = A.N, M = A.M, n = N + M;
    const float* qs = A.qs + (size_t)seg * M;
    const float* ks = A.ks + (size_t)seg * N;
    const float shift = set_shift(s - seg * A.sets);
    const uint8_t* keep = A.keep ? A.keep + (size_t)(seg / A.D) * N : nullptr;       // without A.eq only
    bool odd = false;
    each_of<T>(qs, M, [&](int i, float x) {
        x += shift;
        odd |= !ordinary<KIND>(x);
        sm[i] = x;
    });
    each_of<T>(ks, N, [&](int i, float x) {
        odd |= !ordinary<KIND>(x);
        sm[M + i] = x;
    });
    const bool rare = any_of<T / WAVE>(odd, (uint32_t*)sm + n);
    bool poison = false;
    if (rare) {          // the merge compares floats: NaNs become infinities, on the side that the sort put them
        bool nan = false;
        for (int i = tid; i < n; i += T) {
            const float x = sm[i];
            if (x == x) continue;
            sm[i] = no_nan(x);
            const bool weight = (i >= M) == (A.eq == nullptr);
            const int row = i < M ? (int)A.qp[(size_t)seg * M + i] : (int)A.kp[(size_t)seg * N + i - M];
            const int rows = i < M ? M : N;
            if (weight) nan |= !keep || keep[row] != 0;
            else if (A.bad) A.bad[(size_t)(seg / A.D) * rows + spread(row, rows)] = x;
        }
        __syncthreads();
        poison = any_of<T / WAVE>(nan, (uint32_t*)sm + n);
    }
    const float* sq = sm;
    const float* sk = sm + M;
    float x0 = sk[N / 2];
    // merge path: queries before `diag` (queries come first among equal values)
    const int diag = min(tid * E, n);
    int lo = max(0, diag - N), hi = min(diag, M);
    while (lo < hi) {
        const int mid = (lo + hi) >> 1;
        if (sq[mid] <= sk[diag - 1 - mid]) lo = mid + 1;
        else hi = mid;
    }
    int i = lo, j = diag - lo;
    float prev = 0.f;
    if (diag == 0) prev = fminf(sq[0], sk[0]);
    else if (i == 0) prev = sk[j - 1];
    else if (j == 0) prev = sq[i - 1];
    else prev = fmaxf(sq[i - 1], sk[j - 1]);
    const float xs = prev;
    float qa = sq[min(i, M - 1)], kb = sk[min(j, N - 1)];
    uint32_t eq = 0;
    float val[E];
    Halves<E> src;                      // word of the element in sq / sk
#pragma unroll
    for (int e = 0; e < E; ++e) {
        const bool live = diag + e < n;
        const bool tq = j >= N || (i < M && qa <= kb);
        const float r = tq ? qa : kb;
        src.set(e, (uint32_t)(live ? (tq ? i : M + j) : n));
        if (live && diag + e > 0 && r == prev) eq |= 1u << e;
        val[e] = live ? r : prev;
        if (live) {
            prev = r;
            if (tq) { ++i; qa = sq[min(i, M - 1)]; }
            else { ++j; kb = sk[min(j, N - 1)]; }
        }
    }
    __syncthreads();
    {   // word indices over the values
        uint32_t* w = (uint32_t*)sm;
        const uint32_t* qp = A.qp + (size_t)seg * M;
        const uint32_t* kp = A.kp + (size_t)seg * N;
        each_of<T>(qp, M, [&](int i, uint32_t x) { w[i] = (uint32_t)spread((int)x, M); });
        auto key = [&](int i, int word) { w[M + i] = (uint32_t)(A.K0 + word); };
        if (!keep) each_of<T>(kp, N, [&](int i, uint32_t x) { key(i, spread((int)x, N)); });
        else each_of<T>(kp, N, [&](int i, uint32_t x) { key(i, keep[x] ? spread((int)x, N) : N); });
        __syncthreads();
#pragma unroll
        for (int e = 0; e < E; e += 2) {
            const uint32_t x = src.get(e), y = src.get(e + 1), pad = (uint32_t)(A.K0 + N);
            src.w[e / 2] = ((int)x < n ? w[x] : pad) | ((int)y < n ? w[y] : pad) << 16;
        }
    }
    if (A.eq) A.eq[(size_t)s * T + tid] = eq;
    if (KIND == COL_ABS && keep) {
        x0 = median_key<T, E>(A, val, src, (uint32_t*)sm + n);
        __syncthreads();                                     // read; the emission writes there
    }
    emit_stream<KIND, T, E>(A, sm, s, x0, xs, val, src, rare, poison);
}

// ---------------------------------------------------------------------------------------------------------------
// col_sort: one workgroup per segment, from the unsorted queries and keys (A.qs, A.ks) to the stream
//
// A stable radix sort of queries (first) and keys together, 4 passes of 8 bits. A wave owns 64 E consecutive positions
// and takes them 64 at a time: the lanes with an equal digit find each other by 8 ballots, so that a position's rank in
// its wave is a running count per digit (a wave's own 256 counters in LDS) plus the equal lanes below it; one scan over
// (digit, wave) makes the counts first positions, and values and word indices go to their places through LDS. Nothing
// is read from or written to memory between the inputs and the stream. Masked keys sort last, as padding. What bounds
// it: about 60 vector instructions per element and pass (the ballots), then some 38 cycles of LDS, one after the other:
// 155 us for 768 segments of 16384 elements (the two sorts and the merge: 178).
// ---------------------------------------------------------------------------------------------------------------
__host__ __device__ constexpr int sort_words(int T, int E) { return T * E + T * E / 32 + 1 + 256 * (T / WAVE) + 32; }

// lanes of the wave whose 8-bit digit equals this lane's
__device__ __forceinline__ uint64_t equal_lanes(uint32_t digit) {
    uint32_t lo = 0u, hi = 0u;                               // lanes that differ in some bit
#pragma unroll
    for (int b = 0; b < 8; ++b) {
        uint32_t t = (uint32_t)__builtin_amdgcn_sbfe((int)digit, b, 1);
        asm("" : "+v"(t));                                   // one comparison below, not the bit taken again
        const uint64_t v = __ballot(t != 0);
        lo = __builtin_amdgcn_bitop3_b32(lo, (uint32_t)v, t, 0xf6);              // lo | (v ^ t)
        hi = __builtin_amdgcn_bitop3_b32(hi, (uint32_t)(v >> 32), t, 0xf6);
    }
    return ~((uint64_t)lo | ((uint64_t)hi << 32));
}

template <int KIND, int T, int E>
__global__ __launch_bounds__(T, 4)
void col_sort(const ColMergeArgs A)
{
    constexpr int W = T / WAVE, L = T * E, LP = L + L / 32 + 1;
    extern __shared__ float sm[];
    uint32_t* buf = (uint32_t*)sm;
    uint32_t* all = (uint32_t*)sm + LP;                      // [W][256] counters
    uint32_t* misc = all + 256 * W;                          // [0] live elements, [4 ...] scans, [7 ...] the median
    const int s = blockIdx.x, p = s / A.D, tid = threadIdx.x, lane = lane_id(), wv = wave_in_block();
    const int N = A.N, M = A.M, n = N + M;
    uint32_t* cnt = all + 256 * wv;
    const int first = wv * (WAVE * E) + lane;                // position of element j: first + 64 j
    auto padded = [](int i) { return i + (i >> 5); };
    uint32_t key[E], before_key = 0, last_key = 0;
    Halves<E> idx;
    int live = 0;
    bool odd = false;
    {
        const float* q = A.qs + (size_t)s * M;
        const float* k = A.ks + (size_t)s * N;
        const uint8_t* keep = A.keep ? A.keep + (size_t)p * N : nullptr;
#pragma unroll
        for (int j = 0; j < E; ++j) {
            const int i = first + WAVE * j;
            const float x = i < M ? q[i] : k[min(i - M, N - 1)];
            const bool on = i < n && (i < M || !keep || keep[i - M] != 0);
            odd |= on && !ordinary<KIND>(x);
            key[j] = on ? min(float_to_ordered(x), 0xfffffffeu) : 0xffffffffu;
            idx.set(j, on ? (uint32_t)(i < M ? spread(i, M) : M + spread(i - M, N)) : (uint32_t)n);
            live += (int)__popcll(__ballot(on));
        }
    }
    if (tid == 0) misc[0] = 0;
    const bool rare = any_of<W>(odd, misc + 8);
    if (lane == 0) atomicAdd(&misc[0], (uint32_t)live);      // an integer: the order does not matter
    for (int shift = 0; shift < 32; shift += 8) {
#pragma unroll
        for (int i = 0; i < 256 / WAVE; ++i) cnt[lane + WAVE * i] = 0;
        Halves<E> pos;
#pragma unroll
        for (int j = 0; j < E; ++j) {
            const uint32_t digit = (key[j] >> shift) & 255u;
            const uint64_t same = equal_lanes(digit);
            const uint32_t before = cnt[digit], below = (uint32_t)lanes_below(same), total = (uint32_t)__popcll(same);
            pos.set(j, before + below);
            if (below + 1 == total) cnt[digit] = before + total;
            if (j & 1) __builtin_amdgcn_sched_barrier(0);    // two positions' masks at a time, or all E are live
        }
        __syncthreads();
        {   // counts to first positions: digits in order, the waves of a digit in order
            constexpr int TD = T < 256 ? T : 256, DPT = 256 / TD;     // threads at work, digits each
            uint32_t tot[DPT], sum = 0;
            if (tid < TD) {
#pragma unroll
                for (int x = 0; x < DPT; ++x) {
                    uint32_t c = 0;
                    for (int w = 0; w < W; ++w) {
                        uint32_t* a = all + 256 * w + tid * DPT + x;
                        const uint32_t y = *a;
                        *a = c;
                        c += y;
                    }
                    tot[x] = c;
                    sum += c;
                }
            }
            uint32_t inc = sum;
#pragma unroll
            for (int off = 1; off < WAVE; off <<= 1) {
                const uint32_t y = __shfl_up(inc, off, WAVE);
                if (lane >= off) inc += y;
            }
            if (tid < TD && lane == WAVE - 1) misc[4 + wv] = inc;
            __syncthreads();
            if (tid < TD) {
                uint32_t base = inc - sum;
                for (int w = 0; w < wv; ++w) base += misc[4 + w];
#pragma unroll
                for (int x = 0; x < DPT; ++x) {
                    for (int w = 0; w < W; ++w) all[256 * w + tid * DPT + x] += base;
                    base += tot[x];
                }
            }
            __syncthreads();
        }
        // the last pass pads every 32 words: threads then read E words in a row
        const bool last = shift == 24;
#pragma unroll
        for (int j = 0; j < E; ++j) {
            const uint32_t x = pos.get(j) + cnt[(key[j] >> shift) & 255u], y = last ? x + (x >> 5) : x;
            if (j & 1) pos.w[j / 2] = (pos.w[j / 2] & 0xffffu) | (y << 16);
            else pos.w[j / 2] = (pos.w[j / 2] & 0xffff0000u) | y;
        }
#pragma unroll
        for (int j = 0; j < E; ++j) buf[pos.get(j)] = key[j];
        __syncthreads();
        if (last) {
#pragma unroll
            for (int j = 0; j < E; ++j) key[j] = buf[padded(tid * E + j)];
            before_key = buf[padded(max(tid * E, 1) - 1)];
            last_key = buf[padded((int)misc[0] - 1)];
        } else {
#pragma unroll
            for (int j = 0; j < E; ++j) key[j] = buf[first + WAVE * j];
        }
        __syncthreads();
#pragma unroll
        for (int j = 0; j < E; ++j) buf[pos.get(j)] = idx.get(j);
        __syncthreads();
#pragma unroll
        for (int j = 0; j < E; ++j) idx.set(j, buf[last ? padded(tid * E + j) : first + WAVE * j]);
    }
    const int nl = (int)misc[0];                             // queries and kept keys
    const float lastv = ordered_to_float(last_key);
    float prev = tid == 0 ? ordered_to_float(key[0]) : tid * E - 1 < nl ? ordered_to_float(before_key) : lastv;
    const float xs = prev;
    float val[E];
#pragma unroll
    for (int e = 0; e < E; ++e) {
        if (tid * E + e < nl) prev = ordered_to_float(key[e]);
        val[e] = prev;
    }
    const float x0 = KIND == COL_ABS ? median_key<T, E>(A, val, idx, misc + 7) : 0.f;
    __syncthreads();                                         // buf is read; the emission uses it
    emit_stream<KIND, T, E>(A, sm, s, x0, xs, val, idx, rare, false);
}

// ---------------------------------------------------------------------------------------------------------------
// col_sum: one workgroup per (p, feature share, CH channels)
// ---------------------------------------------------------------------------------------------------------------
struct ColSumArgs {
    const float* val; const uint16_t* tag; const float* xe; const float* xe2;
    const float* w;                  // [P][CW][Nw][CH] weight columns (col_weights): of v, or of g_w with SWAP
    float* out;                      // [P][DS][C][Ma]
    int P, D, N, M, C, DS, K0, CW;
    int sets;                        // D counts streams: features x sets, a feature's sets next to each other
};

// SWAP: the queries carry the weights and the keys the accumulators (the grad_v of the abs sums)
template <int KIND, int T, int E, int CH, bool SWAP, int WPE>
__global__ __launch_bounds__(T, WPE)
void col_sum(const ColSumArgs A)
{
    constexpr int W = T / WAVE;
    extern __shared__ float sm[];
    const int tid = threadIdx.x, wv = wave_in_block();
    const int D = A.D, N = A.N, M = A.M, C = A.C, DS = A.DS;
    const int Nw = SWAP ? M : N, Ma = SWAP ? N : M, w0 = SWAP ? 0 : A.K0, a0 = SWAP ? A.K0 : 0;
    const int CG = (C + CH - 1) / CH;
    const int b = xcd_slice_block(blockIdx.x, gridDim.x);
    const int p = b / (DS * CG), ds = (b / CG) % DS, c = (b % CG) * CH;
    const int d0 = (int)((long)D * ds / DS), d1 = (int)((long)D * (ds + 1) / DS);
    // LDS words: [K0 + N + 1][CH] (the last: padding's), then the aggregates of two features
    {
        const float* wp = A.w + ((size_t)p * A.CW + c / CH) * Nw * CH;
#pragma unroll 8
        for (int i = tid; i < Nw * CH; i += T) sm[w0 * CH + i] = wp[i];
    }
    for (int i = tid; i < Ma * CH; i += T) sm[a0 * CH + i] = 0.f;
    if (tid < CH) sm[(A.K0 + N) * CH + tid] = 0.f;
    const uint32_t aggb = ((uint32_t)(A.K0 + N + 1) * CH * 4 + 15) & ~15u;
    constexpr uint32_t AGGS = (KIND == COL_ABS ? 2 : 3) * CH * W * 4;    // bytes of one feature's aggregates
    __syncthreads();
    const size_t s0 = (size_t)p * D;
    const rsrc_t rv = make_rsrc(A.val + s0 * T * E, (uint32_t)(D * T * E * 4));
    const rsrc_t rt = make_rsrc(A.tag + s0 * T * E, (uint32_t)(D * T * E * 2));
    float dv[E];
    uint32_t tg[E / 2];
    auto load = [&](int d, int g) {                      // elements 4g .. 4g + 3
        const f4_t x = buf_load4(rv, tid * 16, d * (T * E * 4) + g * (T * 16));
        const u2_t y = __builtin_bit_cast(u2_t, __builtin_amdgcn_raw_buffer_load_b64(rt, tid * 8,
                                                                 d * (T * E * 2) + g * (T * 8), 0));
#pragma unroll
        for (int e = 0; e < 4; ++e) dv[4 * g + e] = x[e];
        tg[2 * g] = y.x;
        tg[2 * g + 1] = y.y;
    };
#pragma unroll
    for (int g = 0; g < E / 4; ++g) load(d0, g);
    const float* xp = A.xe + (s0 + d0) * T + tid;        // abs
    float xs = 0.f;
    if constexpr (KIND == COL_ABS) xs = *xp;
    const uint32_t split = (uint32_t)A.K0 * CH * 4;      // queries' words lie below, keys' above
    auto addr = [&](int e) { return tag_addr<CH * 4>(tg[e / 2], e & 1); };
    for (int d = d0; d < d1; ++d) {
        f4_t ya = {0.f, 0.f, 0.f, 0.f};                  // Laplace: its Decays, read after the thread's own sums
        f2_t yb = {0.f, 0.f};
        if constexpr (KIND == COL_LAPLACE) {
            ya = buf_load4(make_rsrc(A.xe + s0 * T * 4, (uint32_t)(D * T * 16)), tid * 16, d * (T * 16));
            yb = __builtin_bit_cast(f2_t, __builtin_amdgcn_raw_buffer_load_b64(
                     make_rsrc(A.xe2 + s0 * T * 2, (uint32_t)(D * T * 8)), tid * 8, d * (T * 8), 0));
            asm volatile("" ::: "memory");               // issued here, not where they are used
        }
        float a[E][CH];
        uint64_t acc[E];                                 // lanes whose element is an accumulator
        // One workgroup per CU (CH = 1): reads run AHEAD elements before their use, in that order, so that a wave's
        // arithmetic overlaps the other waves' reads (abs at N = M = 16384: 957 -> 856 us with the reads first and in
        // order). With several workgroups per CU the compiler's order is better (text size, 16384 elements: 302 against
        // 336 us).
        auto read = [&](int e) {
            const uint32_t x = addr(e);
            lds_read<CH>(a[e], x);
            acc[e] = SWAP ? __ballot(x >= split) : __ballot(x < split);
        };
        constexpr int AHEAD = CH == 1 ? 12 : E;
#pragma unroll
        for (int e = 0; e < AHEAD && e < E; ++e) read(e);
        const int dn = min(d + 1, d1 - 1);
        const uint32_t ab = aggb + (uint32_t)(d & 1) * AGGS;
        const int lane = lane_now(), el = min(lane & 15, W - 1);         // the wave whose aggregate this lane scans
        if constexpr (KIND == COL_ABS) {
            // Half of sum_n |k_n - x| w_n is sum_{k < x} (x - k) w less half of the sum over all keys of (x - k) w.
            // With x and k relative to the thread's anchor, a thread's own keys below give x W - K from its running
            // sums W = sum w, K = sum k w; the keys of the threads before, and the totals, then make one linear term S
            // x + F per thread. Across threads K runs relative to the median key: |k - median| w sums to no more than
            // the terms |k - q| w that the result is measured by.
            float own[E][CH], sw[CH], sk[CH], we[CH], ke[CH];
#pragma unroll
            for (int h = 0; h < CH; ++h) sw[h] = sk[h] = 0.f;
#pragma unroll
            for (int e = 0; e < E; ++e) {
                if (CH == 1 && (e & 3) == 0) {
                    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                    for (int i = e + AHEAD; i < e + AHEAD + 4 && i < E; ++i) read(i);
                }
#pragma unroll
                for (int h = 0; h < CH; ++h) {
                    const float x = unless(a[e][h], acc[e]);
                    if (e > 0) {
                        own[e][h] = fmaf(dv[e], sw[h], -sk[h]);
                        asm("" : "+v"(own[e][h]));    // now, or every element's sw and sk stay live
                        sw[h] += x;
                        sk[h] = fmaf(dv[e], x, sk[h]);
                    } else {
                        own[e][h] = 0.f;
                        sw[h] = x;
                        sk[h] = dv[e] * x;
                    }
                }
            }
            float wi[CH], ki[CH];
#pragma unroll
            for (int h = 0; h < CH; ++h) {
                we[h] = sw[h];
                ke[h] = fmaf(xs, sw[h], sk[h]);
                wi[h] = wave_scan_sum(we[h]);
                ki[h] = wave_scan_sum(ke[h]);
                we[h] = wi[h] - we[h];
                ke[h] = ki[h] - ke[h];
            }
            if (lane == WAVE - 1) {
#pragma unroll
                for (int h = 0; h < CH; ++h) {
                    f2_t x;
                    x.x = wi[h];
                    x.y = ki[h];
                    *(LDS_AS f2_t*)(ab + (wv * CH + h) * 8) = x;
                }
            }
            __syncthreads();
            float S[CH], F[CH];
#pragma unroll
            for (int h = 0; h < CH; ++h) {
                const f2_t x = *(LDS_AS const f2_t*)(ab + (el * CH + h) * 8);
                const float ww = row_scan_sum<W>(x.x), kk = row_scan_sum<W>(x.y);
                const float wtot = bcast(ww, W - 1), ktot = bcast(kk, W - 1);
                const float wb = wv ? bcast(ww, wv ? wv - 1 : 0) : 0.f, kb = wv ? bcast(kk, wv ? wv - 1 : 0) : 0.f;
                S[h] = we[h] + fmaf(-0.5f, wtot, wb);
                F[h] = fmaf(xs, S[h], -(ke[h] + fmaf(-0.5f, ktot, kb)));
            }
#pragma unroll
            for (int g = 0; g < E / 2; ++g) asm volatile("" : "+v"(tg[g]));    // addresses again, not kept in registers
            xp += T;
            if (d + 1 < d1) xs = *xp;
            const float weight = set_weight(A.sets, A.sets == 1 ? 0 : d % 3);
#pragma unroll
            for (int e = 0; e < E; ++e) {
                float o[CH];
#pragma unroll
                for (int h = 0; h < CH; ++h) o[h] = fmaf(weight, fmaf(dv[e], S[h], F[h] + own[e][h]), a[e][h]);
                lds_write_masked<CH>(o, addr(e), acc[e]);
                if ((e & 3) == 3) {                      // the next feature's elements over the ones just used
                    load(dn, e / 4);
                    __builtin_amdgcn_sched_barrier(0x1 | 0x2 | 0x4 | 0x80 | 0x100 | 0x200 | 0x400);
                }
            }
        } else {
            // L = sum over the keys below of e^-(x - k) w, R the same above. A thread's own sums, then the states
            // entering it from both sides, then each query adds L + R.
            const Decays y{ya[0], ya[1], ya[2], ya[3], yb.x, yb.y};
            float l[CH], r[CH], pr = 1.f;
#pragma unroll
            for (int h = 0; h < CH; ++h) l[h] = r[h] = 0.f;
#pragma unroll
            for (int e = 0; e < E; ++e) {
                if (CH == 1 && (e & 3) == 0) {
                    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                    for (int i = e + AHEAD; i < e + AHEAD + 4 && i < E; ++i) read(i);
                }
                pr *= dv[e];
#pragma unroll
                for (int h = 0; h < CH; ++h) {
                    const float x = unless(a[e][h], acc[e]);
                    l[h] = fmaf(dv[e], l[h], x);
                    r[h] = fmaf(pr, x, r[h]);
                }
            }
            wave_affine_up(y, l);
            wave_affine_down(y, r);
            if (lane == WAVE - 1) {
#pragma unroll
                for (int h = 0; h < CH; ++h) *(LDS_AS float*)(ab + (wv * CH + h) * 4) = l[h];
                *(LDS_AS float*)(ab + (2 * W * CH + wv) * 4) = y.before * y.own;
            }
            if (lane == 0) {
#pragma unroll
                for (int h = 0; h < CH; ++h) *(LDS_AS float*)(ab + (W * CH + wv * CH + h) * 4) = r[h];
            }
            float L[CH], R[CH];
#pragma unroll
            for (int h = 0; h < CH; ++h) {
                L[h] = dpp<WAVE_SHR1>(0.f, l[h]);
                R[h] = dpp<WAVE_SHL1>(0.f, r[h]);
            }
            __syncthreads();
            {
                const float a0_ = *(LDS_AS const float*)(ab + (2 * W * CH + el) * 4);
                float up[CH], dw[CH], a1 = a0_, a2 = a0_;
                const bool in = (lane & 15) < W;         // entries past the last wave are the identity
#pragma unroll
                for (int h = 0; h < CH; ++h) {
                    up[h] = *(LDS_AS const float*)(ab + (el * CH + h) * 4);
                    dw[h] = in ? *(LDS_AS const float*)(ab + (W * CH + el * CH + h) * 4) : 0.f;
                }
                row_affine_up<W>(a1, up);
                row_affine_down<W>(a2, dw);
#pragma unroll
                for (int h = 0; h < CH; ++h) {
                    const float lin = wv > 0 ? bcast(up[h], wv > 0 ? wv - 1 : 0) : 0.f;
                    const float rin = wv < W - 1 ? bcast(dw[h], wv < W - 1 ? wv + 1 : 0) : 0.f;
                    L[h] = fmaf(y.before, lin, L[h]);
                    R[h] = fmaf(y.after, rin, R[h]);
                }
            }
#pragma unroll
            for (int g = 0; g < E / 2; ++g) asm volatile("" : "+v"(tg[g]));
            // R at each element beside its word where the registers hold both (one rounding of the word per feature,
            // and fewer instructions: 372 -> 338 us at 12 x 8192, two channels); else added to the word on the way (27
            // spilled registers at 32 elements: 930 -> 1975 us)
            constexpr bool BESIDE = CH == 2 ? E <= 16 : E <= 24;
            float above[BESIDE ? E : 1][CH];
#pragma unroll
            for (int e = E - 1; e >= 0; --e) {
#pragma unroll
                for (int h = 0; h < CH; ++h) {           // R: at the element, without its own weight
                    if constexpr (BESIDE) {
                        above[e][h] = R[h];
                        R[h] = dv[e] * (R[h] + unless(a[e][h], acc[e]));
                    } else {
                        const float t = a[e][h] + R[h];  // query: its word + R; key: R past it
                        R[h] = dv[e] * pick(t, R[h], acc[e]);
                        a[e][h] = pick(a[e][h], t, acc[e]);
                    }
                }
            }
#pragma unroll
            for (int e = 0; e < E; ++e) {
                float o[CH];
#pragma unroll
                for (int h = 0; h < CH; ++h) {
                    if constexpr (BESIDE) {
                        L[h] = fmaf(dv[e], L[h], unless(a[e][h], acc[e]));
                        o[h] = a[e][h] + (L[h] + above[e][h]);
                    } else {
                        const float x = dv[e] * L[h];
                        o[h] = a[e][h] + x;              // query: its word + R + L; key: L past it
                        L[h] = pick(o[h], x, acc[e]);
                    }
                }
                lds_write_masked<CH>(o, addr(e), acc[e]);
                if ((e & 3) == 3) {
                    load(dn, e / 4);
                    __builtin_amdgcn_sched_barrier(0x1 | 0x2 | 0x4 | 0x80 | 0x100 | 0x200 | 0x400);
                }
            }
        }
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");       // the masked stores (lds_write_masked)
        __syncthreads();
    }
    for (int h = 0; h < CH; ++h) {
        if (c + h >= C) break;
        float* o = A.out + ((size_t)(p * DS + ds) * C + c + h) * Ma;
        for (int i = tid; i < Ma; i += T) o[i] = sm[(a0 + i) * CH + h];
    }
}

// ---------------------------------------------------------------------------------------------------------------
// col_dot: one workgroup per segment (p, d), all channels: the gradients of the abs sums in q and k
//
//   grad_q[m] = sum_c g_mc (2 W_c - Wtot_c), W_c the sum of v_nc over the keys below q_m    (an equal key counts above)
//   grad_k[n] = sum_c v_nc (2 G_c - Gtot_c), G_c the sum of g_mc over the queries below k_n (an equal query, too)
//
// The transposed loop of col_sum: a segment's merged order stays in registers (tags, and each element's running dot
// product), and the columns of g_w and v of one channel group after another go through LDS (copied there without
// registers while the previous group's arithmetic finishes). Per element and channel one random LDS read, two running
// sums and two multiply-adds. With g_u there is one more channel, g_u against ones.
// Queries come before equal keys in the merged order, so W is right as it runs; G is taken where the key's run of equal
// values began: kept as the thread goes, and where a run crosses threads (else a workgroup skips it) through LDS from
// the thread in which it began.
// ---------------------------------------------------------------------------------------------------------------
struct ColDotArgs {
    const uint16_t* tag; const uint32_t* eq;
    const float* gt; const float* vt;        // [P][CW][M][CH], [P][CW][N][CH]
    float* gq; float* gk;                    // (P, D, M) and, or null, (P, D, N)
    float* sums;                             // [S][E/4][T][4] scratch: the dot products where no registers are left
    float scale;                             // 2, or -2 for the sgn sum
    int D, N, M, K0, NP, CW;                 // NP: keys' words, N rounded up like K0
};

template <int T, int E, int CH>
__global__ __launch_bounds__(T, 4)
void col_dot(const ColDotArgs A)
{
    constexpr int W = T / WAVE;
    extern __shared__ float sm[];
    const int tid = threadIdx.x, lane = lane_id(), wv = wave_in_block();
    const int s = xcd_slice_block(blockIdx.x, gridDim.x), p = s / A.D;
    const int N = A.N, M = A.M, K0 = A.K0;
    // LDS words: queries [K0][CH], keys [NP + 1][CH], then aggregates [W][2 CH], then run starts [T][CH]
    const uint32_t aggb = ((uint32_t)(K0 + A.NP + 1) * CH * 4 + 15) & ~15u;
    const uint32_t runb = aggb + W * 2 * CH * 4;
    if (tid < CH) sm[(K0 + A.NP) * CH + tid] = 0.f;          // padding's word where N fills its region

    uint32_t tg[E / 2];
    {
        const u2_t* tp = (const u2_t*)(A.tag + (size_t)s * T * E) + tid;
#pragma unroll
        for (int g = 0; g < E / 4; ++g) {
            const u2_t y = tp[(size_t)g * T];
            tg[2 * g] = y.x;
            tg[2 * g + 1] = y.y;
        }
    }
    const uint32_t split = (uint32_t)K0 * CH * 4;
    auto addr = [&](int e) { return tag_addr<CH * 4>(tg[e / 2], e & 1); };
    uint64_t isq[E];
#pragma unroll
    for (int e = 0; e < E; ++e) isq[e] = __ballot(addr(e) < split);

    // runs of equal values within the thread (eq), and the elements that continue the run before it (cont)
    constexpr uint32_t FULL = E == 32 ? 0xffffffffu : (1u << E) - 1;
    const uint32_t eq = A.eq[(size_t)s * T + tid];
    const uint32_t cont = eq & ~(eq + 1);                    // trailing ones: elements of the run from before
    // the last thread before this one in which a run starts
    int from = 0;
    bool crossing = false;                                   // some run crosses threads
    {
        int* any = (int*)((char*)sm + aggb);
        const uint64_t b = __ballot(eq & 1);
        if (lane == 0) any[wv] = b != 0;
        __syncthreads();
        for (int i = 0; i < W; ++i) crossing |= any[i] != 0;
        crossing = uniform_u32(crossing) != 0;
        __syncthreads();
    }
    if (crossing) {
        int x = eq != FULL ? tid : -1;
#pragma unroll
        for (int off = 1; off < WAVE; off <<= 1) {
            const int y = __shfl_up(x, off, WAVE);
            if (lane >= off) x = max(x, y);
        }
        int* last = (int*)((char*)sm + aggb);
        if (lane == WAVE - 1) last[wv] = x;
        int ex = __shfl_up(x, 1, WAVE);
        if (lane == 0) ex = -1;
        __syncthreads();
        for (int i = 0; i < wv; ++i) ex = max(ex, last[i]);
        from = max(ex, 0);
    }

    // one channel group's columns into LDS: chunks of 64 x 16 bytes, shared out over the waves; lanes past a column
    // read 0
    auto fetch = [&](int cg) {
        const rsrc_t rg = make_rsrc(A.gt + ((size_t)p * A.CW + cg) * M * CH, (uint32_t)(M * CH * 4));
        const rsrc_t rv = make_rsrc(A.vt + ((size_t)p * A.CW + cg) * N * CH, (uint32_t)(N * CH * 4));
        const int qc = K0 * CH / 256, kc = A.NP * CH / 256;
        for (int i = wv; i < qc; i += W)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rg, (LDS_AS void*)(uint32_t)(i * 1024), 16, lane * 16, i * 1024, 0,
                                                     0);
        for (int i = wv; i < kc; i += W)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rv, (LDS_AS void*)(uint32_t)((qc + i) * 1024), 16, lane * 16,
                                                     i * 1024, 0, 0);
    };
    // The dot products over 8 groups at a time, then over those: sequential sums over all channels lost half a digit.
    // The latter in memory where registers do not hold both (spilled, their reloads would wait for the columns in
    // flight).
    constexpr bool IN_MEMORY = CH == 1 && E > 24;
    float sum[IN_MEMORY ? 1 : E], part[E];
    f4_t* sums = (f4_t*)(A.sums + (size_t)s * T * E) + tid;
#pragma unroll
    for (int e = 0; e < E; ++e) {
        part[e] = 0.f;
        if constexpr (!IN_MEMORY) sum[e] = 0.f;
    }
    __syncthreads();
    fetch(0);
    for (int cg = 0; cg < A.CW; ++cg) {
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
        float a[E][CH];
        constexpr int AHEAD = CH == 1 ? 12 : E;              // as in col_sum
#pragma unroll
        for (int e = 0; e < AHEAD && e < E; ++e) lds_read<CH>(a[e], addr(e));
        uint32_t eqc = eq, contc = cont;
        asm volatile("" : "+v"(eqc), "+v"(contc));           // their bits' masks are formed here, not kept all along
        float w[CH], g[CH], gr[CH];                          // running W and G, G where the element's run of equals began
#pragma unroll
        for (int h = 0; h < CH; ++h) w[h] = g[h] = gr[h] = 0.f;
        each<E>([&](auto ec) {
            constexpr int e = ec();
            if constexpr (CH == 1 && (e & 3) == 0) {
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int i = e + AHEAD; i < e + AHEAD + 4 && i < E; ++i) lds_read<CH>(a[i], addr(i));
            }
            const uint32_t same = bit_mask<e>(eqc);
#pragma unroll
            for (int h = 0; h < CH; ++h) {
                gr[h] = e > 0 ? bit_pick(g[h], gr[h], same) : 0.f;
                part[e] = fmaf(a[e][h], pick(gr[h], w[h], isq[e]), part[e]);
                w[h] += unless(a[e][h], isq[e]);
                g[h] += pick(0.f, a[e][h], isq[e]);
            }
            asm("" : "+v"(part[e]));
        });
        float w0[CH], g0[CH], wt[CH], gt[CH];
#pragma unroll
        for (int h = 0; h < CH; ++h) {
            w0[h] = wave_scan_sum(w[h]);
            g0[h] = wave_scan_sum(g[h]);
        }
        if (lane == WAVE - 1) {
#pragma unroll
            for (int h = 0; h < CH; ++h) {
                f2_t x;
                x.x = w0[h];
                x.y = g0[h];
                *(LDS_AS f2_t*)(aggb + (wv * CH + h) * 8) = x;
            }
        }
        __syncthreads();                                     // every wave has its words: the next group may land
        if (cg + 1 < A.CW) fetch(cg + 1);
        const int el = min(lane & 15, W - 1);
#pragma unroll
        for (int h = 0; h < CH; ++h) {
            const f2_t x = *(LDS_AS const f2_t*)(aggb + (el * CH + h) * 8);
            const float ww = row_scan_sum<W>(x.x), gg = row_scan_sum<W>(x.y);
            wt[h] = bcast(ww, W - 1);
            gt[h] = bcast(gg, W - 1);
            w0[h] += (wv ? bcast(ww, wv ? wv - 1 : 0) : 0.f) - w[h];
            g0[h] += (wv ? bcast(gg, wv ? wv - 1 : 0) : 0.f) - g[h];
        }
#pragma unroll
        for (int h = 0; h < CH; ++h) {
            w0[h] = fmaf(-0.5f, wt[h], w0[h]);
            gt[h] *= -0.5f;
        }
        if (!crossing) {
#pragma unroll
            for (int h = 0; h < CH; ++h) g0[h] += gt[h];
#pragma unroll
            for (int e = 0; e < E; ++e)
#pragma unroll
                for (int h = 0; h < CH; ++h) part[e] = fmaf(a[e][h], pick(g0[h], w0[h], isq[e]), part[e]);
        } else {
            float gc[CH];                                    // G where the run from before began
#pragma unroll
            for (int h = 0; h < CH; ++h) *(LDS_AS float*)(runb + (tid * CH + h) * 4) = g0[h] + gr[h];
            __syncthreads();
#pragma unroll
            for (int h = 0; h < CH; ++h) {
                gc[h] = *(LDS_AS const float*)(runb + (from * CH + h) * 4) + gt[h];
                g0[h] += gt[h];
            }
#pragma unroll
            for (int h = 0; h < CH; ++h)
                each<E>([&](auto ec) {
                    constexpr int e = ec();
                    const float z = bit_pick(g0[h], gc[h], bit_mask<e>(contc));
                    part[e] = fmaf(a[e][h], pick(z, w0[h], isq[e]), part[e]);
                });
        }
        if ((cg & 7) == 7 && cg + 1 < A.CW) {
            if constexpr (IN_MEMORY) {
#pragma unroll
                for (int g4 = 0; g4 < E / 4; ++g4) {
                    f4_t x = {part[4 * g4], part[4 * g4 + 1], part[4 * g4 + 2], part[4 * g4 + 3]};
                    if (cg > 7) x += sums[(size_t)g4 * T];
                    sums[(size_t)g4 * T] = x;
                }
            }
#pragma unroll
            for (int e = 0; e < E; ++e) {
                if constexpr (!IN_MEMORY) sum[e] += part[e];
                part[e] = 0.f;
            }
        }
    }
    __syncthreads();                                         // every wave has read its last words
#pragma unroll
    for (int e = 0; e < E; ++e) {                            // to query and key order through LDS (one word per element)
        const uint32_t t = tg[e / 2];
        float x = part[e];
        if constexpr (!IN_MEMORY) x += sum[e];
        else if (A.CW > 8) x += sums[(size_t)(e / 4) * T][e % 4];
        sm[(e & 1) ? t >> 16 : t & 0xffffu] = A.scale * x;
    }
    __syncthreads();
    float* gq = A.gq + (size_t)s * M;
    for (int i = tid; i < M; i += T) gq[i] = sm[spread(i, M)];
    if (A.gk) {
        float* gk = A.gk + (size_t)s * N;
        for (int i = tid; i < N; i += T) gk[i] = sm[K0 + spread(i, N)];
    }
}

// ---------------------------------------------------------------------------------------------------------------
// col_weights: the weight rows (P, Nw, C) as columns [P][CW][Nw][CH] in the order of their words, masked rows 0. With
// C1 = C + 1 there is one more channel, `extra` (P, Nw) or all ones. Also clears `bad` (bads words; null: 0) for the
// merge that comes after it.
// ---------------------------------------------------------------------------------------------------------------
constexpr int CF_T = 256, CF_M = 64;        // threads, rows per workgroup (also of col_finish)

template <int CH>
__global__ __launch_bounds__(CF_T)
void col_weights(const float* __restrict__ w, const float* __restrict__ extra, const uint8_t* __restrict__ keep,
                 float* __restrict__ out, float* __restrict__ bad, const int bads, const int Nw, const int C,
                 const int C1)
{
    __shared__ float tile[130][CF_M + 1];
    for (int i = blockIdx.x * CF_T + threadIdx.x; i < bads; i += gridDim.x * CF_T) bad[i] = 0.f;
    const int nb = (Nw + CF_M - 1) / CF_M;
    const int p = blockIdx.x / nb, n0 = (blockIdx.x - p * nb) * CF_M;
    const int rows = min(CF_M, Nw - n0), CW = (C1 + CH - 1) / CH;
    const float* src = w + ((size_t)p * Nw + n0) * C;
    int r = threadIdx.x / C, c = threadIdx.x - r * C;
    const int dr = CF_T / C, dc = CF_T - dr * C;
    for (int i = threadIdx.x; i < rows * C; i += CF_T) {
        const float x = src[i];
        tile[c][r] = (!keep || keep[(size_t)p * Nw + n0 + r] != 0) ? x : 0.f;
        r += dr;
        c += dc;
        if (c >= C) { c -= C; ++r; }
    }
    const int lane = threadIdx.x & (CF_M - 1);
    for (int cc = C + threadIdx.x / CF_M; cc < CW * CH; cc += CF_T / CF_M)
        if (lane < rows) tile[cc][lane] = cc < C1 ? (extra ? extra[(size_t)p * Nw + n0 + lane] : 1.f) : 0.f;
    __syncthreads();
    if (lane >= rows) return;
    float* dst = out + ((size_t)p * CW * Nw + spread(n0 + lane, Nw)) * CH;
    for (int g = threadIdx.x / CF_M; g < CW; g += CF_T / CF_M) {
        if constexpr (CH == 1) {
            dst[(size_t)g * Nw] = tile[g][lane];
        } else {
            f2_t x;
            x.x = tile[2 * g][lane];
            x.y = tile[2 * g + 1][lane];
            *(f2_t*)(dst + (size_t)g * Nw * 2) = x;
        }
    }
}

// ---------------------------------------------------------------------------------------------------------------
// col_finish: the feature shares' columns summed, turned into rows, with the v == 1 terms summed over the features
// ---------------------------------------------------------------------------------------------------------------
// scale: 2 for the abs sums, whose columns hold halves. bad (P, M): NaN at the rows that are NaN whatever the columns
// hold (emit_stream), 0 else. kind < 0: out = w and out_u = u; else the layer's epilogue on them, as
// layer_epilogue_kernel
__global__ __launch_bounds__(CF_T)
void col_finish(const float* __restrict__ cols, const float* __restrict__ u, const float* __restrict__ bad,
                float* __restrict__ out, float* __restrict__ out_u, const float scale, const int kind, const int masked,
                const ReduceEpilogue ep, const int D, const int M, const int C, const int DS)
{
    __shared__ float tile[128][CF_M + 1];
    __shared__ float us[CF_T / CF_M][CF_M];
    const int mb = (M + CF_M - 1) / CF_M;
    const int p = blockIdx.x / mb, m0 = (blockIdx.x - p * mb) * CF_M;
    const int lane = threadIdx.x & (CF_M - 1), wv = threadIdx.x / CF_M;
    const int m = spread(min(m0 + lane, M - 1), M);         // its word
    const float* src = cols + (size_t)p * DS * C * M + m;
    const float spoilt = bad[(size_t)p * M + m];         // 0 or NaN
#pragma unroll 4
    for (int c = wv; c < C; c += CF_T / CF_M) {
        float x = src[(size_t)c * M];
        for (int s = 1; s < DS; ++s) x += src[(size_t)(s * C + c) * M];
        tile[c][lane] = spoilt == spoilt ? scale * x : spoilt;
    }
    if (u) {
        const float* up = u + (size_t)p * D * M + m;
        float x = 0.f;
#pragma unroll 8
        for (int d = wv; d < D; d += CF_T / CF_M) x += up[(size_t)d * M];
        us[wv][lane] = x;
    }
    __syncthreads();
    const int rows = min(CF_M, M - m0);
    if (u && kind < 0 && threadIdx.x < rows)
        out_u[(size_t)p * M + m0 + lane] =
            spoilt == spoilt ? (us[0][lane] + us[1][lane]) + (us[2][lane] + us[3][lane]) : spoilt;
    float* dst = (kind < 0 ? out : ep.out) + ((size_t)p * M + m0) * C;
    const float np = (kind >= 0 && ep.n_pad) ? ep.n_pad[p] : 0.f;
    int r = threadIdx.x / C, c = threadIdx.x - r * C;
    const int dr = CF_T / C, dc = CF_T - dr * C;
    for (int i = threadIdx.x; i < rows * C; i += CF_T) {
        float x = tile[c][r];
        if (kind >= 0) {
            const float uu = (us[0][r] + us[1][r]) + (us[2][r] + us[3][r]);
            const float qv = ep.qt[(size_t)p * M + m0 + r];
            float den;
            if (kind == LAYER_ADD_RIESZ) {
                const float aqe = qv + LAYER_EPS;
                den = masked ? aqe * ((float)M - np) + ep.sak[p] - uu
                             : aqe * (float)M + ep.sak[p] - uu - LAYER_EPS * np;
                x = aqe * ep.vsum[(size_t)p * C + c] + ep.akv[(size_t)p * C + c] - x;
            } else {
                den = masked ? uu : uu - np * qv;
            }
            x /= fmaxf(den, LAYER_CLAMP);
        }
        dst[i] = x;
        r += dr;
        c += dc;
        if (c >= C) { c -= C; ++r; }
    }
}

// ---------------------------------------------------------------------------------------------------------------
// host
// ---------------------------------------------------------------------------------------------------------------
namespace {

constexpr size_t LDS_BYTES = 160 * 1024;

size_t sum_lds(int kind, int T, int CH, int n) {
    const size_t words = ((size_t)(n + 1) * CH * 4 + 15) & ~size_t(15);
    return words + 2 * (size_t)(kind == COL_ABS ? 2 : 3) * CH * (T / WAVE) * 4;
}

// words of a region rounded up to the 1 KB chunks col_dot copies
int pad_words(int n, int CH) { return (n + 256 / CH - 1) / (256 / CH) * (256 / CH); }

size_t dot_lds(int T, int CH, int N, int M) {
    const size_t words = ((size_t)(pad_words(M, CH) + pad_words(N, CH) + 1) * CH * 4 + 15) & ~size_t(15);
    return words + (size_t)(T / WAVE) * 2 * CH * 4 + (size_t)T * CH * 4;
}

// Workgroups of one col_sum launch that a CU holds at once: by LDS, and by the wave slots of 4 waves per SIMD (128
// VGPRs)
int wgs_per_cu(int kind, int T, int CH, int n) {
    return std::max(1, std::min((int)(LDS_BYTES / sum_lds(kind, T, CH, n)), 1024 / T));
}

}  // namespace

bool col_applies(int D, int N, int M) {
    if ((int64_t)N + M > COL_MAX) return false;
    const ColPlan pl = col_plan(COL_ABS, 1, D, N, M, 1);
    return (int64_t)D * pl.T * pl.E * 4 <= (int64_t)INT32_MAX;      // a p's stream within 32-bit buffer offsets
}

ColPlan col_plan(int kind, int P, int D, int N, int M, int C) {
    const int n = N + M;
    ColPlan pl{};
    // Two channels per workgroup where their words fit LDS (an 8-byte LDS read costs what a 4-byte one does, and the
    // stream is read once for both; the second of one channel is 0); the smallest workgroup whose threads hold at most
    // 16 elements then, so that several run per CU and fill each other's waits. The shape depends on n alone: what a
    // stream takes (col_applies) is the same for every C.
    if (n <= COL_MAX2) {
        pl.CH = 2;
        pl.T = 64;
        while (pl.T < 1024 && pl.T * (pl.T < 512 ? 16 : 20) < n) pl.T *= 2;
        pl.E = n <= pl.T * 12 ? 12 : n <= pl.T * 16 ? 16 : 20;
    } else {
        pl.CH = 1;
        pl.T = 1024;
        pl.E = n <= pl.T * 20 ? 20 : n <= pl.T * 24 ? 24 : n <= pl.T * 28 ? 28 : 32;
    }
    // Shares of the features: the fewest rounds of workgroups over the chip, in features walked one after another, plus
    // the loading and storing of the columns per round: about six features' time where a workgroup has a CU to itself,
    // two where others run beside it.
    pl.per_cu = wgs_per_cu(kind, pl.T, pl.CH, n);
    const int64_t wgs = (int64_t)P * ((C + pl.CH - 1) / pl.CH), slots = (int64_t)CUS * pl.per_cu;
    int64_t best = -1;
    for (int s = 1; s <= std::min(D, COL_SHARES); ++s) {
        const int64_t cost = ((wgs * s + slots - 1) / slots) * ((D + s - 1) / s + (pl.CH == 1 ? 6 : 2));
        if (best < 0 || cost < best) { best = cost; pl.DS = s; }
    }
    return pl;
}

// The plan of the abs backward's stream: col_dot's LDS also holds the regions' padding and the run starts.
bool col_bwd_applies(int D, int N, int M) {
    if (!col_applies(D, N, M)) return false;
    const ColPlan pl = col_plan(COL_ABS, 1, D, N, M, 1);
    return dot_lds(pl.T, pl.CH, N, M) <= LDS_BYTES &&
           sum_lds(COL_ABS, pl.T, pl.CH, pad_words(M, pl.CH) + N) <= LDS_BYTES;
}

int col_key0(const ColPlan& pl, int M) { return pad_words(M, pl.CH); }

size_t col_stream_bytes(int kind, const ColPlan& pl, int S) {
    const size_t L = (size_t)pl.T * pl.E, x = (size_t)S * pl.T * 4;
    auto al = [](size_t x) { return (x + 255) & ~size_t(255); };
    return al((size_t)S * L * 4) + al((size_t)S * L * 2) + (kind == COL_ABS ? 2 * al(x) : al(4 * x) + al(2 * x));
}

ColStream col_stream(int kind, const ColPlan& pl, void* base, int S) {
    const size_t L = (size_t)pl.T * pl.E, x = (size_t)S * pl.T * 4;
    auto al = [](size_t x) { return (x + 255) & ~size_t(255); };
    char* b = (char*)base;
    ColStream r{};
    r.val = (float*)b;     b += al((size_t)S * L * 4);
    r.tag = (uint16_t*)b;  b += al((size_t)S * L * 2);
    r.xe = (float*)b;      b += al(kind == COL_ABS ? x : 4 * x);
    if (kind == COL_ABS) r.eq = (uint32_t*)b;
    else r.xe2 = (float*)b;
    return r;
}

namespace {

// every workgroup shape col_plan returns
template <class F>
int dispatch_shape(const ColPlan& pl, F f) {
#define QLKA_COL(TT, EE, CC) \
    if (pl.T == TT && pl.E == EE && pl.CH == CC) \
        return f(std::integral_constant<int, TT>{}, std::integral_constant<int, EE>{},                                 \
                 std::integral_constant<int, CC>{})
    QLKA_COL(64, 12, 2); QLKA_COL(64, 16, 2); QLKA_COL(128, 12, 2); QLKA_COL(128, 16, 2); QLKA_COL(256, 12, 2);
    QLKA_COL(256, 16, 2); QLKA_COL(512, 12, 2); QLKA_COL(512, 16, 2); QLKA_COL(1024, 12, 2); QLKA_COL(1024, 16, 2);
    QLKA_COL(512, 20, 2); QLKA_COL(1024, 20, 2);
    QLKA_COL(1024, 20, 1); QLKA_COL(1024, 24, 1); QLKA_COL(1024, 28, 1); QLKA_COL(1024, 32, 1);
#undef QLKA_COL
    return (int)hipErrorInvalidValue;
}

// Lets the kernel use all of a CU's LDS on the stream's device. The attribute belongs to one device's copy of the
// kernel (and is set for the current device's), so `once`, one per kernel, keeps account by device.
template <class K>
int allow_lds(K kernel, PerDevice& once, hipStream_t st) {
    int cur = 0;
    if (hipError_t e = hipGetDevice(&cur)) return (int)e;
    hipDevice_t dev = cur;
    if (st != nullptr)
        if (hipError_t e = hipStreamGetDevice(st, &dev)) return (int)e;
    return once(dev, [&] {
        hipError_t e = dev == cur ? hipSuccess : hipSetDevice(dev);
        if (e != hipSuccess) return (int)e;
        e = hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)LDS_BYTES);
        const hipError_t back = dev == cur ? hipSuccess : hipSetDevice(cur);
        return (int)(e != hipSuccess ? e : back); });
}

template <int KIND, int T, int E>
int launch_merge(const ColMergeArgs& a, int S, hipStream_t st) {
    static PerDevice once;
    if (int e = allow_lds(col_merge<KIND, T, E>, once, st)) return e;
    const size_t lds = (size_t)(a.N + a.M + 3 * (T / WAVE)) * 4;
    hipLaunchKernelGGL((col_merge<KIND, T, E>), dim3((unsigned)S), dim3(T), lds, st, a);
    return (int)hipGetLastError();
}

template <int KIND, int T, int E, int CH, bool SWAP>
int launch_sum(const ColSumArgs& a, hipStream_t st) {
    static PerDevice once;
    if (int e = allow_lds(col_sum<KIND, T, E, CH, SWAP, 4>, once, st)) return e;
    const unsigned blocks = (unsigned)(a.P * a.DS * ((a.C + CH - 1) / CH));
    hipLaunchKernelGGL((col_sum<KIND, T, E, CH, SWAP, 4>), dim3(blocks), dim3(T), sum_lds(KIND, T, CH, a.K0 + a.N), st,
                       a);
    return (int)hipGetLastError();
}

}  // namespace

// Against the two sorts and the merge, whole prep of a call: 1536 elements 66 -> 47 us (2048 segments), 8192 210 -> 126
// us (1536; with a key mask also the 60 us of its fill), 16384 178 -> 156 us (768). Threads of more than 16 elements
// spill here (32768: 629 against 412 us).
bool col_sort_applies(const ColPlan& pl) { return pl.E <= 16; }

int col_sort_launch(int kind, const ColPlan& pl, const float* q, const float* k, const uint8_t* keep, ColStream str,
                    float* u, float* bad, int S, int D, int N, int M, hipStream_t st) {
    const ColMergeArgs a{q, nullptr, k, nullptr, keep, str.val, str.tag, str.xe, str.xe2, nullptr, u, bad, D, N, M, M,
                         1};
    StageTimer t("col_sort", st);
    return dispatch_shape(pl, [&](auto T, auto E, auto) {
        if constexpr (E() > 16) {
            return (int)hipErrorInvalidValue;
        } else {
            const size_t lds = (size_t)sort_words(T(), E()) * 4;
            if (kind == COL_ABS) {
                static PerDevice once;
                if (int e = allow_lds(col_sort<COL_ABS, T(), E()>, once, st)) return e;
                hipLaunchKernelGGL((col_sort<COL_ABS, T(), E()>), dim3((unsigned)S), dim3(T()), lds, st, a);
            } else {
                static PerDevice once;
                if (int e = allow_lds(col_sort<COL_LAPLACE, T(), E()>, once, st)) return e;
                hipLaunchKernelGGL((col_sort<COL_LAPLACE, T(), E()>), dim3((unsigned)S), dim3(T()), lds, st, a);
            }
            return (int)hipGetLastError();
        } });
}

int col_merge_launch(int kind, const ColPlan& pl, const float* qs, const uint32_t* qp, const float* ks,
                     const uint32_t* kp, const uint8_t* keep, ColStream str, float* u, float* bad, int S, int D, int N,
                     int M, bool bwd, int sets, hipStream_t st) {
    const ColMergeArgs a{qs, qp, ks, kp, keep, str.val, str.tag, str.xe, str.xe2, bwd ? str.eq : nullptr, u, bad, D, N,
                         M, bwd ? col_key0(pl, M) : M, sets};
    S *= sets;
    StageTimer t("col_merge", st);
    return dispatch_shape(pl, [&](auto T, auto E, auto) {
        return kind == COL_ABS ? launch_merge<COL_ABS, T(), E()>(a, S, st)
                               : launch_merge<COL_LAPLACE, T(), E()>(a, S, st); });
}

int col_weights_launch(const ColPlan& pl, const float* w, const uint8_t* keep, bool more, const float* extra, float* wt,
                       float* bad, int bads, int P, int Nw, int C, hipStream_t st) {
    StageTimer t("col_weights", st);
    const dim3 grid((unsigned)(P * ((Nw + CF_M - 1) / CF_M)));
    if (pl.CH == 2)
        hipLaunchKernelGGL(col_weights<2>, grid, dim3(CF_T), 0, st, w, extra, keep, wt, bad, bads, Nw, C,
                           C + (more ? 1 : 0));
    else
        hipLaunchKernelGGL(col_weights<1>, grid, dim3(CF_T), 0, st, w, extra, keep, wt, bad, bads, Nw, C,
                           C + (more ? 1 : 0));
    return (int)hipGetLastError();
}

int col_sum_launch(int kind, const ColPlan& pl, ColStream str, const float* wt, float* cols, int P, int D, int N, int M,
                   int C, int sets, hipStream_t st) {
    const int CW = (C + pl.CH - 1) / pl.CH;
    const ColSumArgs a{str.val, str.tag, str.xe, str.xe2, wt, cols, P, D * sets, N, M, C, pl.DS, M, CW, sets};
    StageTimer t(kind == COL_ABS ? "col_sum_abs" : "col_sum_laplace", st);
    return dispatch_shape(pl, [&](auto T, auto E, auto CH) {
        return kind == COL_ABS ? launch_sum<COL_ABS, T(), E(), CH(), false>(a, st)
                               : launch_sum<COL_LAPLACE, T(), E(), CH(), false>(a, st); });
}

int col_grad_v_launch(const ColPlan& pl, ColStream str, const float* gt, int CW, float* cols, int P, int D, int N,
                      int M, int C, hipStream_t st) {
    const ColSumArgs a{str.val, str.tag, str.xe, str.xe2, gt, cols, P, D, N, M, C, pl.DS, col_key0(pl, M), CW, 1};
    StageTimer t("col_grad_v", st);
    return dispatch_shape(pl, [&](auto T, auto E, auto CH) {
        return launch_sum<COL_ABS, T(), E(), CH(), true>(a, st); });
}

int col_dot_launch(const ColPlan& pl, ColStream str, const float* gt, const float* vt, int CW, float scale, float* gq,
                   float* gk, int S, int D, int N, int M, hipStream_t st) {
    const ColDotArgs a{str.tag, str.eq, gt, vt, gq, gk, str.val, scale, D, N, M, col_key0(pl, M), pad_words(N, pl.CH),
                       CW};
    StageTimer t("col_dot", st);
    return dispatch_shape(pl, [&](auto T, auto E, auto CH) {
        static PerDevice once;
        if (int e = allow_lds(col_dot<T(), E(), CH()>, once, st)) return e;
        hipLaunchKernelGGL((col_dot<T(), E(), CH()>), dim3((unsigned)S), dim3(T()), dot_lds(T(), CH(), N, M), st, a);
        return (int)hipGetLastError(); });
}

int col_finish_launch(int kind, int layer, bool masked, const ColPlan& pl, const float* cols, const float* u,
                      const float* bad, float* out, float* out_u, const ReduceEpilogue& ep, int P, int D, int M, int C,
                      hipStream_t st) {
    StageTimer t("col_finish", st);
    hipLaunchKernelGGL(col_finish, dim3((unsigned)(P * ((M + CF_M - 1) / CF_M))), dim3(CF_T), 0, st, cols, u, bad, out,
                       out_u, kind == COL_ABS ? 2.f : 1.f, layer, masked ? 1 : 0, ep, D, M, C, pl.DS);
    return (int)hipGetLastError();
}

}  // namespace qlka
