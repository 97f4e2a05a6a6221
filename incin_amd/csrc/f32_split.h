// Single precision on the 16-bit matrix instructions: an f32 value is the sum of three bf16 values (8 + 8 + 8 of its 24 significant bits;
// exact down to 2^-110, below which the last of them loses bits), and a product of two such sums is six products of bf16
// operands - those down to 2^-16 of the leading one - accumulated in f32, smallest first.  What is left out is at most 2^-25 of a
// product, half a rounding of single precision.  Against 64 bits, N(0,1) operands, sums over 64 / 128 values: 1.10e-7 / 1.63e-7 of the
// 2-norm, where the IEEE-f32 instruction, which rounds four times as often, leaves 1.44e-7 / 2.04e-7 (all nine products: no change).
//
// What it is for: v_mfma_f32_32x32x2_f32 runs at a sixteenth of the bf16 rate and, measured, lets no vector instruction of either
// wavefront of the SIMD run beside it (a loop of it with an equal time of v_fma, v_exp or v_add_u32 on the other wavefront takes the sum of both, 177
// against 91 us; v_mfma_f32_32x32x16_bf16 with as much 224 against 186).  Six of the latter for eight of the former: 192 cycles instead of 512.
//
// What the parts do not hold: an infinity (inf - inf is a NaN in the second part, so what it reaches is NaN), a value whose first part rounds to
// infinity, and the last bits below 2^-110.  Kernels look at their results and at the sizes of their operands, and do a block
// over with EXACT, in the IEEE-f32 instruction on the same operands (then kept whole, in two halves), where a result is not finite or where the bits
// lost - at most 2^-134 of each operand - could be more than half of a rounding of the smallest result.
#pragma once
#include "sdpa_mfma_common.h"

namespace incin_rocm {

typedef float float8v __attribute__((ext_vector_type(8)));
typedef unsigned uint4p __attribute__((ext_vector_type(4)));

// Eight values: three operands of the 16-bit matrix instructions.
struct Split8 { uint4p h, m, l; };

// Two values into parts (the first in the low halves).
template <bool EXACT> __device__ __forceinline__ void split_pair(float a, float b, unsigned& h, unsigned& m, unsigned& l)
{
    if (!EXACT) {
        // (whole() keeps the compiler from converting a value once more, by itself, where only its half of a pair is looked at)
        auto whole = [](unsigned w) __attribute__((always_inline)) { asm("" : "+v"(w)); return w; };
        h = whole(pack2<bf16_t>(a, b));
        const float ra = a - __uint_as_float(h << 16), rb = b - __uint_as_float(h & 0xffff0000u);
        m = whole(pack2<bf16_t>(ra, rb));
        l = pack2<bf16_t>(ra - __uint_as_float(m << 16), rb - __uint_as_float(m & 0xffff0000u));
        return;
    }
    // the values as they are: their upper halves, their lower halves
    h = __float_as_uint(a) >> 16 | (__float_as_uint(b) & 0xffff0000u);
    m = (__float_as_uint(a) & 0xffffu) | __float_as_uint(b) << 16;
    l = 0;
}
// Eight values times c.  (The parts are those of the products before they are rounded: what the first leaves is one fused operation.)
template <bool EXACT> __device__ __forceinline__ Split8 split8_scaled(const float8v& x, float c)
{
    Split8 o;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const float x0 = x[2 * i], x1 = x[2 * i + 1], a = x0 * c, b = x1 * c;
        unsigned h, m, l;
        if (EXACT) split_pair<true>(a, b, h, m, l);
        else {
            auto whole = [](unsigned w) __attribute__((always_inline)) { asm("" : "+v"(w)); return w; };
            h = whole(pack2<bf16_t>(a, b));
            const float ra = __builtin_fmaf(x0, c, -__uint_as_float(h << 16)), rb = __builtin_fmaf(x1, c, -__uint_as_float(h & 0xffff0000u));
            m = whole(pack2<bf16_t>(ra, rb));
            l = pack2<bf16_t>(ra - __uint_as_float(m << 16), rb - __uint_as_float(m & 0xffff0000u));
        }
        o.h[i] = h;
        o.m[i] = m;
        o.l[i] = l;
    }
    return o;
}

// c += a b, 32 x 32 over 16 values of the summed axis: lane (n = lane % 32, g = lane / 32) holds values 8 g .. 8 g + 7 of row (a) or
// column (b) n.
template <bool EXACT> __device__ __forceinline__ floatx16 mma_split(const Split8& a, const Split8& b, floatx16 c)
{
    if (!EXACT) {
        auto run = [&](const uint4p& x, const uint4p& y) __attribute__((always_inline)) { c = Mma<bf16_t>::run(__builtin_bit_cast(bf16x8, x), __builtin_bit_cast(bf16x8, y), c); };
        run(a.l, b.h);
        run(a.m, b.m);
        run(a.h, b.l);
        run(a.m, b.h);
        run(a.h, b.m);
        run(a.h, b.h);
        return c;
    }
    // (value e of the two lanes of a row is one step of two values)
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        auto whole = [&](const Split8& x) __attribute__((always_inline)) {
            return __uint_as_float(e & 1 ? (x.h[e / 2] & 0xffff0000u) | x.m[e / 2] >> 16 : x.h[e / 2] << 16 | (x.m[e / 2] & 0xffffu));
        };
        c = __builtin_amdgcn_mfma_f32_32x32x2f32(whole(a), whole(b), c, 0, 0, 0);
    }
    return c;
}

// The same one instruction at a time (K of 6), for vector work in between; EXACT: all with the last.
template <bool EXACT, int K> __device__ __forceinline__ void mma_split_term(const Split8& a, const Split8& b, floatx16& c)
{
    if (EXACT) {
        if (K == 5) c = mma_split<true>(a, b, c);
        return;
    }
    const uint4p& x = K == 0 ? a.l : K == 1 || K == 3 ? a.m : a.h;
    const uint4p& y = K == 2 ? b.l : K == 1 || K == 4 ? b.m : b.h;
    c = Mma<bf16_t>::run(__builtin_bit_cast(bf16x8, x), __builtin_bit_cast(bf16x8, y), c);
}

// Two values into parts in three pieces of three to five instructions.
struct SplitPair {
    float ra, rb;
    template <bool EXACT, int PART> __device__ __forceinline__ void step(float a, float b, unsigned& h, unsigned& m, unsigned& l)
    {
        if (EXACT) {
            if (PART == 2) split_pair<true>(a, b, h, m, l);
            return;
        }
        auto whole = [](unsigned w) __attribute__((always_inline)) { asm("" : "+v"(w)); return w; };
        if (PART == 0) {
            h = whole(pack2<bf16_t>(a, b));
            ra = a - __uint_as_float(h << 16);
        } else if (PART == 1) {
            rb = b - __uint_as_float(h & 0xffff0000u);
            m = whole(pack2<bf16_t>(ra, rb));
        } else {
            l = pack2<bf16_t>(ra - __uint_as_float(m << 16), rb - __uint_as_float(m & 0xffff0000u));
        }
    }
};

// ---- sizes: the largest of what is split (one instruction for two values), the smallest of what comes out --------------------------------
// (the inputs of `largest` are values as loaded or multiplied, not results of matrix instructions: the compiler places no wait states for those here)
__device__ __forceinline__ float largest(float top, float a, float b)
{
    asm("v_max3_f32 %0, |%1|, |%2|, %0" : "+v"(top) : "v"(a), "v"(b));
    return top;
}
// Twice the bits of the smallest magnitude that is not zero, less one (zeros only: all ones).
__device__ __forceinline__ unsigned smallest(unsigned low, float x) { return min(low, (__float_as_uint(x) << 1) - 1u); }
__device__ __forceinline__ unsigned smallest_of(float x) { return (__float_as_uint(x) << 1) - 1u; }      // (x > 0)
// A wavefront's maximum / minimum.
template <bool MAX> __device__ __forceinline__ unsigned wave_extreme(unsigned x)
{
    auto take = [](unsigned a, unsigned b) __attribute__((always_inline)) { return MAX ? max(a, b) : min(a, b); };
    x = take(x, (unsigned)__builtin_amdgcn_mov_dpp((int)x, 0xb1, 0xf, 0xf, true));       // lane ^ 1
    x = take(x, (unsigned)__builtin_amdgcn_mov_dpp((int)x, 0x4e, 0xf, 0xf, true));       // lane ^ 2
    x = take(x, (unsigned)__builtin_amdgcn_mov_dpp((int)x, 0x141, 0xf, 0xf, true));      // 7 - lane of the eight
    x = take(x, (unsigned)__builtin_amdgcn_mov_dpp((int)x, 0x140, 0xf, 0xf, true));      // 15 - lane of the sixteen
    auto at = [&](int lane) __attribute__((always_inline)) { return (unsigned)__builtin_amdgcn_readlane((int)x, lane); };
    return take(take(at(0), at(16)), take(at(32), at(48)));
}
constexpr float SPLIT_TINY = 0x1p-100f;      // (parts hold values from 2^-110 on whole)
constexpr float SPLIT_LOST = 0x1p-110f;      // 2^24 times the 2^-134 that a value below 2^-110 loses at most

// Tiles of ROWS rows of a tensor as three planes of bf16 rows in LDS, 2 D bytes a row, 16-byte chunks swizzled as the 16-bit kernels'
// K (BY_K) or V tiles: a workgroup's THREADS threads fetch the next tile's values into registers, eight to a thread at a time, and put
// their parts into LDS when the place is free.  DC: the columns that anybody reads.
template <int D, int DC, int ROWS, int THREADS> struct SplitTile {
    typedef PfLayout<D> L;
    static constexpr int ROWB = L::ROWB, PLANE = ROWS * ROWB, BYTES = 3 * PLANE;
    static constexpr int CPR = DC / 8, N = ROWS * CPR / THREADS;      // eights per row; of a thread
    static constexpr int STEPS = N * 4 * 3;                           // pieces of the splitting of a thread's values
    static_assert(ROWS * CPR % THREADS == 0, "whole eights per thread");
    float8v x[N];
    // rows [row0, row0 + ROWS) of `rows` rows (`width` values each, `stride` apart); what lies beyond arrives as zeros
    __device__ __forceinline__ void fetch(const float* base, int64_t stride, int width, int rows, int row0, int tid)
    {
        int64_t rem = (int64_t)(rows - row0 - 1) * stride * 4 + width * 4;
        rem = rem < 0 || row0 >= rows ? 0 : rem > 0x7fffffffLL ? 0x7fffffffLL : rem;
        const __amdgpu_buffer_rsrc_t r = __builtin_amdgcn_make_buffer_rsrc((void*)(base + (int64_t)row0 * stride), 0, (int)rem, 0x00020000);
#pragma unroll
        for (int i = 0; i < N; ++i) {
            const int pos = i * THREADS + tid, row = pos / CPR, c = pos % CPR;
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const uint4p w = __builtin_bit_cast(uint4p, __builtin_amdgcn_raw_buffer_load_b128(r, dma_chunk_offset(row, (int)stride * 4, 2 * c + h, width * 4), 0, 0));
#pragma unroll
                for (int e = 0; e < 4; ++e) x[i][4 * h + e] = __uint_as_float(w[e]);
            }
        }
    }
    // The same for rows of any stride; those beyond the last repeat it (nobody stores what they give).
    __device__ __forceinline__ void fetch_any(const float* base, int64_t stride, int width, int rows, int row0, int tid)
    {
#pragma unroll
        for (int i = 0; i < N; ++i) {
            const int pos = i * THREADS + tid, row = pos / CPR, c = pos % CPR;
            const float* at = base + (int64_t)min(row0 + row, rows - 1) * stride;
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const bool in = 8 * c + 4 * h < width;
                const uint4p w = *(const uint4p*)(at + (in ? 8 * c + 4 * h : 0));
#pragma unroll
                for (int e = 0; e < 4; ++e) x[i][4 * h + e] = in ? __uint_as_float(w[e]) : 0.0f;
            }
        }
    }
    // Piece k of STEPS of splitting what is fetched; eight values are in `s` after twelve of them, and put_step stores them then.
    struct State { SplitPair pair; Split8 o; };
    template <bool EXACT> __device__ __forceinline__ void split_step(int k, State& s, Split8& o)
    {
        const int i = k / 12, q = k / 3 % 4, part = k % 3;
        unsigned h = o.h[q], m = o.m[q], l = o.l[q];
        if (part == 0) s.pair.template step<EXACT, 0>(x[i][2 * q], x[i][2 * q + 1], h, m, l);
        else if (part == 1) s.pair.template step<EXACT, 1>(x[i][2 * q], x[i][2 * q + 1], h, m, l);
        else s.pair.template step<EXACT, 2>(x[i][2 * q], x[i][2 * q + 1], h, m, l);
        o.h[q] = h;
        o.m[q] = m;
        o.l[q] = l;
    }
    // The largest magnitude of a thread's values, piece by piece of the splitting.
    __device__ __forceinline__ float largest_step(int k, float top) const
    {
        return k % 3 ? top : largest(top, x[k / 12][2 * (k / 3 % 4)], x[k / 12][2 * (k / 3 % 4) + 1]);
    }
    __device__ __forceinline__ float largest_of(float top) const
    {
#pragma unroll
        for (int k = 0; k < STEPS; k += 3) top = largest_step(k, top);
        return top;
    }
    __device__ __forceinline__ unsigned smallest_in(unsigned low) const
    {
#pragma unroll
        for (int i = 0; i < N; ++i)
#pragma unroll
            for (int e = 0; e < 8; ++e) low = smallest(low, x[i][e]);
        return low;
    }
    template <bool BY_K> static __device__ __forceinline__ void store(char* tile, const Split8& o, int tid, int i = 0)      // (eight i of the thread's)
    {
        const int pos = i * THREADS + tid, row = pos / CPR, c = pos % CPR;
        char* at = tile + row * ROWB + ((c ^ (BY_K ? L::fk(row) : L::fv(row))) << 4);
        *(uint4p*)at = o.h;
        *(uint4p*)(at + PLANE) = o.m;
        *(uint4p*)(at + 2 * PLANE) = o.l;
    }
    template <bool EXACT, bool BY_K> __device__ __forceinline__ void put_step(int k, State& s, char* tile, int tid)
    {
        split_step<EXACT>(k, s, s.o);
        if (k % 12 == 11) store<BY_K>(tile, s.o, tid, k / 12);
    }
    template <bool EXACT, bool BY_K> __device__ __forceinline__ void put(char* tile, int tid)
    {
        State s;
#pragma unroll
        for (int k = 0; k < STEPS; ++k) put_step<EXACT, BY_K>(k, s, tile, tid);
    }
    // All of a thread's values times c.
    template <bool EXACT, bool BY_K> __device__ __forceinline__ void put_scaled(char* tile, float c, int tid)
    {
#pragma unroll
        for (int i = 0; i < N; ++i) store<BY_K>(tile, split8_scaled<EXACT>(x[i], c), tid, i);
    }
    // Whether one of them times c is outside of 2^-100 (zero apart) to 2^60.
    // (`width`: as fetched.  Where no value is zero, one instruction a value)
    __device__ __forceinline__ bool scaled_beyond(float c, int width, int tid) const
    {
        float least = INFINITY;
#pragma unroll
        for (int i = 0; i < N; ++i) {
            float of = INFINITY;
#pragma unroll
            for (int e = 0; e < 8; ++e) of = __builtin_fminf(of, __builtin_fabsf(x[i][e]));
            if ((i * THREADS + tid) % CPR * 8 < width) least = __builtin_fminf(least, of);
        }
        const float most = largest_of(0.0f) * __builtin_fabsf(c);
        if (most <= 0x1p60f && least * __builtin_fabsf(c) >= SPLIT_TINY) return false;
        const float low = __uint_as_float((smallest_in(~0u) + 1u) >> 1);      // (zeros only: zero)
        return !(most <= 0x1p60f) || (low * __builtin_fabsf(c) < SPLIT_TINY && low * c != 0.0f);
    }
    static __device__ __forceinline__ Split8 rows_operand(const char* at)      // at: this lane's chunk in the first plane
    {
        return Split8{*(const uint4p*)at, *(const uint4p*)(at + PLANE), *(const uint4p*)(at + 2 * PLANE)};
    }
    // 16 rows by columns: two transposing reads a plane (addresses of the rows 4 g .. and 8 + 4 g ..)
    static __device__ __forceinline__ Split8 cols_operand(const char* tile, int lo, int hi)
    {
        Split8 o;
#pragma unroll
        for (int x = 0; x < 3; ++x) {
            short8v v;
            v.lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((short4v __attribute__((address_space(3)))*)(tile + lo + x * PLANE));
            v.hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((short4v __attribute__((address_space(3)))*)(tile + hi + x * PLANE));
            (x == 0 ? o.h : x == 1 ? o.m : o.l) = __builtin_bit_cast(uint4p, v);
        }
        return o;
    }
};

// Every wavefront of the workgroup is here and its LDS accesses are done.  (Loads into registers stay in flight.)
__device__ __forceinline__ void lds_barrier()
{
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}

}  // namespace incin_rocm
