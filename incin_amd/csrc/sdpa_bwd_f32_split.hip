// f32 attention backward for head dimensions up to 64 with the products of sdpa_bwd_f32.hip through the bf16 matrix instruction, every
// value as the sum of three bf16 ones (f32_split.h: six instructions for eight of the IEEE-f32 one, 192 cycles for 512, no larger error).  The
// formulas, the row statistics that start the accumulators and the meeting of wavefronts that share a block are that file's, which see.
//
// A workgroup of eight wavefronts owns 128 rows of one operand pair and streams 64-row tiles of the other:
//
//   dK / dV item   owns keys: X = K' (K * scale * log2 e), Y = V; streams A = Q, B = dO of the group's heads, and their -L log2 e, -D
//   dQ item        owns queries: X = Q', Y = dO; streams A = K, B = V
//
//   s = A X^T (lane owns a row of X, registers are rows of A), dp = B Y^T, P = exp2(s), dS = P dp,
//   dX^T += A^T dS,  and for keys  dV^T += B^T P
//
// for both.  Four blocks of 32 owned rows side by side, two wavefronts to each, which take a block of 32 rows of every tile each.  The owned
// rows' parts stay in LDS (96 KiB): as operands in registers they would be 96 of them beside 64 accumulators, and a wavefront that has its SIMD
// to itself hides nothing.  The tile's parts (48 KiB) are split once per workgroup, by the threads that fetched them, while the last
// product of the tile before runs.  Between the products' instructions, where vector instructions cost least (f32_split.h): the exponentials and
// parts of P under dp, those of dS under dV (for queries: its second half under the first half of dQ), the next tile's under dK.
// One barrier before a tile's parts are replaced and one behind; what a product starts with is read while the one before ends.  P and dP are summed
// smaller products first, the row statistics added last: gradients are 0.3 - 0.45 of what the IEEE products left off 64 bits (2-norm, 24 heads x 600,
// D = 64: 1.24e-6 -> 4.2e-7).
//
// What bounds it: the matrix instructions of a block (96 for keys, 72 for queries; 32 heads x 1024 causal, pipes busy for 48 % of the time in which a compute unit has work) under
// the clock the device keeps with them, and waits for LDS and barriers (36 % of wavefront time; both wavefronts of a SIMD belong to one workgroup).
// Measured, backward call with the row statistics, us, IEEE products / so: 32 heads x 1024 causal 144 / 96, nothing masked 242 / 156, 96 x 2048 causal 1486 / 965, 96 x
// 512 133 / 94, 96 x 128 26.5 / 19.9, 32 x 1000 with a bias per head under a causal mask, as a tensor, 163 / 114.
#include <type_traits>

#include "f32_split.h"
#include "sdpa_bwd.h"

namespace incin_rocm {

constexpr int BS_OWN = 128, BS_KT = 64, BS_THREADS = 512;
typedef SplitTile<64, 64, BS_KT, BS_THREADS> BsTile;          // a streamed tile, one eight of values per thread
typedef SplitTile<64, 64, BS_OWN, BS_THREADS> BsOwn;
constexpr int BS_LDS = 2 * BsOwn::BYTES + 2 * BsTile::BYTES;  // X, Y, A, B

template <bool KEYS, bool DENSE>
__device__ __forceinline__ void bwd_f32_split_body(const SdpaBwdParams& bp, char* smem, float (&s_stats)[2][BS_KT], int (&s_vote)[6][8], int id)
{
#if defined(__HIP_DEVICE_COMPILE__)
    constexpr float LOG2E = 1.4426950408889634f;
    typedef BsTile::L L;
    typedef float float4v __attribute__((ext_vector_type(4)));
    const SdpaParams& p = bp.f;
    char* const own_x = smem;
    char* const own_y = smem + BsOwn::BYTES;
    char* const tile_a = smem + 2 * BsOwn::BYTES;
    char* const tile_b = tile_a + BsTile::BYTES;

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int own = wave % 4, rs = wave / 4;
    const int ql = lane & 31, g = lane >> 5;
    const int Sq = p.Sq, Skv = p.Skv, coff = Skv - Sq;

    // ---- which item: the orders of sdpa_bwd_f32.hip ----
    int b, hkv, hq = 0, o0;      // o0: first owned row
    if (KEYS) {
        // All key blocks of a (batch, KV head) pair read the same Q and dO rows: a pair is given to one XCD.  Under a mask first blocks first
        // (a causal mask leaves those the most rows).
        const int nkb = (Skv + BS_OWN - 1) / BS_OWN, pairs = p.B * p.Hkv, xcds = (pairs & 7) == 0 ? 8 : 1;
        const int xcd = xcds == 8 ? id & 7 : 0, r = xcds == 8 ? id >> 3 : id, per = pairs / xcds;
        const bool uneven = p.causal || DENSE;
        o0 = (uneven ? r / per : r % nkb) * BS_OWN;
        const int bhkv = (uneven ? r % per : r / nkb) * xcds + xcd;
        hkv = bhkv % p.Hkv;
        b = bhkv / p.Hkv;
    } else {
        const int nqb = (Sq + BS_OWN - 1) / BS_OWN, total = nqb * p.Hq * p.B;
        const WorkItem wi = work_item_of(p, id, total, nqb);
        hkv = wi.bhkv % p.Hkv;
        b = wi.bhkv / p.Hkv;
        hq = hkv * p.G + wi.gq;
        o0 = wi.qblk * BS_OWN;
    }
    const int kv_len = p.kv_lens ? clampi(p.kv_lens[b], 0, Skv) : Skv;
    const int rows_b = p.q_lens ? clampi(p.q_lens[b], 0, Sq) : Sq;      // query rows at and beyond are padding
    const int mine = o0 + own * 32 + ql;                                // this lane's key or query
    const int n_own = KEYS ? kv_len : rows_b, n_all_own = KEYS ? Skv : Sq, n_stream = KEYS ? rows_b : kv_len;

    // ---- the streamed rows that matter: [first, end) of them for the workgroup; of a wavefront, rows outside [w_first, w_end) see or are
    // seen by none of its owned rows, and inside [w_all, w_all_end) by all; of this lane, from lane_lo on and before lane_hi ----
    int first = 0, end = n_stream;
    int w_first = 0, w_end = n_stream, w_all = 0, w_all_end = n_stream, lane_lo = 0, lane_hi = n_stream;
    if (p.causal) {
        const int w0 = o0 + own * 32;
        if (KEYS) {
            first = clampi(o0 - coff, 0, n_stream);
            w_first = max(w0 - coff, 0);
            w_all = max(w0 + 31 - coff, 0);
            lane_lo = mine - coff;
        } else {
            end = clampi(min(o0 + BS_OWN - 1, rows_b - 1) + coff + 1, 0, kv_len);
            w_end = clampi(min(w0 + 31, rows_b - 1) + coff + 1, 0, kv_len);
            w_all_end = clampi(w0 + coff + 1, 0, kv_len);
            lane_hi = clampi(mine + coff + 1, 0, kv_len);
        }
    }
    if (o0 + own * 32 >= n_own) w_end = 0;
    int t_begin = first / BS_KT, t_end = o0 < n_own ? (end + BS_KT - 1) / BS_KT : 0;
    if (DENSE && p.mask_flags && t_end > t_begin) {
        // the tiles between the first and the last with a block that sees, or is seen by, any of the owned rows (keys: in any head of the group)
        const int nkb32 = (Skv + 31) >> 5, nrb32 = (Sq + 31) >> 5, lo32 = 2 * t_begin, n32 = min(2 * t_end, KEYS ? nrb32 : nkb32) - lo32;
        if (tid == 0) { s_vote[0][0] = 0x7fffffff; s_vote[0][1] = -1; }
        __syncthreads();
        int lo = 0x7fffffff, hi = -1;
        for (int x = tid; x < n32 * (KEYS ? p.G : 1); x += BS_THREADS) {
            const int s32 = lo32 + x % n32;
            const uint8_t* fl = mask_flags_of(p, b, KEYS ? hkv * p.G + x / n32 : hq);
            bool seen = false;
#pragma unroll
            for (int w = 0; w < 4; ++w) {
                const int o32 = min((o0 >> 5) + w, (KEYS ? nkb32 : nrb32) - 1);
                seen = seen || fl[KEYS ? (int64_t)s32 * nkb32 + o32 : (int64_t)o32 * nkb32 + s32] != 2;
            }
            if (seen) { lo = min(lo, s32); hi = max(hi, s32); }
        }
        if (hi >= 0) { atomicMin(&s_vote[0][0], lo); atomicMax(&s_vote[0][1], hi); }
        __syncthreads();
        const int a = __builtin_amdgcn_readfirstlane(s_vote[0][0]), z = __builtin_amdgcn_readfirstlane(s_vote[0][1]);
        t_end = z < 0 ? t_begin : z / 2 + 1;
        t_begin = z < 0 ? t_begin : a / 2;
        __syncthreads();
    }
    const int tiles = max(t_end - t_begin, 0), n_tiles = tiles * (KEYS ? p.G : 1);      // keys: the group's query heads one after another

    const float* const kp = (const float*)p.k + (int64_t)b * p.k_sb + (int64_t)hkv * p.k_sh;
    const float* const vp = (const float*)p.v + (int64_t)b * p.v_sb + (int64_t)hkv * p.v_sh;
    auto q_of = [&](int h) __attribute__((always_inline)) { return (const float*)p.q + (int64_t)b * p.q_sb + (int64_t)h * p.q_sh; };
    auto g_of = [&](int h) __attribute__((always_inline)) { return (const float*)bp.d_o + (int64_t)b * bp.do_sb + (int64_t)h * bp.do_sh; };

    // operand addresses in a tile: row ql of this wavefront's block by rows (chunk 2 s + g: ^ (s << 5)), by columns block db, half h of 16 rows;
    // and of the owned rows
    const int swz = ((g ^ (L::fk(ql) & 1)) << 4) + ((L::fk(ql) & ~1) << 4);
    const int row_base = (rs * 32 + ql) * L::ROWB + swz, own_base = (own * 32 + ql) * L::ROWB + swz;
    int col_addr[2][2];
    {
        const int n = lane & 15, dh = (lane >> 4) & 1;
#pragma unroll
        for (int db = 0; db < 2; ++db)
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const int r = 8 * h + 4 * g + (n >> 2), c = 4 * db + 2 * dh + ((n & 3) >> 1);
                col_addr[db][h] = (rs * 32 + r) * L::ROWB + ((c ^ L::fk(r)) << 4) + (n & 1) * 8;
            }
    }
    // queries: -L log2 e and -D of this lane's row
    float seed_s = 0.0f, seed_d = 0.0f;
    if (!KEYS && n_tiles > 0) {
        const int64_t stat = ((int64_t)b * p.Hq + hq) * Sq + min(mine, rows_b - 1);
        seed_s = bp.neg_l2[stat];
        seed_d = bp.neg_delta[stat];
    }

    constexpr int NACC = KEYS ? 4 : 2;
    floatx16 acc[NACC];      // dX^T (columns 0 - 31, 32 - 63), dV^T
    auto walk = [&](auto exact_) __attribute__((always_inline)) {
        constexpr bool EXACT = decltype(exact_)::value;
        BsTile xa, xb;
        float stat = 0.0f;      // keys: threads 0 - 63 fetch -L log2 e, 64 - 127 -D of the tile's rows
        auto fetch = [&](int n) __attribute__((always_inline)) {
            const int h = KEYS ? hkv * p.G + n / tiles : hq, row0 = (t_begin + n % tiles) * BS_KT;
            if (KEYS) {
                xa.fetch(q_of(h), p.q_ss, p.D, n_stream, row0, tid);
                xb.fetch(g_of(h), bp.do_ss, p.Dv, n_stream, row0, tid);
                const float* src = (tid < 64 ? bp.neg_l2 : bp.neg_delta) + ((int64_t)b * p.Hq + h) * Sq;
                const int r = row0 + (tid & 63);
                if (tid < 128) stat = r < n_stream ? src[r] : 0.0f;
            } else {
                xa.fetch(kp, p.k_ss, p.D, end, row0, tid);
                xb.fetch(vp, p.v_ss, p.Dv, end, row0, tid);
            }
        };
        auto put_stats = [&]() __attribute__((always_inline)) {
            if (KEYS && tid < 128) s_stats[tid >> 6][tid & 63] = stat;
        };
        fetch(0);
        [[maybe_unused]] float top_a = 0.0f, top_b = 0.0f;      // the largest magnitudes of this thread's share of A and B; A infinity: X wants EXACT
        {
            BsOwn x;
            const int rows = max(n_own, 1);
            if (KEYS) x.fetch_any(kp, p.k_ss, p.D, rows, o0, tid);
            else x.fetch_any(q_of(hq), p.q_ss, p.D, rows, o0, tid);
            // (a score's error by what A loses is negligible under an X up to 2^60, and X itself loses nothing from 2^-100 on)
            if (!EXACT && x.scaled_beyond(p.scale * LOG2E, p.D, tid)) top_a = INFINITY;
            x.template put_scaled<EXACT, true>(own_x, p.scale * LOG2E, tid);
            if (KEYS) x.fetch_any(vp, p.v_ss, p.Dv, rows, o0, tid);
            else x.fetch_any(g_of(hq), bp.do_ss, p.Dv, rows, o0, tid);
            if (!EXACT) {
                const unsigned top = wave_extreme<true>(__float_as_uint(x.largest_of(0.0f)));
                if (lane == 0) s_vote[5][wave] = (int)top;
            }
            x.template put<EXACT, true>(own_y, tid);
        }
        if (!EXACT) {
            top_a = xa.largest_of(top_a);
            top_b = xb.largest_of(top_b);
        }
        xa.template put<EXACT, true>(tile_a, tid);
        xb.template put<EXACT, true>(tile_b, tid);
        put_stats();
#pragma unroll
        for (int x = 0; x < NACC; ++x)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[x][r] = 0.0f;
        lds_barrier();
        for (int n = 0; n < n_tiles; ++n) {
            const bool more = n + 1 < n_tiles;
            if (more) fetch(n + 1);
            const int i0 = (t_begin + n % tiles) * BS_KT + rs * 32;      // first streamed row of this wavefront's block
            Split8 na, nb;                                               // the next tile's values, parts of this thread's
            BsTile::State sa, sb;
            // piece k of 24 of splitting them
            auto split_next = [&](int k) __attribute__((always_inline)) {
                if (k < 12) {
                    if (!EXACT) top_a = xa.largest_step(k, top_a);
                    xa.template split_step<EXACT>(k, sa, na);
                } else {
                    if (!EXACT) top_b = xb.largest_step(k - 12, top_b);
                    xb.template split_step<EXACT>(k - 12, sb, nb);
                }
            };
            // (EXACT: a block that the mask hides is left out, like those that the causal flag hides: its rows may hold anything)
            bool seen = i0 < w_end && i0 + 32 > w_first && i0 < n_stream;
            if (EXACT && DENSE && p.mask_flags && seen) {
                const int own32 = (o0 >> 5) + own, row32 = KEYS ? i0 >> 5 : own32, key32 = KEYS ? own32 : i0 >> 5;
                seen = mask_flags_of(p, b, KEYS ? hkv * p.G + n / tiles : hq)[(int64_t)row32 * ((Skv + 31) >> 5) + key32] != 2;
            }
            if (seen) {      // (uniform)
                [[maybe_unused]] float mv[16];
                if (DENSE) {
                    if (KEYS) {
                        // (a lane owns a key: down its column of the mask; rows past the last read zeros)
                        const int h = hkv * p.G + n / tiles;
                        const float* mc = (const float*)p.mask + (int64_t)b * p.m_sb + (int64_t)h * p.m_sh + (int64_t)i0 * p.m_si;
                        const int64_t left = ((int64_t)(Sq - 1 - i0) * p.m_si + (int64_t)(Skv - 1) * p.m_sj + 1) * 4;
                        const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc((void*)mc, 0, (int)min(left, (int64_t)0x7fffffff), 0x00020000);
                        const int at = (int)(((int64_t)min(mine, Skv - 1) * p.m_sj + (int64_t)(4 * g) * p.m_si) * 4), row4 = (int)(p.m_si * 4);
#pragma unroll
                        for (int r = 0; r < 16; ++r) mv[r] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rsrc, at, (8 * (r / 4) + (r % 4)) * row4, 0));
                    } else {
                        // (padding rows may hold anything, what starts EXACT among it: the last row in their place, as in Q' and dO)
                        const float* mrow = (const float*)p.mask + (int64_t)b * p.m_sb + (int64_t)hq * p.m_sh + (int64_t)min(mine, rows_b - 1) * p.m_si;
                        const bool vec = p.m_sj == 1 && ((p.m_sb | p.m_sh | p.m_si) & 3) == 0 && (reinterpret_cast<uintptr_t>(p.mask) & 15u) == 0;
                        if (vec && i0 + 32 <= Skv) {
#pragma unroll
                            for (int r4 = 0; r4 < 4; ++r4) {
                                const float4v w = *(const float4v*)(mrow + i0 + 8 * r4 + 4 * g);
#pragma unroll
                                for (int e = 0; e < 4; ++e) mv[4 * r4 + e] = w[e];
                            }
                        } else {
#pragma unroll
                            for (int r = 0; r < 16; ++r) mv[r] = mrow[(int64_t)min(i0 + 8 * (r / 4) + 4 * g + r % 4, Skv - 1) * p.m_sj];
                        }
                    }
                }
                // register r is streamed row i0 + 8 (r / 4) + 4 g + r % 4
                floatx16 s, dp;
                // (what a product starts with is read while the one before ends)
                Split8 first_a = BsTile::rows_operand(tile_a + row_base), first_o = BsOwn::rows_operand(own_x + own_base);
                // c = (32 rows of a tile) (owned rows)^T, `between(i)` behind each of its 24 instructions; operands are read a step ahead.  (The five
                // smaller products of all steps, then the leading ones: the sum is rounded at its own size four times)
                auto rows_product = [&](floatx16& c, const char* tile, const char* owned, auto between, auto ahead) __attribute__((always_inline)) {
#pragma unroll
                    for (int r = 0; r < 16; ++r) c[r] = 0.0f;
                    Split8 a = first_a, o = first_o;
                    uint4p lead_a[4], lead_o[4];
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        Split8 a1 = a, o1 = o;
                        if (i + 1 < 4) {
                            a1 = BsTile::rows_operand(tile + (row_base ^ ((i + 1) << 5)));
                            o1 = BsOwn::rows_operand(owned + (own_base ^ ((i + 1) << 5)));
                        }
                        __builtin_amdgcn_sched_barrier(0);
                        lead_a[i] = a.h;
                        lead_o[i] = o.h;
                        if (EXACT) c = mma_split<true>(a, o, c);
                        mma_split_term<EXACT, 0>(a, o, c); between(5 * i);
                        mma_split_term<EXACT, 1>(a, o, c); between(5 * i + 1);
                        mma_split_term<EXACT, 2>(a, o, c); between(5 * i + 2);
                        mma_split_term<EXACT, 3>(a, o, c); between(5 * i + 3);
                        mma_split_term<EXACT, 4>(a, o, c); between(5 * i + 4);
                        a = a1;
                        o = o1;
                    }
                    ahead();
                    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        a.h = lead_a[i];
                        o.h = lead_o[i];
                        if (!EXACT) mma_split_term<EXACT, 5>(a, o, c);
                        between(20 + i);
                    }
                };
                // c[0 .. 1] += (tile's columns) (16 rows of each half h in x[h]), the halves one behind the other
                auto cols_product = [&](floatx16* c, const char* tile, const Split8 (&x)[2], auto between, auto ahead) __attribute__((always_inline)) {
                    Split8 a = first_a;
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        const int h = i / 2, db = i % 2, hn = (i + 1) / 2, dn = (i + 1) % 2;
                        Split8 a1 = a;
                        if (i + 1 < 4) a1 = BsTile::cols_operand(tile + hn * 16 * L::ROWB, col_addr[dn][0], col_addr[dn][1]);
                        else ahead();
                        __builtin_amdgcn_sched_barrier(0);
                        mma_split_term<EXACT, 0>(a, x[h], c[db]); between(6 * i);
                        mma_split_term<EXACT, 1>(a, x[h], c[db]); between(6 * i + 1);
                        mma_split_term<EXACT, 2>(a, x[h], c[db]); between(6 * i + 2);
                        mma_split_term<EXACT, 3>(a, x[h], c[db]); between(6 * i + 3);
                        mma_split_term<EXACT, 4>(a, x[h], c[db]); between(6 * i + 4);
                        mma_split_term<EXACT, 5>(a, x[h], c[db]); between(6 * i + 5);
                        a = a1;
                    }
                };
                auto fenced = [](auto f) { return [=](int i) __attribute__((always_inline)) { __builtin_amdgcn_sched_barrier(0); f(i); __builtin_amdgcn_sched_barrier(0); }; };
                rows_product(s, tile_a, own_x, [](int) {}, [&]() __attribute__((always_inline)) {
                    first_a = BsTile::rows_operand(tile_b + row_base);
                    first_o = BsOwn::rows_operand(own_y + own_base);
                });
                // (-L log2 e and -D of the rows: a lane's own, or of its registers' rows)
                auto add_stats = [&](floatx16& c, int which, float mine) __attribute__((always_inline)) {
#pragma unroll
                    for (int r4 = 0; r4 < 4; ++r4) {
                        float4v a = {mine, mine, mine, mine};
                        if (KEYS) a = *(const float4v*)&s_stats[which][rs * 32 + 8 * r4 + 4 * g];
#pragma unroll
                        for (int e = 0; e < 4; ++e) c[4 * r4 + e] += a[e];
                    }
                };
                add_stats(s, 0, seed_s);
                if (DENSE) {
#pragma unroll
                    for (int r = 0; r < 16; ++r) s[r] = __builtin_fmaf(mv[r], LOG2E, s[r]);
                }
                if (i0 < w_all || i0 + 32 > w_all_end) {      // (uniform) some pair of the block is hidden
                    asm volatile("");
                    const int lo = lane_lo - i0 - 4 * g, hi = lane_hi - i0 - 4 * g;
#pragma unroll
                    for (int r = 0; r < 16; ++r)
                        if (8 * (r / 4) + (r % 4) < lo || 8 * (r / 4) + (r % 4) >= hi) s[r] = -INFINITY;
                }
                // P, and for keys its parts, under dp; dS = P dp (a hidden pair has P = 0 and a finite second factor), its parts under dV or,
                // the second half of them, under the first of dQ
                Split8 pp[2], pd[2];
                SplitPair pair;
                auto soft = [&](int k) __attribute__((always_inline)) {
                    const int q = k / 3, part = k % 3, h = q / 4;
                    if (part == 0) {
                        s[2 * q] = __builtin_amdgcn_exp2f(s[2 * q]);
                        s[2 * q + 1] = __builtin_amdgcn_exp2f(s[2 * q + 1]);
                    }
                    if (!KEYS) return;
                    unsigned x = pp[h].h[q % 4], y = pp[h].m[q % 4], z = pp[h].l[q % 4];
                    if (part == 0) pair.template step<EXACT, 0>(s[2 * q], s[2 * q + 1], x, y, z);
                    else if (part == 1) pair.template step<EXACT, 1>(s[2 * q], s[2 * q + 1], x, y, z);
                    else pair.template step<EXACT, 2>(s[2 * q], s[2 * q + 1], x, y, z);
                    pp[h].h[q % 4] = x;
                    pp[h].m[q % 4] = y;
                    pp[h].l[q % 4] = z;
                };
                auto split_ds = [&](int k) __attribute__((always_inline)) {
                    const int q = k / 3, part = k % 3, h = q / 4;
                    unsigned x = pd[h].h[q % 4], y = pd[h].m[q % 4], z = pd[h].l[q % 4];
                    if (part == 0) {
                        dp[2 * q] *= s[2 * q];
                        dp[2 * q + 1] *= s[2 * q + 1];
                        pair.template step<EXACT, 0>(dp[2 * q], dp[2 * q + 1], x, y, z);
                    } else if (part == 1) pair.template step<EXACT, 1>(dp[2 * q], dp[2 * q + 1], x, y, z);
                    else pair.template step<EXACT, 2>(dp[2 * q], dp[2 * q + 1], x, y, z);
                    pd[h].h[q % 4] = x;
                    pd[h].m[q % 4] = y;
                    pd[h].l[q % 4] = z;
                };
                rows_product(dp, tile_b, own_y, fenced([&](int i) __attribute__((always_inline)) { soft(i); }),
                             [&]() __attribute__((always_inline)) { first_a = BsTile::cols_operand(KEYS ? tile_b : tile_a, col_addr[0][0], col_addr[0][1]); });
                add_stats(dp, 1, seed_d);
                if constexpr (KEYS) {
                    cols_product(acc + 2, tile_b, pp, fenced([&](int i) __attribute__((always_inline)) { split_ds(i); }),
                                 [&]() __attribute__((always_inline)) { first_a = BsTile::cols_operand(tile_a, col_addr[0][0], col_addr[0][1]); });
                    cols_product(acc, tile_a, pd, fenced([&](int i) __attribute__((always_inline)) { split_next(i); }), []() {});
                } else {
#pragma unroll
                    for (int k = 0; k < 12; ++k) split_ds(k);
                    cols_product(acc, tile_a, pd, fenced([&](int i) __attribute__((always_inline)) {
                        if (i < 12) split_ds(12 + i);
                        else {
                            split_next(2 * (i - 12));
                            split_next(2 * (i - 12) + 1);
                        }
                    }), []() {});
                }
            } else {
#pragma unroll
                for (int k = 0; k < 24; ++k) split_next(k);
            }
            lds_barrier();      // everyone is done with the tile
            if (more) {
                BsTile::store<true>(tile_a, na, tid);
                BsTile::store<true>(tile_b, nb, tid);
                put_stats();
            }
            lds_barrier();
        }
        // A result that is not finite, or one so small that what the parts lose (f32_split.h) could show.  With a, b, y the largest
        // magnitudes of A, B and Y: dp is at most 128 y b and off by 64 (y + b) units of 2^-134, P and dS by one each, A and B likewise.  Operands
        // whose products are small throughout may leave zeros and are done over as well.
        float chk = 0.0f;
        unsigned lx = ~0u, lv = ~0u;
#pragma unroll
        for (int x = 0; x < NACC; ++x)
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                chk = __builtin_fmaf(acc[x][r], 0.0f, chk);
                if (x < 2) lx = smallest(lx, acc[x][r]);
                else lv = smallest(lv, acc[x][r]);
            }
        const bool bad = __builtin_amdgcn_ballot_w64(chk != 0.0f) != 0;
        const unsigned w_a = wave_extreme<true>(__float_as_uint(top_a)), w_b = wave_extreme<true>(__float_as_uint(top_b));
        const unsigned w_x = wave_extreme<false>(lx), w_v = wave_extreme<false>(lv);
        if (lane == 0) {
            s_vote[0][wave] = bad ? 1 : 0;
            s_vote[1][wave] = (int)w_a;
            s_vote[2][wave] = (int)w_b;
            s_vote[3][wave] = (int)w_x;
            s_vote[4][wave] = (int)w_v;
        }
        lds_barrier();
        auto over_waves = [&](int i, auto take) __attribute__((always_inline)) {
            unsigned v = (unsigned)s_vote[i][0];
#pragma unroll
            for (int w = 1; w < 8; ++w) v = take(v, (unsigned)s_vote[i][w]);
            return (unsigned)__builtin_amdgcn_readfirstlane((int)v);
        };
        auto most = [](unsigned x, unsigned y) { return max(x, y); };
        auto least = [](unsigned x, unsigned y) { return min(x, y); };
        const unsigned any_bad = over_waves(0, most), low_x = over_waves(3, least), low_v = over_waves(4, least);
        const float big_a = __uint_as_float(over_waves(1, most)), big_b = __uint_as_float(over_waves(2, most)), big_y = __uint_as_float(over_waves(5, most));
        lds_barrier();
        const float lost = SPLIT_LOST * (float)n_tiles * BS_KT, yb = big_y * big_b;
        const float bound_x = lost * (big_a * (128.0f * yb + 64.0f * (big_y + big_b) + 1.0f) + 128.0f * yb), bound_v = lost * (big_b + 1.0f);
        const bool tiny = big_a > 0.0f && big_b > 0.0f && big_y > 0.0f && (big_b < SPLIT_TINY || yb < SPLIT_TINY || yb * big_a < SPLIT_TINY);
        return any_bad != 0 || !(big_a < INFINITY) || !(big_b < INFINITY) || tiny || low_x < smallest_of(bound_x) || low_v < smallest_of(bound_v);      // (uniform)
    };
    if (n_tiles > 0) {
        if (walk(std::integral_constant<bool, false>{})) walk(std::integral_constant<bool, true>{});      // (f32_split.h)
    } else {
#pragma unroll
        for (int x = 0; x < NACC; ++x)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[x][r] = 0.0f;
    }

    // ---- the two wavefronts of a block: each adds and stores half of the registers (units of four: 32 columns are four units) ----
    constexpr int NU = NACC * 4;
    float4v* const red = (float4v*)smem;      // (everyone is past the last tile)
#pragma unroll
    for (int u = 0; u < NU; ++u) red[(wave * NU + u) * 64 + lane] = float4v{acc[u / 4][u % 4 * 4], acc[u / 4][u % 4 * 4 + 1], acc[u / 4][u % 4 * 4 + 2], acc[u / 4][u % 4 * 4 + 3]};
    lds_barrier();
    if (mine < n_all_own) {
        float* const xrow = KEYS ? (float*)bp.d_k + (int64_t)b * bp.dk_sb + (int64_t)hkv * bp.dk_sh + (int64_t)mine * bp.dk_ss
                                 : (float*)bp.d_q + (int64_t)b * bp.dq_sb + (int64_t)hq * bp.dq_sh + (int64_t)mine * bp.dq_ss;
        float* const vrow = KEYS ? (float*)bp.d_v + (int64_t)b * bp.dv_sb + (int64_t)hkv * bp.dv_sh + (int64_t)mine * bp.dv_ss : nullptr;
        const bool live = mine < n_own;      // (padding rows and keys past the count get zeros)
#pragma unroll
        for (int x = 0; x < NU / 2; ++x) {
            const int u = 2 * x + rs, c = (u % 8) * 8 + g * 4;
            const bool is_v = x >= 4;
            float4v w = red[(own * NU + u) * 64 + lane] + red[((own + 4) * NU + u) * 64 + lane];
#pragma unroll
            for (int e = 0; e < 4; ++e) w[e] = live ? (is_v ? w[e] : w[e] * p.scale) : 0.0f;
            if (c < (is_v ? p.Dv : p.D)) *(float4v*)((is_v ? vrow : xrow) + c) = w;
        }
    }
#endif
}

// One list: the dK/dV items, which are the longer ones, then the dQ items; a launch takes those from `first` on.
template <bool DENSE> __global__ __launch_bounds__(BS_THREADS, 2) void bwd_f32_split_kernel(SdpaBwdParams bp, int n_dkv, int first)
{
#if defined(__HIP_DEVICE_COMPILE__)
    __shared__ __attribute__((aligned(1024))) char smem[BS_LDS];
    __shared__ __attribute__((aligned(16))) float s_stats[2][BS_KT];
    __shared__ int s_vote[6][8];
    const int id = first + blockIdx.x;
    if (id < n_dkv) bwd_f32_split_body<true, DENSE>(bp, smem, s_stats, s_vote, id);
    else bwd_f32_split_body<false, DENSE>(bp, smem, s_stats, s_vote, id - n_dkv);
#endif
}

// Host has validated what sdpa_bwd_f32.hip asks for, D and Dv <= 64, and the row statistics are written.
hipError_t launch_sdpa_bwd_f32_split(const SdpaBwdParams& bp0, hipStream_t stream)
{
    SdpaBwdParams bp = bp0;
    SdpaParams& p = bp.f;
    const int nqb = (p.Sq + BS_OWN - 1) / BS_OWN, nkb = (p.Skv + BS_OWN - 1) / BS_OWN;
    const int64_t n_dq = (int64_t)nqb * p.Hq * p.B, n_dkv = (int64_t)nkb * p.Hkv * p.B;
    work_order(p, 1, nqb);
    if (n_dkv + n_dq > 0x7fffffffLL) return hipErrorInvalidValue;
    hipError_t e = hipSuccess;
    for (int64_t first = 0; first < n_dkv + n_dq && e == hipSuccess; first += max_blocks(BS_THREADS)) {
        const dim3 grid((unsigned)min(n_dkv + n_dq - first, max_blocks(BS_THREADS)));
        if (p.mask) hipLaunchKernelGGL(bwd_f32_split_kernel<true>, grid, dim3(BS_THREADS), 0, stream, bp, (int)n_dkv, (int)first);
        else hipLaunchKernelGGL(bwd_f32_split_kernel<false>, grid, dim3(BS_THREADS), 0, stream, bp, (int)n_dkv, (int)first);
        e = hipGetLastError();
    }
    return e;
}

}  // namespace incin_rocm
