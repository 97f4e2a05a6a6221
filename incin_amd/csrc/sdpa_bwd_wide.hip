// bf16 / f16 attention backward on the gfx950 matrix cores for head dimensions above 128 (up to 256, D and Dv in whole 16-byte
// vectors, zero-padded into the 256 instance on the way into LDS and registers): dQ, dK, dV of O = softmax(Q K^T s + mask) V with a
// causal flag, key and query counts and grouped queries.  The formulas are those of sdpa_bwd_mfma.hip; a dense mask tensor at
// these head dimensions stays with sdpa_bwd_generic.hip.
//
// What bounds it is the matrix pipe, and what shapes it are the registers: at 256 elements the two rows that a lane owns (Q and
// dO for dQ, K and V for dK) take 128 of them and one gradient's 32 x 256 block of accumulators 128 more, which is all that two
// wavefronts per SIMD have.  So a workgroup computes 128 rows of ONE gradient, and the launch's items are the blocks of all three:
//
//             owns (a lane: one)   streams            products per 32 x 32 block (16 matrix instructions each)
//   dQ item   query: Q, dO         K, V tiles         S^T = K Q^T    dP^T = V dO^T    dQ^T += K^T dS^T  (twice: see below)
//   dK item   key:   K, V          Q, dO tiles        S = Q K^T      dP = dO V^T      dK^T += Q^T dS    (twice)
//   dV item   key:   K             Q, dO tiles        S = Q K^T                       dV^T += dO^T P    (twice)
//
// one code for all three: the streamed tensors' rows are the A operands of the first two products (16-byte LDS reads), the owned
// rows the B operands, and the accumulator layout they leave is the B-operand layout of the third, whose A operand is a
// streamed tile again, through the transposing LDS read.  S is computed three times and dP twice (a dK + dV item would need 256
// accumulators).  A pair of wavefronts shares 32 owned rows: one computes S, the other dP (dV: S over half the head dimension
// each), they exchange half of either through LDS, each makes P and dS of 16 of the tile's 32 rows, they exchange those, and each
// accumulates the third product for its half of the columns: 64 registers of owned rows and 64 accumulators, 240 in all.
// (Without the pairs - a wavefront alone on its SIMD with 461 registers, half of them accumulation registers - nothing covers a
// wavefront's LDS latencies and vector work: 144 us for the backward of 2 x 16 / 8 heads x 1024, causal, against 133.)
//
// P and dS enter the third product as two 16-bit values each - the rounded value and what the rounding left - through two matrix
// instructions that share one LDS operand, so that such a call keeps the precision of f32 arithmetic (sdpa_bwd_generic.hip), for
// 176 matrix instructions per block over the three items instead of 128.  bf16 leaves 16 significant bits of them whatever their size:
// gradients 1.7 - 1.9e-3 off the float64 result in the 2-norm, as with f32 arithmetic, which is the rounding of the gradients
// themselves (with P and dS rounded once: 3e-3).  f16 ends at 65504 above and at steps of 2^-24 below, so there they are split times
// a power of two of the owned row's own, which follows the largest value the row has met (k_acc below): 22 bits of the largest, 2^-36 of it
// for the others, no overflow.  Off the float64 result in the 2-norm, dQ, unscaled / so / f32 arithmetic: 8192 positions, dO of 1e-2
// 5.7e-4 / 2.1e-4 / 2.1e-4, of 1e-3 5.4e-3 / 9.4e-4 / 9.4e-4 (subnormal gradients); and a dS beyond 65504 was a NaN in its row.  It costs
// f16 2 - 4 % of the call (2 x 16 on 8 x 1024, causal 136 -> 138 us, 8 on 1 x 4096 520 -> 536).
//
// Tiles of 32 rows (16 KiB each of both tensors), three stages: t - 1 and t in use, t + 1 arriving by global -> LDS copies.  A
// step is the first products of tile t, a barrier, and the third product of tile t - 1 with the exponentials and splits of
// tile t between its matrix instructions.  The copies of tile t + 1 are started behind the first LDS reads of tile t, and the first
// operands of the third product are read before the barrier, with the last first products: neither then waits behind a barrier
// (2 x 16 on 8 x 1024 causal 128.5 -> 126 us, nothing masked 234 -> 229, 8 x 2048 123.5 -> 119.5, 4 x 3000 at D = 160 161 -> 158).
//
// Measured, backward call, bf16: 2 x 16 heads on 8 x 1024 positions, D = 256, causal 13.86 -> 0.14 ms (302 TFLOP/s of
// useful work; the generic kernels 3.1), 8 on 1 x 4096 0.48 ms, 4 x 16 on 4 x 1024 0.25 ms.  That causal launch is bound by its longest item: the
// dK block of the first keys, 64 tiles of four products, is 1.45 times a compute unit's share of the whole.  Where items are equal (nothing
// masked) the matrix pipes are busy 45 % of the time a workgroup is on a compute unit, and beside them the LDS is the bound - in the first products every
// matrix instruction takes 1 KiB of it, 128 bytes a clock over the four SIMDs.  With parts left out (2 x 16 on 8 x 1024, nothing masked, 229 us): no
// copies 210, no exponentials and splits 209, neither 191.
#include <type_traits>

// (three bodies in one kernel spill scalar registers, copy descriptors among them: their copies take the five wait states)
#define INCIN_DMA_WAIT "s_nop 4"
#include "sdpa_bwd.h"
#include "sdpa_mfma_common.h"

namespace incin_rocm {

constexpr int BW_D = 256;
constexpr int BW_ROWS = 128;                                    // rows of a gradient per workgroup
constexpr int BW_KT = 32;                                       // rows per streamed tile
constexpr int BW_TILE = BW_KT * BW_D * 2;                       // 16 KiB
constexpr int BW_STAGE = 2 * BW_TILE + 512;                     // both tensors' tiles; 32 x -L_i log2(e), 32 x -D_i (64 floats arrive)
constexpr int BW_PAIR = 8192 + 512;                             // a pair's exchange area: 8 KiB of values, two exponents per owned row
constexpr int BW_XCHG = 4 * BW_PAIR;
constexpr int BW_TOP = 15, BW_AIM = 11, BW_LOOSE = 60;          // f16: powers of two that bound and place the split values (see bwd_wide_item)
constexpr int BW_RING = 4;                                      // LDS operands in flight ahead of their matrix instructions

enum { BW_DQ = 0, BW_DK = 1, BW_DV = 2 };

template <typename T, int ROLE>
__device__ __forceinline__ void bwd_wide_item(const SdpaBwdParams& bp, char* smem, int b, int hkv, int gq, int blk, int part, int parts)
{
    typedef typename Mma<T>::vec8 vec8;
    typedef PfLayout<BW_D> L;
    typedef float float4v __attribute__((ext_vector_type(4)));
    constexpr bool WITH_DP = ROLE != BW_DV;
    constexpr int R = BW_RING, LPW = BW_TILE / 1024 / 8;
    constexpr int NA = WITH_DP ? BW_D / 16 : BW_D / 32;      // matrix instructions (k-steps) of a wavefront's share of the first products
    constexpr int NDB = BW_D / 64;                           // 32-wide column blocks of its half of the gradient
    constexpr bool SCALED = std::is_same<T, f16_t>::value;
    const SdpaParams& p = bp.f;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int pr = wave & 3, role = wave >> 2;               // which 32 rows of the block, which wavefront of their pair
    const int ql = lane & 31, g = lane >> 5;
    const int Sq = p.Sq, Skv = p.Skv, coff = Skv - Sq;
    const int kv_len = p.kv_lens ? clampi(p.kv_lens[b], 0, Skv) : Skv;
    const int rows_b = p.q_lens ? clampi(p.q_lens[b], 0, Sq) : Sq;      // query rows at and beyond are padding
    const int own0 = blk * BW_ROWS, wave0 = own0 + pr * 32, mine = wave0 + ql;
    const int hq0 = hkv * p.G + gq;

    const T* kp = (const T*)p.k + (int64_t)b * p.k_sb + (int64_t)hkv * p.k_sh;
    const T* vp = (const T*)p.v + (int64_t)b * p.v_sb + (int64_t)hkv * p.v_sh;
    const T* qp = (const T*)p.q + (int64_t)b * p.q_sb + (int64_t)hq0 * p.q_sh;
    const T* gp = (const T*)bp.d_o + (int64_t)b * bp.do_sb + (int64_t)hq0 * bp.do_sh;

    // ---- the walk: tiles [n_lo, n_hi) of heads x tiles_per_head ------------------------------------------------------------
    // dQ: the key tiles that the block's last row sees.  dK, dV: for each query head of the group the query tiles that see the
    // block's first key; a walk may be dealt to several workgroups (part of parts), each leaving its sums in a plane.
    int t_begin = 0, tiles_per_head, heads = 1, stream_rows;
    int lim_lane = 0, edge = 0;      // dQ: this lane's key count, the pair's smallest; dK, dV: first row that sees the lane's key, that sees all keys of the pair
    if (ROLE == BW_DQ) {
        int j_end = kv_len;
        lim_lane = edge = kv_len;
        if (p.causal) {
            j_end = clampi(min(own0 + BW_ROWS - 1, rows_b - 1) + coff + 1, 0, kv_len);
            lim_lane = clampi(mine + coff + 1, 0, kv_len);
            edge = clampi(wave0 + coff + 1, 0, kv_len);
        }
        if (own0 >= rows_b) j_end = 0;
        stream_rows = kv_len;
        tiles_per_head = (j_end + BW_KT - 1) / BW_KT;
    } else {
        t_begin = p.causal ? clampi(own0 - coff, 0, Sq) / BW_KT : 0;
        lim_lane = p.causal ? mine - coff : -0x40000000;
        edge = p.causal ? max(wave0 + 31 - coff, 0) : 0;
        stream_rows = rows_b;
        heads = p.G;
        tiles_per_head = own0 < kv_len ? max((rows_b + BW_KT - 1) / BW_KT - t_begin, 0) : 0;
    }
    const int n_all = tiles_per_head * heads;
    const int n_lo = parts > 1 ? (int)((int64_t)n_all * part / parts) : 0;
    const int n_hi = parts > 1 ? (int)((int64_t)n_all * (part + 1) / parts) : n_all;

    // ---- global -> LDS copies: wavefront-wide load wave * LPW + c fills bytes [.. * 1024, + 1024) of a tile ------------------
    const int64_t x_ss = ROLE == BW_DQ ? p.k_ss : p.q_ss, y_ss = ROLE == BW_DQ ? p.v_ss : bp.do_ss;
    int x_voff[LPW], y_voff[LPW];
#pragma unroll
    for (int c = 0; c < LPW; ++c) {
        const int pos = (wave * LPW + c) * 64 + lane;
        const int row = pos / L::CPR, slot = pos % L::CPR;
        x_voff[c] = dma_chunk_offset(row, (int)x_ss * 2, slot ^ L::fk(row), p.D * 2);
        y_voff[c] = dma_chunk_offset(row, (int)y_ss * 2, slot ^ L::fk(row), p.Dv * 2);
    }
    const unsigned lds0 = lds_address(smem);
    auto clamp31 = [](int64_t x) { return x < 0 ? 0 : (x >> 31) ? 0x7fffffff : (int)x; };
    // The copies walk the tiles with running addresses: next tile's rows of both tensors, its per-row floats, and how many bytes
    // and rows there are from there to the end (rows past stream_rows arrive as zeros).
    const int64_t x_step = (int64_t)BW_KT * x_ss * 2, y_step = (int64_t)BW_KT * y_ss * 2;
    const char *nx_x = nullptr, *nx_y = nullptr, *nx_s = nullptr;
    int64_t nx_xrem = 0, nx_yrem = 0;
    int nx_rows = 0, nx_t = 0, nx_h = 0;
    auto to_head = [&](int h, int t) __attribute__((always_inline)) {      // tile t of the group's head h
        const int row0 = (t_begin + t) * BW_KT;
        nx_x = (const char*)((ROLE == BW_DQ ? kp : qp + h * p.q_sh) + row0 * x_ss);
        nx_y = (const char*)((ROLE == BW_DQ ? vp : gp + h * bp.do_sh) + row0 * y_ss);
        nx_rows = stream_rows - row0;
        nx_xrem = (nx_rows - 1) * x_ss * 2 + p.D * 2;
        nx_yrem = (nx_rows - 1) * y_ss * 2 + p.Dv * 2;
        if (ROLE != BW_DQ) nx_s = (const char*)((wave == 0 ? bp.neg_l2 : bp.neg_delta) + ((int64_t)b * p.Hq + hq0 + h) * Sq + row0);
        nx_t = t;
        nx_h = h;
    };
    auto issue = [&](int stage) __attribute__((always_inline)) {
        const uint4v xd = dma_descriptor(nx_x, clamp31(nx_xrem)), yd = dma_descriptor(nx_y, clamp31(nx_yrem));
        const unsigned st = lds0 + stage * BW_STAGE + wave * LPW * 1024;
#pragma unroll
        for (int c = 0; c < LPW; ++c) dma_copy16(xd, st + c * 1024, x_voff[c]);
#pragma unroll
        for (int c = 0; c < LPW; ++c) dma_copy16(yd, st + BW_TILE + c * 1024, y_voff[c]);
        if (ROLE != BW_DQ && wave < (WITH_DP ? 2 : 1))      // 32 floats of -L_i log2(e) (wavefront 0) or -D_i (1)
            dma_copy4(dma_descriptor(nx_s, min(nx_rows, BW_KT) * 4), lds0 + stage * BW_STAGE + 2 * BW_TILE + wave * 256, lane * 4);
        if (++nx_t == tiles_per_head && ROLE != BW_DQ) {
            if (nx_h + 1 < heads) to_head(nx_h + 1, 0);
        } else {
            nx_x += x_step; nx_y += y_step; nx_s += BW_KT * 4;
            nx_xrem -= x_step; nx_yrem -= y_step; nx_rows -= BW_KT;
        }
    };
    static_assert(BW_STAGE >= 2 * BW_TILE + 512, "two arrays of 64 floats");

    // ---- the owned rows, as B operands: lane (ql, g) holds elements 16 s + 8 g .. + 7 of its row per k-step s ---------------
    // Role 0 of a pair holds the rows of the first product (Q or K), role 1 those of the second (dO or V); a dV item has only the
    // first, of which each holds half the k-steps.  (Through 4 KiB per wavefront of the third stage, which nothing is copied
    // into before the loop's first barrier.)
    if (n_lo < n_hi) {
        to_head(n_lo / tiles_per_head, n_lo % tiles_per_head);
        issue(0);
    }
    vec8 own[NA];
    {
        const bool second = WITH_DP && role == 1;
        const T* op = ROLE == BW_DQ ? (second ? gp : qp) : (second ? vp : kp);
        const int64_t o_ss = ROLE == BW_DQ ? (second ? bp.do_ss : p.q_ss) : (second ? p.v_ss : p.k_ss);
        const int c0 = WITH_DP ? 0 : role * (BW_D / 2);      // first column
        uint4v raw[NA / 4][4];
        fetch_q_rows(raw, op + c0, wave0, ROLE == BW_DQ ? Sq : Skv, o_ss, (second ? p.Dv : p.D) - c0, lane);
        stage_q_rows(own, raw, smem + 2 * BW_STAGE + wave * 4096, lane);
    }
    const float c2 = p.scale * 1.4426950408889634f;
    float my_l = 0.0f, my_d = 0.0f;      // dQ: -L log2(e) and -D of the lane's query
    if (ROLE == BW_DQ) {
        const int64_t stat = ((int64_t)b * p.Hq + hq0) * Sq + min(mine, Sq - 1);
        my_l = bp.neg_l2[stat];
        my_d = bp.neg_delta[stat];
    }

    // Operand addresses.  By rows: M index ql is row ql of the tile for role 0 and row ql ^ 16 for role 1, so that either finds
    // the rows 16 role .. + 15 - its half of the pair's P and dS - in its first eight accumulator registers; chunk 2 s + g of a
    // row is at row_base ^ (s << 5).  Transposed: column block db of the wavefront's half, half h of 16 rows: tr_base[h] ^ (db << 6).
    const int row_base = (ql ^ (role << 4)) * L::ROWB + (((g | (WITH_DP ? 0 : role << 4)) ^ L::fk(ql)) << 4) + (WITH_DP && role ? BW_TILE : 0);
    int tr_base[2];
    {
        const int n = lane & 15, dh = (lane >> 4) & 1;
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const int r = 8 * h + 4 * g + (n >> 2), chunk = role * 16 + 2 * dh + ((n & 3) >> 1);
            tr_base[h] = r * L::ROWB + ((chunk ^ L::fk(r)) << 4) + (n & 1) * 8 + (ROLE == BW_DV ? BW_TILE : 0);
        }
    }
    // Exchange areas of the pair: what a role sends of its first products (8 floats per lane), and its half of dS (dV: P) as two
    // operands of 16 bytes per lane.
    char* const x1 = smem + 3 * BW_STAGE + pr * BW_PAIR + lane * 16;
    char* const x2 = x1 + 4096;
    [[maybe_unused]] int* const x3 = (int*)(smem + 3 * BW_STAGE + pr * BW_PAIR + 8192) + lane;      // f16: what power of two a role's half is times

    floatx16 acc[NDB];
#pragma unroll
    for (int db = 0; db < NDB; ++db)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[db][r] = 0.0f;

    vec8 w_hi, w_lo;      // this role's half of dS (dV: P) of the previous tile: the rounded value and the rest
    // f16: the lane's owned row, and with it its column of the third product, has a power of two of its own.  k_acc: the accumulators
    // are the sums times 2^k_acc, and the next tile is split times that; k_w: w_hi and w_lo are times 2^k_w <= 2^k_acc.  It starts
    // so high that what it leaves unsplit is nothing, and comes down to where a tile's largest value is 2^BW_AIM whenever one
    // passes 2^BW_TOP: the largest has its 22 bits, all others of the row 2^-36 of it, and nothing overflows.
    [[maybe_unused]] int k_acc = BW_LOOSE, k_w = BW_LOOSE;
    // One tile: the first products of tile t, whose eight registers that the partner needs go to the exchange area; a barrier;
    // the third product of tile t - 1 with P and dS of tile t made between its matrix instructions.
    auto step = [&](const char* st, const char* pst, int r0, auto copies, auto WITH_A_, auto WITH_B_) __attribute__((always_inline)) {
        constexpr bool WITH_A = decltype(WITH_A_)::value, WITH_B = decltype(WITH_B_)::value;
        floatx16 f;
        vec8 o_hi, o_lo;
        [[maybe_unused]] int k_o = 0;
        auto read_partner = [&]() __attribute__((always_inline)) {      // the partner's half of tile t - 1's dS
            if constexpr (WITH_B) {
                o_hi = *(const vec8*)(x2 + (1 - role) * 2048);
                o_lo = *(const vec8*)(x2 + (1 - role) * 2048 + 1024);
                if constexpr (SCALED) k_o = x3[(1 - role) * 64];
            }
        };
        float4v nl[2], nd[2];
        vec8 bring[R];
        auto fetch_b = [&](int m) __attribute__((always_inline)) {      // m: column block m % NDB, rows 16 (role ^ (m / NDB)) .. + 15: the own half first
            const char* tt = pst + (role ^ (m / NDB)) * 16 * L::ROWB;
            short8v av;
            av.lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((short4v __attribute__((address_space(3)))*)(tt + (tr_base[0] ^ ((m % NDB) << 6))));
            av.hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((short4v __attribute__((address_space(3)))*)(tt + (tr_base[1] ^ ((m % NDB) << 6))));
            bring[m % R] = __builtin_bit_cast(vec8, av);
        };
        if constexpr (WITH_A) {
#pragma unroll
            for (int r = 0; r < 16; ++r) f[r] = 0.0f;
            vec8 ring[R];
            auto fetch = [&](int i) __attribute__((always_inline)) { ring[i % R] = *(const vec8*)(st + (row_base ^ (i << 5))); };
#pragma unroll
            for (int i = 0; i < R; ++i) fetch(i);
            read_partner();
            __builtin_amdgcn_sched_barrier(0);
            copies();      // (behind the first reads: their latency covers what starting copies takes)
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int i = 0; i < NA; ++i) {
                f = Mma<T>::run(ring[i % R], own[i], f);
                if (i + R < NA) fetch(i + R);
                else if (WITH_B) fetch_b(i + R - NA);      // (the third product's first operands are there when the barrier opens)
                __builtin_amdgcn_sched_barrier(0);      // (the scheduler would put every read right in front of its matrix instruction)
            }
            // -L_i log2(e) and -D_i of the 16 rows this role makes P and dS of: register r is streamed row r0 + 16 role + 8 (r / 4) + 4 g + r % 4
#pragma unroll
            for (int r4 = 0; r4 < 2; ++r4) {
                if (ROLE == BW_DQ) {
                    nl[r4] = float4v{my_l, my_l, my_l, my_l};
                    nd[r4] = float4v{my_d, my_d, my_d, my_d};
                } else {
                    nl[r4] = *(const float4v*)(st + 2 * BW_TILE + (16 * role + 8 * r4 + 4 * g) * 4);
                    if (WITH_DP) nd[r4] = *(const float4v*)(st + 2 * BW_TILE + 256 + (16 * role + 8 * r4 + 4 * g) * 4);
                }
            }
            // (what the mask hides ends as P = 0)
            if (ROLE == BW_DQ ? r0 + BW_KT > edge : r0 < edge) {
                asm volatile("" ::: "memory");      // (a real branch)
                const int rel = lim_lane - r0 - 16 * role - 4 * g;
#pragma unroll
                for (int r = 0; r < 8; ++r) {
                    const int row = 8 * (r / 4) + (r % 4);
                    if (ROLE == BW_DQ ? row >= rel : row < rel) nl[r / 4][r % 4] = -INFINITY;
                }
            }
            *(float4v*)(x1 + role * 2048) = float4v{f[8], f[9], f[10], f[11]};
            *(float4v*)(x1 + role * 2048 + 1024) = float4v{f[12], f[13], f[14], f[15]};
            __syncthreads();
        } else {
            read_partner();
#pragma unroll
            for (int m = 0; m < R; ++m) fetch_b(m);
        }
        if constexpr (WITH_B && SCALED) {
            const int k = min(k_w, k_o);
            if (__builtin_amdgcn_ballot_w64(k_w != k_acc || k_o != k_acc)) {      // (rare: a row's largest value so far grew eightfold or more)
                auto shift = [](vec8& v, int d) __attribute__((always_inline)) {
#pragma unroll
                    for (int e = 0; e < 8; ++e) v[e] = (T)__builtin_ldexpf((float)v[e], d);
                };
                shift(w_hi, k - k_w);
                shift(w_lo, k - k_w);
                shift(o_hi, k - k_o);
                shift(o_lo, k - k_o);
#pragma unroll
                for (int db = 0; db < NDB; ++db)
#pragma unroll
                    for (int r = 0; r < 16; ++r) acc[db][r] = __builtin_ldexpf(acc[db][r], k - k_acc);
                k_acc = k;
            }
        }
        float4v other[2];
        if constexpr (WITH_A) {
            other[0] = *(const float4v*)(x1 + (1 - role) * 2048);
            other[1] = *(const float4v*)(x1 + (1 - role) * 2048 + 1024);
        }
        vec8 n_hi, n_lo;
        auto split = [&](int r, float x) __attribute__((always_inline)) {
            const T hi = (T)x;
            n_hi[r] = hi;
            n_lo[r] = (T)(x - (float)hi);
        };
        [[maybe_unused]] const float two_k = __builtin_bit_cast(float, (127 + k_acc) << 23);
        auto soft = [&](int r) __attribute__((always_inline)) {
            if constexpr (WITH_A) {
                const float a = f[r], o = other[r / 4][r % 4];
                float x;
                if constexpr (WITH_DP) {
                    const float s = role ? o : a, d = role ? a : o;
                    x = __builtin_amdgcn_exp2f(__builtin_fmaf(s, c2, nl[r / 4][r % 4])) * (d + nd[r / 4][r % 4]);
                } else
                    x = __builtin_amdgcn_exp2f(__builtin_fmaf(a + o, c2, nl[r / 4][r % 4]));
                if constexpr (SCALED) {
                    f[r] = x;
                    split(r, x * two_k);
                } else
                    split(r, x);
            }
        };
        if constexpr (WITH_B) {
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int m = 0; m < 2 * NDB; ++m) {
                acc[m % NDB] = Mma<T>::run(bring[m % R], m < NDB ? w_hi : o_hi, acc[m % NDB]);
                acc[m % NDB] = Mma<T>::run(bring[m % R], m < NDB ? w_lo : o_lo, acc[m % NDB]);
                if (m + R < 2 * NDB) fetch_b(m + R);
                soft(m);
                __builtin_amdgcn_sched_barrier(0);      // (likewise: the vector work would gather behind the matrix instructions)
            }
        } else {
#pragma unroll
            for (int r = 0; r < 8; ++r) soft(r);
        }
        if constexpr (WITH_A && SCALED) {
            k_w = k_acc;
            float top = 0.0f;
#pragma unroll
            for (int r = 0; r < 8; ++r) top = fmaxf(top, fabsf(f[r]));
            constexpr float LIMIT = 1 << BW_TOP;
            if (__builtin_amdgcn_ballot_w64(top * two_k > LIMIT)) {
                top = xor32_max(top);      // (the other half of the row's values)
                if (top * two_k > LIMIT) k_w = BW_AIM + 127 - (__builtin_bit_cast(int, top) >> 23);
                const float two_w = __builtin_bit_cast(float, (127 + k_w) << 23);
#pragma unroll
                for (int r = 0; r < 8; ++r) split(r, f[r] * two_w);
            }
            x3[role * 64] = k_w;
        }
        if constexpr (WITH_A) {      // (the partner has read tile t - 1's before this step's barrier)
            w_hi = n_hi;
            w_lo = n_lo;
            *(vec8*)(x2 + role * 2048) = n_hi;
            *(vec8*)(x2 + role * 2048 + 1024) = n_lo;
        }
    };

    // Tile n has landed for everyone, tile n - 1's dS is in the exchange area, and everyone is done with tile n - 2: its stage is
    // free for tile n + 1.  Every wavefront computes every tile (one that sees nothing of it would wait at the next barrier for
    // the others anyway).  (The first tile's step, which has no third product, is code of its own: a branch inside the loop makes
    // the compiler move the accumulators around it.)
    int stage = 0, pstage = 0, n = n_lo, r0 = (t_begin + (tiles_per_head > 0 ? n_lo % tiles_per_head : 0)) * BW_KT;
    const int r_end = (t_begin + tiles_per_head) * BW_KT;
    auto next_tile = [&]() __attribute__((always_inline)) {
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
        const int nstage = stage == 2 ? 0 : stage + 1;
        return nstage;
    };
    auto advance = [&](int nstage) __attribute__((always_inline)) {
        pstage = stage;
        stage = nstage;
        r0 = r0 + BW_KT >= r_end ? t_begin * BW_KT : r0 + BW_KT;      // (then: the group's next head)
        ++n;
    };
    if (n_lo < n_hi) {
        const int first = next_tile();
        step(smem, smem, r0, [&]() __attribute__((always_inline)) { if (n + 1 < n_hi) issue(first); }, std::true_type{}, std::false_type{});
        advance(first);
        while (n < n_hi) {
            const int nstage = next_tile();
            step(smem + stage * BW_STAGE, smem + pstage * BW_STAGE, r0, [&]() __attribute__((always_inline)) { if (n + 1 < n_hi) issue(nstage); }, std::true_type{}, std::true_type{});
            advance(nstage);
        }
        __syncthreads();      // (the last tile's dS)
        step(smem, smem + pstage * BW_STAGE, 0, []() {}, std::false_type{}, std::true_type{});
    }

    // ---- out: this role's half of the columns -----------------------------------------------------------------------------------
    const float unit = ROLE == BW_DV ? 1.0f : p.scale, out_scale = SCALED ? __builtin_ldexpf(unit, -k_acc) : unit;
    const int width = ROLE == BW_DV ? p.Dv : p.D, c0 = role * (BW_D / 2);
    if (mine >= (ROLE == BW_DQ ? rows_b : kv_len)) {      // padding rows and keys past the count: zeros
#pragma unroll
        for (int db = 0; db < NDB; ++db)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[db][r] = 0.0f;
    }
    if (ROLE != BW_DQ && parts > 1) {
        if (mine < Skv) {
            float* row = (ROLE == BW_DK ? bp.part_dk : bp.part_dv) + ((((int64_t)part * p.B + b) * p.Hkv + hkv) * Skv + mine) * width;
#pragma unroll
            for (int db = 0; db < NDB; ++db)
#pragma unroll
                for (int r4 = 0; r4 < 4; ++r4) {
                    const int col = c0 + db * 32 + r4 * 8 + g * 4;
                    float4v w;
#pragma unroll
                    for (int e = 0; e < 4; ++e) w[e] = acc[db][r4 * 4 + e] * out_scale;
                    if (col < width) *(float4v*)(row + col) = w;
                }
        }
        return;
    }
    // (staged through LDS of the stage after the last one: nobody reads it any more, nothing is copied into it)
    T* out = ROLE == BW_DQ ? (T*)bp.d_q + (int64_t)b * bp.dq_sb + (int64_t)hq0 * bp.dq_sh
             : ROLE == BW_DK ? (T*)bp.d_k + (int64_t)b * bp.dk_sb + (int64_t)hkv * bp.dk_sh
                             : (T*)bp.d_v + (int64_t)b * bp.dv_sb + (int64_t)hkv * bp.dv_sh;
    store_o_rows(acc, out_scale, smem + stage * BW_STAGE + wave * 4096, out + c0, wave0, ROLE == BW_DQ ? Sq : Skv,
                 ROLE == BW_DQ ? bp.dq_ss : ROLE == BW_DK ? bp.dk_ss : bp.dv_ss, width - c0, lane);
}

// The items, longest first (under a causal mask the last query block and the first key block): rank r holds the r-th longest
// blocks of every head - dK and dV blocks of all (batch, KV head) pairs, then dQ blocks of all heads, the pairs innermost, so that
// with a multiple of 8 pairs one XCD has all items of a pair.
template <typename T>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2, 2))) void sdpa_bwd_wide_kernel(SdpaBwdParams bp, int first)
{
#if defined(__HIP_DEVICE_COMPILE__)
    __shared__ __attribute__((aligned(1024))) char smem[3 * BW_STAGE + BW_XCHG];
    const SdpaParams& p = bp.f;
    const int nqb = (p.Sq + BW_ROWS - 1) / BW_ROWS, nkb = (p.Skv + BW_ROWS - 1) / BW_ROWS;
    const int pairs = p.B * p.Hkv, parts = bp.parts_kv;
    const int kv_items = 2 * parts * pairs, q_items = p.G * pairs, both = min(nqb, nkb);
    int id = first + (int)blockIdx.x, rank;
    bool kv;
    if (id < both * (kv_items + q_items)) {
        rank = id / (kv_items + q_items);
        id -= rank * (kv_items + q_items);
        kv = id < kv_items;
        if (!kv) id -= kv_items;
    } else {
        id -= both * (kv_items + q_items);
        kv = nkb > nqb;
        rank = both + id / (kv ? kv_items : q_items);
        id %= kv ? kv_items : q_items;
    }
    const int pair = id % pairs, sub = id / pairs;
    const int b = pair / p.Hkv, hkv = pair % p.Hkv;
    if (!kv) bwd_wide_item<T, BW_DQ>(bp, smem, b, hkv, sub, nqb - 1 - rank, 0, 1);
    else if (sub < parts) bwd_wide_item<T, BW_DK>(bp, smem, b, hkv, 0, rank, sub, parts);
    else bwd_wide_item<T, BW_DV>(bp, smem, b, hkv, 0, rank, sub - parts, parts);
#endif
}

// Host has validated: dtype f16 / bf16, 128 < max(D, Dv) <= 256 in whole 16-byte vectors, no dense mask, finite scale, unit last-axis
// strides, 16-byte aligned rows, row strides below 2^24 elements, lse and the workspace present.
hipError_t launch_sdpa_bwd_wide(const SdpaBwdParams& bp, int dtype, hipStream_t stream)
{
    const SdpaParams& p = bp.f;
    const int64_t nqb = (p.Sq + BW_ROWS - 1) / BW_ROWS, nkb = (p.Skv + BW_ROWS - 1) / BW_ROWS, pairs = (int64_t)p.B * p.Hkv;
    const int64_t total = pairs * (nqb * p.G + nkb * 2 * bp.parts_kv);
    if (total > 0x7fffffffLL) return hipErrorInvalidValue;
    hipError_t e = launch_sdpa_bwd_delta(bp, dtype, stream);
    if (e != hipSuccess) return e;
    for (int64_t first = 0; first < total && e == hipSuccess; first += max_blocks(512)) {
        const dim3 grid((unsigned)min(total - first, max_blocks(512)));
        if (dtype == 1) hipLaunchKernelGGL((sdpa_bwd_wide_kernel<f16_t>), grid, dim3(512), 0, stream, bp, (int)first);
        else hipLaunchKernelGGL((sdpa_bwd_wide_kernel<bf16_t>), grid, dim3(512), 0, stream, bp, (int)first);
        e = hipGetLastError();
    }
    if (e == hipSuccess && bp.parts_kv > 1) e = launch_sdpa_bwd_sum_planes(bp, dtype, stream);
    return e;
}

}  // namespace incin_rocm
