// f32 attention forward on the gfx950 matrix cores, for head dimensions up to 128 (instances for 64 and 128; a smaller D or Dv, in
// whole 16-byte vectors, is zero-padded on the way into LDS), optional causal mask, per-batch key lengths, a dense additive mask with
// arbitrary broadcast strides, MHA and GQA.  f32 is the one dtype the reference's own operator runs end to end
// (crates/incin-backends/src/cpu/ops/shape_ops.rs:1245-1269 over cpu/ops/matmul.rs:234,254), with a 1e-5 bar.
//
// Products go through the bf16 matrix instruction, every value as the sum of three bf16 ones (f32_split.h: six instructions, no
// larger error than the IEEE-f32 instruction's and 2.7 times its rate; it also lets the vector work of the other wavefronts run beside it).
//
// A workgroup (4 wavefronts) computes 64 query rows of one head; two wavefronts share 32 rows and take a block of 32 keys each of every
// tile of 64, their results meet in LDS at the end.  Operand layouts as in the 16-bit prefill kernels:
//   S^T = K Q'^T     A = K rows (16-byte LDS reads), B = Q'^T (Q' = Q * scale * log2 e, parts kept in registers): a lane owns one
//                    query (column lane % 32) and 16 keys (register r is key 8 (r / 4) + 4 g + r % 4)
//   O^T += V^T P^T   registers 8 h .. 8 h + 7 of P^T are the B operand of 16 keys; A = V^T by transposing LDS reads of the same keys
// A tile's values go global -> registers -> three planes of bf16 rows in LDS, so each is split once per workgroup.  A matrix instruction
// hides about six vector instructions of its own wavefront or another's, no more, so they are dealt out between them, and the loop is a step of two halves:
//   S(t + 1) = K Q', between its products the exponentials and parts of P(t) | barrier
//   O += V(t) P(t), between its products K(t + 2) and V(t + 1) into LDS, K(t + 3) and V(t + 2) asked for | barrier
//
// What bounds it: the 48 matrix instructions of a 32 x 32 block at D = 64 (1536 cycles) and the clock the device keeps under them (about 2.0 GHz with
// N(0,1) data), then the vector instructions beside them, ten to one of those, of which half split K and V: under a causal flag, 4 x 8 x 1024 x 64, the matrix pipes are busy for
// 37 % of the time in which a compute unit has work, wavefronts wait for 19 % of theirs and for their turn to issue for 33 %.  At D > 64 a workgroup has its
// compute unit to itself (434 registers, 144 KiB of LDS).  The instance for mask tensors at D = 64 keeps 11 registers in scratch (48 bytes a lane, 5.6 MB written
// beside 8.4 MB of O in that launch); the others have none.
// Measured, forward, us, IEEE-f32 products (the kernel of 128 rows, or that of 32 for launches it was ahead on) / so: 4 x 8 x 1024 x 64 causal 50.4 /
// 37.1, nothing masked 77.5 / 54.8, 8 x 12 x 2048 x 64 822 / 586, 4 x 12 x 2000 x 64 causal 244 / 166, 8 on 2 x 256 over 8192 keys 85 / 41; 4 x 8 x
// 1024 x 128 causal 90 / 76, 8 x 12 x 2048 x 128 causal 876 / 793, 4 x 8 x 1024 x 80 causal 70 / 60; the causal mask as a tensor, 4 x 8 x 1024 x 64, with the pass over
// it 58.4 / 43.2.  The looks at sizes that decide about a second walk (f32_split.h) are 1 - 3 % of these.  Its error against 64 bits is 0.5 - 0.6 of what it was (2-norm, 4 x 8 x
// 1024 x 64 3.4e-7 -> 2.0e-7, 8 x 12 x 2048 x 64 8.4e-7 -> 2.6e-7, 4 x 8 x 1024 x
// 128 causal 2.3e-7 -> 1.3e-7): sums are rounded at their own size once per product of leading parts, the smaller products meet apart.
//
// A dense additive mask comes with one flag per block of 32 rows x 32 keys (mask_blocks.hip): blocks the mask hides
// completely are skipped, blocks where it is zero run without it, the rest add its values to the scores.  Where the mask's row limits are there
// too (small launches) and all rows of the workgroup have one, those are the mask.
#include <type_traits>

#include "f32_split.h"

namespace incin_rocm {

// SPLIT: the launch is a grid of (work items) x (splits of the key axis); a workgroup handles the keys of its split only and
// writes, per row, the unnormalised O, the maximum and the sum in the partial-result format of the split-KV kernels, whose
// combine kernel finishes - for launches with too few (batch, head, row block) items to fill the device over a long key axis.
//
// DC: the columns that are multiplied, D or fewer: the head dimensions are at most DC, and the products with the zeros beyond are
// left out (the LDS rows keep the layout of D).
template <int D, int DC, bool DENSE, bool SPLIT>
__global__ __launch_bounds__(256, D == 64 ? 2 : 1)
void sdpa_prefill_f32_kernel(SdpaParams p, int paired, int first, int total)
{
#if defined(__HIP_DEVICE_COMPILE__)   // the body uses device-only types (buffer descriptors); the host pass needs only the stub
    constexpr int KT = 64, RW = 2, KW = 4 / RW, OWN = 32 * KW;      // keys per tile, wavefronts that share rows, blocks of 32 rows side by side, rows of the workgroup
    constexpr int NSTEP = DC / 16, NDB = DC / 32;
    constexpr int MAX_FLAGS = 1024;
    constexpr float LOG2E = 1.4426950408889634f;
    typedef SplitTile<D, DC, KT, 256> Tile;
    typedef typename Tile::L L;
    __shared__ __attribute__((aligned(1024))) char smem[3 * Tile::BYTES];      // K, V of even tiles, V of odd ones
    __shared__ int s_vote[12];
    __shared__ uint8_t s_flags[DENSE ? MAX_FLAGS : 1];
    char* const kbuf = smem;

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int own = wave % KW, rs = wave / KW;
    const int ql = lane & 31, g = lane >> 5;
    const int Sq = p.Sq, Skv = p.Skv;

    // ---- which (batch, head, query block): the work order of the 16-bit kernels (longest blocks first, an XCD keeps
    // the heads that share K/V) -----------------------------------------------------------------------------------
    const int nqb = (Sq + OWN - 1) / OWN;
    const int id = first + blockIdx.x;
    int item = id >> 3;
    // (one round, two workgroups to a compute unit, blocks of different lengths: behind the first `paired` of an XCD, one for each of its compute units, the
    // order is reversed, a long one with a short one)
    if (D == 64 && paired && item >= paired) item = paired + ((total >> 3) - 1 - item);
    const WorkItem wi = work_item_of(p, item * 8 + (id & 7), total, nqb);
    const int gq = wi.gq, bhkv = wi.bhkv;
    const int hkv = bhkv % p.Hkv, b = bhkv / p.Hkv;
    const int hq = hkv * p.G + gq;
    const int q0 = wi.qblk * OWN;

    const float* qp = (const float*)p.q + (int64_t)b * p.q_sb + (int64_t)hq * p.q_sh;
    const float* kp = (const float*)p.k + (int64_t)b * p.k_sb + (int64_t)hkv * p.k_sh;
    const float* vp = (const float*)p.v + (int64_t)b * p.v_sb + (int64_t)hkv * p.v_sh;
    float* op = (float*)p.o + (int64_t)b * p.o_sb + (int64_t)hq * p.o_sh;

    int kv_len = Skv;
    if (p.kv_lens) kv_len = clampi(p.kv_lens[b], 0, Skv);
    // a split ends where the next begins: to this workgroup the keys beyond do not exist (split_len is a multiple of the tile)
    const int split = SPLIT ? (int)blockIdx.y : 0;
    if (SPLIT) kv_len = min(kv_len, (split + 1) * p.split_len);
    const int rows_b = p.q_lens ? clampi(p.q_lens[b], 0, Sq) : Sq;      // query rows at and beyond are padding
    if (q0 >= rows_b) return;                                           // (uniform: before any barrier)
    const int coff = Skv - Sq;
    const int my_i = q0 + own * 32 + ql;
    // keys the workgroup walks, this lane's row sees, all rows of the wavefront see
    int j_end = kv_len, lim_lane = kv_len, lim_wave_min = kv_len;
    if (p.causal) {
        j_end = clampi(min(q0 + OWN - 1, rows_b - 1) + coff + 1, 0, kv_len);
        lim_lane = clampi(my_i + coff + 1, 0, kv_len);
        lim_wave_min = clampi(q0 + own * 32 + coff + 1, 0, kv_len);
    }
    bool values = DENSE;      // the mask's values are looked at
    if (DENSE && p.mask_lims != nullptr && p.lims_rows) {
        // a launch of the f32 split-KV kernel went before this one and computed the 128-row blocks whose mask rows are all n
        // zeros and then -inf from their limits (sdpa_decode_f32.hip, LIMS): such a block is done
        const int32_t* lims = mask_lims_of(p, b, hq);
        const int blk0 = q0 / 128 * 128, i = min(blk0 + (tid & 127), min(blk0 + 127, Sq - 1));
        const bool wave_ok = __builtin_amdgcn_ballot_w64(lims[p.m_si ? i : 0] < 0) == 0;
        if (lane == 0) s_vote[wave] = wave_ok ? 1 : 0;
        __syncthreads();
        if ((s_vote[0] & s_vote[1] & s_vote[2] & s_vote[3]) != 0) return;      // (uniform)
        __syncthreads();
    } else if (DENSE && p.mask_lims != nullptr) {
        int lim = my_i < rows_b ? mask_lims_of(p, b, hq)[p.m_si ? my_i : 0] : 0;
        const bool ok = __builtin_amdgcn_ballot_w64(lim < 0) == 0;
        lim = min(lim, lim_lane);
        int hi = lim, lo = my_i < rows_b ? lim : 0x7fffffff;
#pragma unroll
        for (int off = 16; off >= 1; off >>= 1) {
            hi = max(hi, __shfl_xor(hi, off, 64));
            lo = min(lo, __shfl_xor(lo, off, 64));
        }
        if (lane == 0) {
            s_vote[wave] = ok ? 1 : 0;
            s_vote[4 + wave] = hi;
        }
        __syncthreads();
        if ((s_vote[0] & s_vote[1] & s_vote[2] & s_vote[3]) != 0) {      // (uniform)
            values = false;
            lim_lane = lim;
            lim_wave_min = min(__builtin_amdgcn_readfirstlane(lo), kv_len);
            j_end = __builtin_amdgcn_readfirstlane(max(max(s_vote[4], s_vote[5]), max(s_vote[6], s_vote[7])));
        }
        __syncthreads();
    }
    int n_tiles = (j_end + KT - 1) / KT;
    const int t_first = SPLIT ? min(split * (p.split_len / KT), n_tiles) : 0;
    if (DENSE && values) {
        // the flags of a tile's four blocks (0 mixed, 1 all zero, 2 all -inf), two bits each; tiles at the end that the mask hides are left out
        const int nkb32 = (Skv + 31) >> 5, nrb32 = (Sq + 31) >> 5;
        const uint8_t* fl = mask_flags_of(p, b, hq) + (int64_t)(q0 >> 5) * nkb32;
        const int second = (q0 >> 5) + 1 < nrb32 ? nkb32 : 0;
        int last = -1;
        for (int t = tid; t < n_tiles; t += 256) {
            const bool both = 2 * t + 1 < nkb32;
            const unsigned f = fl[2 * t] | (both ? fl[2 * t + 1] : 2u) << 2 | (unsigned)fl[second + 2 * t] << 4 | (both ? fl[second + 2 * t + 1] : 2u) << 6;
            if (t < MAX_FLAGS) s_flags[t] = (uint8_t)f;
            if (f != 0xaau) last = t;
        }
#pragma unroll
        for (int off = 32; off >= 1; off >>= 1) last = max(last, __shfl_xor(last, off, 64));
        if (lane == 0) s_vote[wave] = last;
        __syncthreads();
        n_tiles = __builtin_amdgcn_readfirstlane(max(max(s_vote[0], s_vote[1]), max(s_vote[2], s_vote[3]))) + 1;
        __syncthreads();
    }
    auto flags_of = [&](int t) __attribute__((always_inline)) {
        return !DENSE || !values ? 0x55 : t < MAX_FLAGS ? __builtin_amdgcn_readfirstlane((int)s_flags[t]) : 0;
    };
    // the first tile at or behind t in which any row of the workgroup sees a key, n_tiles if there is none
    auto visible_from = [&](int t) __attribute__((always_inline)) {
        if (DENSE && values)
            while (t < n_tiles && flags_of(t) == 0xaa) ++t;
        return t;
    };

    // operand addresses: K row ql of a block, chunk 2 s + g; V transposed, column block db, half h of 16 rows
    const int k_base = rs * 32 * L::ROWB + ql * L::ROWB + ((g ^ (L::fk(ql) & 1)) << 4) + ((L::fk(ql) & ~1) << 4);      // chunk 2 s + g: ^ (s << 5)
    int v_addr[NDB][2];
    {
        const int n = lane & 15, dh = (lane >> 4) & 1;
#pragma unroll
        for (int db = 0; db < NDB; ++db)
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const int r = 8 * h + 4 * g + (n >> 2), c = 4 * db + 2 * dh + ((n & 3) >> 1);
                v_addr[db][h] = (rs * 32 + r) * L::ROWB + ((c ^ L::fv(r)) << 4) + (n & 1) * 8;
            }
    }
    const float* mrow = nullptr;          // this lane's row of the dense mask
    if (DENSE) mrow = (const float*)p.mask + (int64_t)b * p.m_sb + (int64_t)hq * p.m_sh + (int64_t)min(my_i, rows_b - 1) * p.m_si;
    const bool m_vec = DENSE && p.m_sj == 1 && ((p.m_sb | p.m_sh | p.m_si) & 3) == 0 && (reinterpret_cast<uintptr_t>(p.mask) & 15u) == 0;
    const int flag_shift = own * 4 + rs * 2;

    floatx16 o_acc[NDB];
    float m_run = 0.0f, l_run = 0.0f;      // the reference the row's probabilities are taken against (log2 units), this lane's share of their sum
    auto walk = [&](auto exact_) __attribute__((always_inline)) {
        constexpr bool EXACT = decltype(exact_)::value;
        Tile xk, xv;                     // values on their way into LDS
        Split8 qreg[NSTEP];              // Q', resident
        [[maybe_unused]] float top = 0.0f;      // the largest magnitude of this thread's share of V; infinity: Q' wants EXACT
        int t = visible_from(t_first), t1 = visible_from(t + 1), t2 = visible_from(t1 + 1);
        // ---- Q' into operands, through the place of the second V tile; the first K and V tiles ----
        {
            Tile xq;
            xq.fetch_any(qp, p.q_ss, p.D, rows_b, q0, tid);      // (padding rows may hold anything, what starts EXACT among it: the last row in their place)
            xk.fetch(kp, p.k_ss, p.D, j_end, t * KT, tid);
            xv.fetch(vp, p.v_ss, p.Dv, j_end, t * KT, tid);
            // (a score's error by what K loses is negligible under a Q' up to 2^60, and Q' itself loses nothing from 2^-100 on)
            if (!EXACT && xq.scaled_beyond(p.scale * LOG2E, p.D, tid)) top = INFINITY;
            if (!EXACT) top = xv.largest_of(top);
            xq.template put_scaled<EXACT, true>(smem + 2 * Tile::BYTES, p.scale * LOG2E, tid);
            xk.template put<EXACT, true>(kbuf, tid);
            xv.template put<EXACT, false>(smem + Tile::BYTES, tid);
        }
        xk.fetch(kp, p.k_ss, p.D, j_end, t1 * KT, tid);
        xv.fetch(vp, p.v_ss, p.Dv, j_end, t1 * KT, tid);
        lds_barrier();
#pragma unroll
        for (int s = 0; s < NSTEP; ++s) qreg[s] = Tile::rows_operand(smem + 2 * Tile::BYTES + ((k_base + (own - rs) * 32 * L::ROWB) ^ (s << 5)));

        [[maybe_unused]] float mv[16];      // dense mask values of this lane's 16 keys
        [[maybe_unused]] auto fetch_mask = [&](int t) __attribute__((always_inline)) {
            typedef float float4v __attribute__((ext_vector_type(4)));
            if (t >= n_tiles || ((flags_of(t) >> flag_shift) & 3) != 0) return;
            const int j0 = t * KT + rs * 32;
            if (m_vec && j0 + 32 <= Skv) {
#pragma unroll
                for (int r4 = 0; r4 < 4; ++r4) {
                    const float4v w = *(const float4v*)(mrow + j0 + 8 * r4 + 4 * g);
#pragma unroll
                    for (int e = 0; e < 4; ++e) mv[4 * r4 + e] = w[e];
                }
            } else {
#pragma unroll
                for (int r = 0; r < 16; ++r) mv[r] = mrow[(int64_t)min(j0 + 8 * (r / 4) + 4 * g + (r % 4), Skv - 1) * p.m_sj];
            }
        };
        // S^T = K Q'^T of the tile in kbuf, `between(i)` behind each of its 6 NSTEP instructions
        auto scores = [&](floatx16& s, auto between) __attribute__((always_inline)) {
#pragma unroll
            for (int r = 0; r < 16; ++r) s[r] = 0.0f;
            // (the five smaller products of all steps, then the leading ones: the sum is rounded at its own size NSTEP times, not 6 NSTEP)
            Split8 a = Tile::rows_operand(kbuf + k_base);
            uint4p lead[NSTEP];
#pragma unroll
            for (int i = 0; i < NSTEP; ++i) {
                Split8 n = a;
                if (i + 1 < NSTEP) n = Tile::rows_operand(kbuf + (k_base ^ ((i + 1) << 5)));
                __builtin_amdgcn_sched_barrier(0);
                lead[i] = a.h;
                if (EXACT) s = mma_split<true>(a, qreg[i], s);
                mma_split_term<EXACT, 0>(a, qreg[i], s); between(5 * i);
                mma_split_term<EXACT, 1>(a, qreg[i], s); between(5 * i + 1);
                mma_split_term<EXACT, 2>(a, qreg[i], s); between(5 * i + 2);
                mma_split_term<EXACT, 3>(a, qreg[i], s); between(5 * i + 3);
                mma_split_term<EXACT, 4>(a, qreg[i], s); between(5 * i + 4);
                a = n;
            }
#pragma unroll
            for (int i = 0; i < NSTEP; ++i) {
                a.h = lead[i];
                if (!EXACT) mma_split_term<EXACT, 5>(a, qreg[i], s);
                between(5 * NSTEP + i);
            }
        };
        floatx16 s;
        scores(s, [](int) {});
        if (DENSE && values) fetch_mask(t);
        lds_barrier();
        if (t1 < n_tiles) xk.template put<EXACT, true>(kbuf, tid);
        xk.fetch(kp, p.k_ss, p.D, j_end, t2 * KT, tid);
#pragma unroll
        for (int db = 0; db < NDB; ++db)
#pragma unroll
            for (int r = 0; r < 16; ++r) o_acc[db][r] = 0.0f;
        m_run = 0.0f;
        l_run = 0.0f;
        float rise = -INFINITY;      // the reference moves where a block's maximum passes it by more than this: at the first key seen, then by 2^8
        lds_barrier();
        for (int even = 0; t < n_tiles; even ^= 1) {
            const int j0 = t * KT + rs * 32;
            if (DENSE && values) {
                const int flag = (flags_of(t) >> flag_shift) & 3;
                if (flag == 0) {
                    asm volatile("");
#pragma unroll
                    for (int r = 0; r < 16; ++r) s[r] = __builtin_fmaf(mv[r], LOG2E, s[r]);
                } else if (flag == 2) {
                    asm volatile("");
#pragma unroll
                    for (int r = 0; r < 16; ++r) s[r] = -INFINITY;
                }
            }
            if (j0 + 32 > lim_wave_min) {                     // (uniform) the block crosses a limit of this wavefront
                asm volatile("");      // (a branch, not sixteen selects in every block)
                const int rel = lim_lane - (j0 + 4 * g);
#pragma unroll
                for (int r = 0; r < 16; ++r)
                    if (8 * (r / 4) + (r % 4) >= rel) s[r] = -INFINITY;
            }
            // EXACT: a block that none of the wavefront's rows sees is left out of the product with V, whose rows may hold anything there
            const bool unseen = EXACT && (((flags_of(t) >> flag_shift) & 3) == 2 || __builtin_amdgcn_ballot_w64(my_i < rows_b && j0 < lim_lane) == 0);
            // ---- online softmax: probabilities are taken against a reference that moves rarely (they stay <= 2^8; EXACT: <= 1, so that values
            // of V up to the largest finite one do not overflow where the result does not) ----
            float tmax = s[0];
#pragma unroll
            for (int r = 1; r < 16; ++r) tmax = fmaxf(tmax, s[r]);
            if (__builtin_amdgcn_ballot_w64(tmax - m_run > rise) != 0) {
                tmax = xor32_max(tmax);
                const bool need = tmax - m_run > rise;
                const float to = need ? tmax : m_run, alpha = rise == -INFINITY ? 1.0f : __builtin_amdgcn_exp2f(m_run - to);      // (first key: nothing summed yet)
                if (need) rise = EXACT ? 0.0f : PF_RESCALE_THRESHOLD;
                m_run = to;
                l_run *= alpha;
#pragma unroll
                for (int db = 0; db < NDB; ++db)
#pragma unroll
                    for (int r = 0; r < 16; ++r) o_acc[db][r] *= alpha;
            }
            // ---- P^T and its parts, between the next tile's first products ----
            Split8 pr[2];
            SplitPair pair;
            float e0 = 0.0f, e1 = 0.0f, bsum = 0.0f;
            auto soft = [&](int k) __attribute__((always_inline)) {      // piece k of 24: three per two values
                const int q = k / 3, part = k % 3, h = q / 4;
                if (part == 0) {
                    e0 = __builtin_amdgcn_exp2f(s[2 * q] - m_run);
                    e1 = __builtin_amdgcn_exp2f(s[2 * q + 1] - m_run);
                    return;
                }
                unsigned x = pr[h].h[q % 4], y = pr[h].m[q % 4], z = pr[h].l[q % 4];
                if (part == 1) {
                    bsum += e0;
                    bsum += e1;
                    pair.template step<EXACT, 0>(e0, e1, x, y, z);
                } else {
                    pair.template step<EXACT, 1>(e0, e1, x, y, z);
                    pair.template step<EXACT, 2>(e0, e1, x, y, z);
                }
                pr[h].h[q % 4] = x;
                pr[h].m[q % 4] = y;
                pr[h].l[q % 4] = z;
            };
            floatx16 s1;
            if (t1 < n_tiles) {
                scores(s1, [&](int i) __attribute__((always_inline)) {
                    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                    for (int k = 24 * i / (6 * NSTEP); k < 24 * (i + 1) / (6 * NSTEP); ++k) soft(k);
                    __builtin_amdgcn_sched_barrier(0);
                });
            } else {
#pragma unroll
                for (int k = 0; k < 24; ++k) soft(k);
            }
            l_run += bsum;
            lds_barrier();
            // ---- O^T += V^T P^T, between them the next tiles' values into LDS ----
            const int t3 = visible_from(t2 + 1);
            if (DENSE && values) fetch_mask(t1);
            const char* const vcur = smem + (1 + even) * Tile::BYTES;
            char* const vnext = smem + (2 - even) * Tile::BYTES;
            typename Tile::State st;
            constexpr int NM = 12 * NDB, NS = Tile::STEPS;
            auto put = [&](int i) __attribute__((always_inline)) {      // behind matrix instruction i
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int k = 2 * NS * i / NM; k < 2 * NS * (i + 1) / NM; ++k) {
                    if (k < NS) xk.template put_step<EXACT, true>(k, st, kbuf, tid);
                    else {
                        if (!EXACT) top = xv.largest_step(k - NS, top);
                        xv.template put_step<EXACT, false>(k - NS, st, vnext, tid);
                    }
                    if (k == NS - 1) xk.fetch(kp, p.k_ss, p.D, j_end, t3 * KT, tid);
                }
                __builtin_amdgcn_sched_barrier(0);
            };
            // (the five smaller products of a block meet in registers of their own before the sums so far take them: O is rounded at its own
            // size three times per 32 keys instead of twelve)
            Split8 a = Tile::cols_operand(vcur, v_addr[0][0], v_addr[0][1]);
            floatx16 small;
#pragma unroll
            for (int i = 0; i < 2 * NDB; ++i) {
                const int db = i / 2, h = i % 2, dn = (i + 1) / 2, hn = (i + 1) % 2;
                Split8 n = a;
                if (i + 1 < 2 * NDB) n = Tile::cols_operand(vcur + hn * 16 * L::ROWB, v_addr[dn][0], v_addr[dn][1]);
                __builtin_amdgcn_sched_barrier(0);
                if (h == 0) {
                    if (db > 0) {
#pragma unroll
                        for (int r = 0; r < 16; ++r) o_acc[db > 0 ? db - 1 : 0][r] += small[r];
                    }
#pragma unroll
                    for (int r = 0; r < 16; ++r) small[r] = 0.0f;
                }
                mma_split_term<EXACT, 0>(a, pr[h], small); put(6 * i);
                mma_split_term<EXACT, 1>(a, pr[h], small); put(6 * i + 1);
                mma_split_term<EXACT, 2>(a, pr[h], small); put(6 * i + 2);
                mma_split_term<EXACT, 3>(a, pr[h], small); put(6 * i + 3);
                mma_split_term<EXACT, 4>(a, pr[h], small); put(6 * i + 4);
                if (!unseen) mma_split_term<EXACT, 5>(a, pr[h], o_acc[db]);
                put(6 * i + 5);
                a = n;
            }
#pragma unroll
            for (int r = 0; r < 16; ++r) o_acc[NDB - 1][r] += small[r];
            xv.fetch(vp, p.v_ss, p.Dv, j_end, t2 * KT, tid);
            lds_barrier();
            s = s1;
            t = t1;
            t1 = t2;
            t2 = t3;
        }
        if constexpr (EXACT) return false;
        // A result that is not finite, or one so small that what the parts lose (f32_split.h) could show: of V under the sum of the weights, of the
        // weights under V.  (The sum is at most 2^8 a key.)  First whether all of a lane's are in a range where it could not, or zeros that no tiny V explains:
        // two instructions for two values, where the precise look takes five, and a workgroup meets its instructions for the first time here.
        {
            float hi = 0.0f, lo = INFINITY;
            auto take = [&](float x) __attribute__((always_inline)) {
                hi = __builtin_elementwise_maximum(hi, __builtin_fabsf(x));      // (keeps a NaN)
                lo = __builtin_fminf(lo, __builtin_fabsf(x));
            };
#pragma unroll
            for (int db = 0; db < NDB; ++db)
#pragma unroll
                for (int r4 = 0; r4 < 4; ++r4) {
                    if (DC < 128 && db * 32 + r4 * 8 >= p.Dv) continue;      // (uniform: columns of padding, zeros)
                    if (DC < 128) asm volatile("");
#pragma unroll
                    for (int e = 0; e < 4; ++e) take(o_acc[db][r4 * 4 + e]);
                }
            const bool fine = hi < INFINITY && l_run < INFINITY && (lo >= 0x1p-40f || hi == 0.0f) && top <= 0x1p50f && n_tiles - t_first <= (1 << 20) / KT;
            const bool wave_fine = __builtin_amdgcn_ballot_w64(!fine) == 0 && __builtin_amdgcn_ballot_w64(top >= SPLIT_TINY) != 0;
            if (lane == 0) s_vote[wave] = wave_fine ? 1 : 0;
            lds_barrier();
            if ((s_vote[0] & s_vote[1] & s_vote[2] & s_vote[3]) != 0) return false;      // (uniform)
            lds_barrier();
        }
        float chk = l_run * 0.0f;
        unsigned low = ~0u;
#pragma unroll
        for (int db = 0; db < NDB; ++db)
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                chk = __builtin_fmaf(o_acc[db][r], 0.0f, chk);
                low = smallest(low, o_acc[db][r]);
            }
        const bool bad = __builtin_amdgcn_ballot_w64(chk != 0.0f) != 0;
        const unsigned w_top = wave_extreme<true>(__float_as_uint(top)), w_low = wave_extreme<false>(low);
        if (lane == 0) {
            s_vote[wave] = bad ? 1 : 0;
            s_vote[4 + wave] = (int)w_top;
            s_vote[8 + wave] = (int)w_low;
        }
        lds_barrier();
        const float v_top = __uint_as_float(max(max(s_vote[4], s_vote[5]), max(s_vote[6], s_vote[7])));
        low = min(min((unsigned)s_vote[8], (unsigned)s_vote[9]), min((unsigned)s_vote[10], (unsigned)s_vote[11]));
        const float bound = SPLIT_LOST * (float)((n_tiles - t_first) * KT) * (v_top + 256.0f);
        return (s_vote[0] | s_vote[1] | s_vote[2] | s_vote[3]) != 0 || !(v_top < INFINITY) || low < smallest_of(bound) || (v_top > 0.0f && v_top < SPLIT_TINY);      // (uniform)
    };
    if (n_tiles > t_first) {
        if (walk(std::integral_constant<bool, false>{})) {
            lds_barrier();
            walk(std::integral_constant<bool, true>{});
        }
    } else {
#pragma unroll
        for (int db = 0; db < NDB; ++db)
#pragma unroll
            for (int r = 0; r < 16; ++r) o_acc[db][r] = 0.0f;
    }

    // ---- the two wavefronts that share rows: each keeps the column blocks db with db % 2 == rs, and has the other's of them added ----
    constexpr int NKEEP = (NDB + 1) / 2;
    float l_tot = xor32_sum(l_run);
    {
        // (the tiles are done with) [wavefront][column block it gives away][16][64], behind them m and l of each wavefront's rows
        float* const give = (float*)smem;
        float* const ml = give + 4 * NKEEP * 16 * 64;
#pragma unroll
        for (int db = 0; db < NDB; ++db)
            if (db % 2 != rs) {
#pragma unroll
                for (int r = 0; r < 16; ++r) give[((wave * NKEEP + db / 2) * 16 + r) * 64 + lane] = o_acc[db][r];
            }
        if (g == 0) {
            ml[(wave * 32 + ql) * 2] = m_run;
            ml[(wave * 32 + ql) * 2 + 1] = l_tot;
        }
        lds_barrier();
        const int other = wave ^ KW;
        const float m2 = ml[(other * 32 + ql) * 2], l2 = ml[(other * 32 + ql) * 2 + 1];
        // (a wavefront that saw no key has l = 0, and its reference says nothing)
        const float top = l_tot == 0.0f ? m2 : l2 == 0.0f ? m_run : fmaxf(m_run, m2);
        const float f1 = l_tot == 0.0f ? 0.0f : __builtin_amdgcn_exp2f(m_run - top), f2 = l2 == 0.0f ? 0.0f : __builtin_amdgcn_exp2f(m2 - top);
        m_run = top;
        l_tot = l_tot * f1 + l2 * f2;
#pragma unroll
        for (int k = 0; k < NKEEP; ++k) {
            if (2 * k + rs >= NDB) break;
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const float mine = 2 * k + 1 < NDB && rs == 1 ? o_acc[2 * k + 1 < NDB ? 2 * k + 1 : 0][r] : o_acc[2 * k][r];
                o_acc[k][r] = mine * f1 + give[((other * NKEEP + k) * 16 + r) * 64 + lane] * f2;
            }
        }
        lds_barrier();      // (what follows stages rows in the same place)
    }
    // o_acc[k]: column block 2 k + rs
    // ---- normalise and store --------------------------------------------------------------------------------------
    if constexpr (SPLIT) {
        // partial result of this split: unnormalised O, and (maximum, sum) in the natural-log units the combine kernel takes
        // for f32 storage; a row that saw no key in this split has the maximum -inf
        typedef float float4v __attribute__((ext_vector_type(4)));
        if (my_i < rows_b) {
            const int64_t slot = (((int64_t)b * p.Hq + hq) * Sq + my_i) * p.num_splits + split;
            float* arow = p.ws_acc + slot * D + g * 4;
#pragma unroll
            for (int k = 0; k < NKEEP; ++k)
#pragma unroll
                for (int r4 = 0; r4 < 4; ++r4) {
                    float4v w = {o_acc[k][r4 * 4], o_acc[k][r4 * 4 + 1], o_acc[k][r4 * 4 + 2], o_acc[k][r4 * 4 + 3]};
                    if (2 * k + rs < NDB) *(float4v*)(arow + (2 * k + rs) * 32 + r4 * 8) = w;
                }
            if (g == 0 && rs == 0) {
                p.ws_ml[slot * 2 + 0] = l_tot == 0.0f ? -INFINITY : m_run * 0.6931471805599453f;
                p.ws_ml[slot * 2 + 1] = l_tot;
            }
        }
        return;
    }
    const float inv = (l_tot == 0.0f) ? __builtin_nanf("") : 1.0f / l_tot;   // no visible key: NaN, as the reference
    if (p.lse && g == 0 && rs == 0 && my_i < rows_b)
        p.lse[((int64_t)b * p.Hq + hq) * Sq + my_i] = l_tot == 0.0f ? -INFINITY : (m_run + __builtin_log2f(l_tot)) * 0.6931471805599453f;
#pragma unroll
    for (int k = 0; k < NKEEP; ++k) {
        const floatx16 one[1] = {o_acc[k]};
        const int c0 = (2 * k + rs) * 32;
        if (c0 >= DC) break;
        store_o_rows_f32(one, inv, smem + wave * 4096, op + c0, q0 + own * 32, rows_b, p.o_ss, p.Dv - c0, lane);
    }
#endif
}

hipError_t launch_sdpa_combine(const SdpaParams& p, int dtype, hipStream_t stream);

template <int D, int DC, bool DENSE>
static hipError_t launch_prefill_f32_t(const SdpaParams& p0, hipStream_t stream)
{
    constexpr int OWN = 64;
    SdpaParams p = p0;
    const int nqb = (p.Sq + OWN - 1) / OWN;
    const int64_t total = (int64_t)nqb * p.Hq * p.B;
    if (total <= 0) return hipSuccess;
    if (total > 0x7fffffffLL) return hipErrorInvalidValue;
    const bool uneven = p.causal != 0 || p.mask != nullptr;
    work_order(p, D == 64 ? 2 : 1, nqb);
    const int64_t cus = device_cus();
    const int paired = D == 64 && uneven && (total & 7) == 0 && total > cus && total <= 2 * cus ? (int)(cus / 8) : 0;
    const bool split = !DENSE && p.num_splits > 1;      // partial results, then the split-KV kernels' combine pass
    hipError_t e = hipSuccess;
    for (int64_t first = 0; first < total && e == hipSuccess; first += max_blocks(256)) {
        const dim3 grid((unsigned)std::min(total - first, max_blocks(256)), split ? (unsigned)p.num_splits : 1u);
        if (split) hipLaunchKernelGGL((sdpa_prefill_f32_kernel<D, DC, false, !DENSE>), grid, dim3(256), 0, stream, p, 0, (int)first, (int)total);
        else hipLaunchKernelGGL((sdpa_prefill_f32_kernel<D, DC, DENSE, false>), grid, dim3(256), 0, stream, p, paired, (int)first, (int)total);
        e = hipGetLastError();
    }
    return split && e == hipSuccess ? launch_sdpa_combine(p, 0, stream) : e;
}
template <int D, int DC> static hipError_t launch_prefill_f32_m(const SdpaParams& p, hipStream_t stream)
{
    return p.mask ? launch_prefill_f32_t<D, DC, true>(p, stream) : launch_prefill_f32_t<D, DC, false>(p, stream);
}

// Host has validated: f32, D and Dv <= 128 in whole 16-byte vectors (p.Dp = the instance: 64 or 128), finite scale, rows 16-byte aligned with unit last-dim stride, row
// strides of K and V below 2^22 elements (tile offsets fit the 32-bit buffer offset); the dense mask, if any, has any strides.
hipError_t launch_sdpa_prefill_f32(const SdpaParams& p, hipStream_t stream)
{
    if (p.Dp == 64) return launch_prefill_f32_m<64, 64>(p, stream);
    // up to head dimension 96 in the 128 layout: three quarters of the products
    if (p.D <= 96 && p.Dv <= 96) return launch_prefill_f32_m<128, 96>(p, stream);
    return launch_prefill_f32_m<128, 128>(p, stream);
}

}  // namespace incin_rocm
