// Split-KV attention on the matrix cores for a batch whose sequences differ in length (key counts on the device), f16 / bf16, one to a
// few query rows per KV head: the function, the operand layouts and the arithmetic of sdpa_decode_mfma.hip, which see.
//
// That kernel gives a workgroup one split of one sequence, and the host, which does not know the counts, makes splits of the
// capacity: with counts spread evenly from an eighth of it to all of it the compute units are left with very different amounts,
// and the memory system idles while the longest finish (12 sequences of 2048 - 16384 keys on 8 KV heads: 91.6 us where 453 MB take
// 64; dealt 75.4).  Here the keys of all sequences are dealt to the workgroups of one round in equal shares (decode_deal.h).  A share is a run of
// one to a few sequences' keys, and the ring of copies runs through it without a break: when the blocks of one sequence are
// all on their way, the next copies are the next sequence's, so that while the four wavefronts' results of the first meet
// and its rows of Q give way to the next one's, the ring fills on.  For that the results have LDS of their own, behind the
// rings: rows x columns of each wavefront, which is why this form is for few rows (rows x head dimension up to 1024).
// (With a ring drained and refilled for each sequence 32 x 1031 - 8192 keys took 103 us instead of 98, equal counts of 4608 95.9 instead of 93.5.)
#include <atomic>

#include "decode_deal.h"
#include "sdpa_decode_ring.h"

namespace incin_rocm {

// A place in a workgroup's share: column, sequence, unit of it to go on from, units left of the share.
struct DealCursor {
    int column, b, from, left;
};

template <typename T, int D, int NSLOT>
__global__ __launch_bounds__(256) void sdpa_decode_deal_kernel(SdpaParams p)
{
#if defined(__HIP_DEVICE_COMPILE__)
    typedef typename Mma<T>::vec8 vec8;
    typedef PfLayout<D> L;
    typedef float f4 __attribute__((ext_vector_type(4)));
    constexpr int NSTEP = D / 16, NDB = D / 32;
    constexpr int SLOT = D > 128 ? 2 * DM_SLOT_BYTES : DM_SLOT_BYTES;      // a slot holds 8 KiB, at D = 256 the 16 KiB of 32 keys
    constexpr int KB = SLOT / (32 * L::ROWB);          // 32-key sub-blocks of a block: 2 at D = 64, else 1
    constexpr int BLOCK = 32 * KB;                     // keys per block
    constexpr int CPB = SLOT / 1024;                   // wavefront-wide 1 KiB copies per block
    constexpr int UNIT = deal_unit<T, D>();
    static_assert(UNIT == 4 * BLOCK, "a unit is one block per wavefront");
    extern __shared__ __attribute__((aligned(1024))) char smem[];

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int ql = lane & 31, g = lane >> 5;
    const int Sq = p.Sq, Skv = p.Skv;
    const int R = p.G * Sq;                            // at most DEAL_MAX_VALUES / D

    // ---- this workgroup's share ------------------------------------------------------------------------------------
    DealCursor in, out;      // where copies are started, where blocks are used
    {
        const DealColumn col = deal_column<UNIT>(p);
        const DealShares shares(col.total * p.Hkv, p.deal);
        if ((int)blockIdx.x >= shares.count) return;
        const int pos = shares.begin(blockIdx.x);
        int first;
        in.column = pos / col.total;
        deal_find(col, pos - in.column * col.total, &in.b, &first);
        in.from = pos - in.column * col.total - first;
        in.left = shares.begin(blockIdx.x + 1) - pos;
    }
    out = in;
    auto len_of = [&](int b) __attribute__((always_inline)) { return p.kv_lens ? clampi(p.kv_lens[b], 0, Skv) : Skv; };
    // the part of a share that lies in the cursor's sequence: its keys, and whether the sequence goes on behind the share
    struct Part { int begin, end, units; bool goes_on; };
    auto part_of = [&](const DealCursor& c) __attribute__((always_inline)) {
        const int len = len_of(c.b), units = max(1, (len + UNIT - 1) / UNIT);
        Part a;
        a.units = min(units - c.from, c.left);
        a.goes_on = c.from + a.units < units;
        a.begin = c.from * UNIT;
        a.end = min((c.from + a.units) * UNIT, len);
        return a;
    };
    auto next_sequence = [&](DealCursor& c, const Part& a) __attribute__((always_inline)) {
        c.left -= a.units;
        c.from = 0;
        if (++c.b == p.B) { c.b = 0; ++c.column; }
    };
    auto blocks_of = [&](const Part& a) __attribute__((always_inline)) {      // of this wavefront: wave, wave + 4, ...
        const int n = a.end > a.begin ? (a.end - a.begin + BLOCK - 1) / BLOCK : 0;
        return n > wave ? (n - wave + 3) >> 2 : 0;
    };

    // ---- global -> LDS copies: K(block 0) V(0) K(1) V(1) ... of this wavefront, copy number n into slot n % NSLOT ----------
    int k_voff[CPB], v_voff[CPB];
#pragma unroll
    for (int c = 0; c < CPB; ++c) {
        const int pos = c * 64 + lane;
        const int r = pos / L::CPR, slot = pos % L::CPR;
        k_voff[c] = dma_chunk_offset(r, (int)p.k_ss * 2, slot ^ L::fk(r), p.D * 2);
        v_voff[c] = dma_chunk_offset(r, (int)p.v_ss * 2, slot ^ L::fv(r), p.Dv * 2);
    }
    const int64_t k_step = (int64_t)4 * BLOCK * p.k_ss * 2, v_step = (int64_t)4 * BLOCK * p.v_ss * 2;
    const char *k_next = (const char*)p.k, *v_next = (const char*)p.v;
    int64_t k_rem = 0, v_rem = 0;      // bytes from there to the end of the part's last row; 0: nothing is left to copy
    int to_copy = 0;                   // blocks of the part whose copies have not been started
    auto clamp31 = [](int64_t x) __attribute__((always_inline)) {
        const unsigned hi = (unsigned)((unsigned long long)x >> 32), lo = (unsigned)x;
        return x <= 0 ? 0 : (hi | (lo >> 31)) != 0 ? 0x7fffffff : (int)lo;
    };
    auto next_part = [&]() __attribute__((always_inline)) {      // the next part in which this wavefront has a block
        k_rem = v_rem = 0;
        while (to_copy == 0 && in.left > 0) {
            const Part a = part_of(in);
            to_copy = blocks_of(a);
            const int first_key = a.begin + wave * BLOCK;
            k_next = (const char*)((const T*)p.k + (int64_t)in.b * p.k_sb + (int64_t)in.column * p.k_sh + (int64_t)first_key * p.k_ss);
            v_next = (const char*)((const T*)p.v + (int64_t)in.b * p.v_sb + (int64_t)in.column * p.v_sh + (int64_t)first_key * p.v_ss);
            if (to_copy > 0) {
                k_rem = (int64_t)(a.end - first_key - 1) * p.k_ss * 2 + p.D * 2;
                v_rem = (int64_t)(a.end - first_key - 1) * p.v_ss * 2 + p.Dv * 2;
            }
            next_sequence(in, a);
        }
    };
    next_part();
    const unsigned ring = lds_address(smem) + wave * NSLOT * SLOT;
    // (started unconditionally, NSLOT ahead of their use: past the share's last block the descriptor covers nothing and the copy
    // delivers zeros into a slot nobody reads, so that the wait for the oldest copy is the same from the first block to the last)
    static_assert(NSLOT % 2 == 0, "the slot a K block leaves takes a K block");
    int slot_in = 0;
    auto start = [&](const char* from, int64_t rem, const int (&voff)[CPB]) __attribute__((always_inline)) {
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");      // (this wavefront's reads of the slot have delivered)
        const uint4v r = dma_descriptor(from, clamp31(rem));
#pragma unroll
        for (int c = 0; c < CPB; ++c) dm_copy16(r, ring + slot_in * SLOT + c * 1024, voff[c]);
        slot_in = slot_in + 1 == NSLOT ? 0 : slot_in + 1;
    };
    auto next_k = [&]() __attribute__((always_inline)) {
        start(k_next, k_rem, k_voff);
        k_next += k_step;
        k_rem -= k_step;
    };
    auto next_v = [&]() __attribute__((always_inline)) {
        start(v_next, v_rem, v_voff);
        v_next += v_step;
        v_rem -= v_step;
        if (to_copy > 0 && --to_copy == 0) next_part();
    };
    for (int u = 0; u < NSLOT / 2; ++u) {
        next_k();
        next_v();
    }

    // operand addresses (sdpa_decode_mfma.hip)
    int k_addr[NSTEP];
#pragma unroll
    for (int s = 0; s < NSTEP; ++s) k_addr[s] = ql * L::ROWB + (((2 * s + g) ^ L::fk(ql)) << 4);
    int v_addr[NDB][2];
    {
        const int n = lane & 15, dh = (lane >> 4) & 1;
#pragma unroll
        for (int db = 0; db < NDB; ++db)
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const int r = 8 * h + 4 * g + (n >> 2);
                const int chunk = 4 * db + 2 * dh + ((n & 3) >> 1);
                v_addr[db][h] = r * L::ROWB + ((chunk ^ L::fv(r)) << 4) + (n & 1) * 8;
            }
    }
    const float sc2 = p.scale * 1.4426950408889634f;      // scores in log2 units
    const bool valid = ql < R;
    const int gq = !valid ? 0 : Sq > 1 ? ql / Sq : ql, qi = valid ? ql - gq * Sq : 0;
    // results of the wavefronts: [4][R] (maximum, sum), [4][R][D] numerators
    float2* const s_ml = (float2*)(smem + 4 * NSLOT * SLOT);
    float* const s_o = (float*)(smem + 4 * NSLOT * SLOT + 4 * (DEAL_MAX_VALUES / D) * sizeof(float2));

    int slot_out = 0;              // slot of the copy consumed next
    while (out.left > 0) {
        const Part part = part_of(out);
        const int b = out.b, hkv = out.column;
        // keys that this lane's row, and any row, may see of the part
        const int lim = !valid ? 0 : p.causal ? min(part.end, causal_limit(qi, Sq, Skv)) : part.end;
        const int mask_from = p.causal ? min(part.end, causal_limit(0, Sq, Skv)) : part.end;      // blocks that end at or before need no mask
        vec8 qreg[NSTEP];
        {
            const T* qrow = (const T*)p.q + (int64_t)b * p.q_sb + (int64_t)(hkv * p.G + gq) * p.q_sh + (int64_t)qi * p.q_ss;
#pragma unroll
            for (int s = 0; s < NSTEP; ++s) qreg[s] = *(const vec8*)(qrow + (s * 16 + g * 8 < p.D ? s * 16 + g * 8 : 0));
#pragma unroll
            for (int s = 0; s < NSTEP; ++s)
                if (!valid || s * 16 + g * 8 >= p.D)      // (rows that do not exist, and beyond the head dimension: zeros, like K's)
#pragma unroll
                    for (int e = 0; e < 8; ++e) qreg[s][e] = (T)0.0f;
        }
        float m_run = -INFINITY, l_run = 0.0f;
        floatx16 o_acc[NDB];
#pragma unroll
        for (int db = 0; db < NDB; ++db)
#pragma unroll
            for (int r = 0; r < 16; ++r) o_acc[db][r] = 0.0f;

        const int my_blocks = blocks_of(part), first_key = part.begin + wave * BLOCK;
        for (int j = 0; j < my_blocks; ++j) {
            const int j0 = first_key + j * 4 * BLOCK;
            // ---- S^T = K Q^T ----
            wait_oldest_copy<NSLOT, CPB>();
            const char* kb = smem + (wave * NSLOT + slot_out) * SLOT;
            slot_out = slot_out + 1 == NSLOT ? 0 : slot_out + 1;
            floatx16 sacc[KB];
#pragma unroll
            for (int kb2 = 0; kb2 < KB; ++kb2)
#pragma unroll
                for (int r = 0; r < 16; ++r) sacc[kb2][r] = 0.0f;
#pragma unroll
            for (int s = 0; s < NSTEP; ++s)
#pragma unroll
                for (int kb2 = 0; kb2 < KB; ++kb2) sacc[kb2] = Mma<T>::run(*(const vec8*)(kb + k_addr[s] + kb2 * 32 * L::ROWB), qreg[s], sacc[kb2]);
            next_k();                  // (the block's values are in registers: its slot takes the next copy)
            // register r of sub-block kb2 is key j0 + 32 kb2 + 8 (r / 4) + 4 g + (r % 4)
#pragma unroll
            for (int kb2 = 0; kb2 < KB; ++kb2)
#pragma unroll
                for (int r = 0; r < 16; ++r) sacc[kb2][r] *= sc2;
            if (j0 + BLOCK > mask_from) {
                const int rel = lim - (j0 + 4 * g);
#pragma unroll
                for (int kb2 = 0; kb2 < KB; ++kb2)
#pragma unroll
                    for (int r = 0; r < 16; ++r)
                        if (32 * kb2 + 8 * (r / 4) + (r % 4) >= rel) sacc[kb2][r] = -INFINITY;
            }
            float tmax = sacc[0][0];
#pragma unroll
            for (int kb2 = 0; kb2 < KB; ++kb2)
#pragma unroll
                for (int r = 0; r < 16; ++r) tmax = fmaxf(tmax, sacc[kb2][r]);
            tmax = xor32_max(tmax);              // largest score of the row in this block (log2 units)
            // the reference moves only when a block's maximum passes it by more than 2^8 (or the row sees its first key)
            const bool need = tmax > m_run + PF_RESCALE_THRESHOLD;      // (-inf + 8 = -inf: any finite maximum passes it)
            if (__builtin_amdgcn_ballot_w64(need) != 0) {
                const float alpha = need ? __builtin_amdgcn_exp2f(m_run - tmax) : 1.0f;   // (first key: exp2(-inf) = 0 times 0)
                if (need) m_run = tmax;
                l_run *= alpha;
#pragma unroll
                for (int db = 0; db < NDB; ++db)
#pragma unroll
                    for (int r = 0; r < 16; ++r) o_acc[db][r] *= alpha;
            }
            const float m_use = (m_run == -INFINITY) ? 0.0f : m_run;
            // P^T in storage precision: element e of k-step ks is register 8 (ks % 2) + e of sub-block ks / 2; the denominator is
            // summed from the rounded values
            vec8 pb[2 * KB];
            float rsum = 0.0f;
#pragma unroll
            for (int ks = 0; ks < 2 * KB; ++ks) {
#pragma unroll
                for (int e = 0; e < 8; ++e) pb[ks][e] = (T)__builtin_amdgcn_exp2f(sacc[ks / 2][8 * (ks % 2) + e] - m_use);
#pragma unroll
                for (int e = 0; e < 8; e += 2) {
                    typename Mma<T>::vec2 pr = {pb[ks][e], pb[ks][e + 1]};
                    rsum = Mma<T>::add2(pr, rsum);
                }
            }
            l_run += rsum;
            // ---- O^T += V^T P^T ----
            wait_oldest_copy<NSLOT, CPB>();
            const char* vb = smem + (wave * NSLOT + slot_out) * SLOT;
            slot_out = slot_out + 1 == NSLOT ? 0 : slot_out + 1;
#pragma unroll
            for (int ks = 0; ks < 2 * KB; ++ks)
#pragma unroll
                for (int db = 0; db < NDB; ++db) {
                    short8v av;
                    av.lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((short4v __attribute__((address_space(3)))*)(vb + v_addr[db][0] + ks * 16 * L::ROWB));
                    av.hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((short4v __attribute__((address_space(3)))*)(vb + v_addr[db][1] + ks * 16 * L::ROWB));
                    o_acc[db] = Mma<T>::run(__builtin_bit_cast(vec8, av), pb[ks], o_acc[db]);
                }
            next_v();
        }

        // ---- the four wavefronts' results meet; the next part's copies are in flight meanwhile ---------------------------
        const float l_wave = xor32_sum(l_run);
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");      // (everyone has read the last part's results)
        if (valid) {
            if (g == 0) s_ml[wave * R + ql] = float2{m_run, l_wave};
#pragma unroll
            for (int db = 0; db < NDB; ++db)
#pragma unroll
                for (int r4 = 0; r4 < 4; ++r4)
                    *(f4*)(s_o + (wave * R + ql) * D + 32 * db + 8 * r4 + 4 * g) = f4{o_acc[db][4 * r4], o_acc[db][4 * r4 + 1], o_acc[db][4 * r4 + 2], o_acc[db][4 * r4 + 3]};
        }
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
        const bool whole = out.from == 0 && !part.goes_on;
        for (int i = tid; i < R * (D / 4); i += 256) {      // four columns of a row per thread
            const int row = i / (D / 4), col = (i % (D / 4)) * 4;
            float M = -INFINITY;
#pragma unroll
            for (int w = 0; w < 4; ++w) M = fmaxf(M, s_ml[w * R + row].x);
            const float M_use = (M == -INFINITY) ? 0.0f : M;
            f4 o = {0.0f, 0.0f, 0.0f, 0.0f};
            float l_tot = 0.0f;
#pragma unroll
            for (int w = 0; w < 4; ++w) {
                const float2 ml = s_ml[w * R + row];
                const float f = __builtin_amdgcn_exp2f(ml.x - M_use);
                const f4 x = *(const f4*)(s_o + (w * R + row) * D + col);
                l_tot += ml.y * f;
#pragma unroll
                for (int e = 0; e < 4; ++e) o[e] += x[e] * f;
            }
            if (whole) {
                const int gr = Sq > 1 ? row / Sq : row, ir = row - gr * Sq, hq = hkv * p.G + gr;
                const float inv = (l_tot == 0.0f) ? __builtin_nanf("") : 1.0f / l_tot;      // no visible key: NaN, as the reference
                typedef T vec4 __attribute__((ext_vector_type(4)));
                vec4 w;
#pragma unroll
                for (int e = 0; e < 4; ++e) w[e] = (T)(o[e] * inv);
                if (col < p.Dv) *(vec4*)((T*)p.o + (int64_t)b * p.o_sb + (int64_t)hq * p.o_sh + (int64_t)ir * p.o_ss + col) = w;
                if (p.lse && col == 0)      // the row's softmax normaliser, natural log (M and the sum are in log2 units)
                    p.lse[((int64_t)b * p.Hq + hq) * Sq + ir] = l_tot == 0.0f ? -INFINITY : (M + __builtin_log2f(l_tot)) * 0.6931471805599453f;
            } else {
                const int64_t slot = deal_slot(blockIdx.x, part.goes_on, R, row);
                *(f4*)(p.ws_acc + slot * D + col) = o;
                if (col == 0) {
                    p.ws_ml[slot * 2 + 0] = M;      // log2 units, as the combine kernel takes them for 16-bit storage
                    p.ws_ml[slot * 2 + 1] = l_tot;
                }
            }
        }
        next_sequence(out, part);
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");      // (the empty copies started past the last block)
#endif
}

hipError_t launch_sdpa_combine(const SdpaParams& p, int dtype, hipStream_t stream);

template <typename T, int D, int NSLOT>
static hipError_t launch_decode_deal_t(const SdpaParams& p, hipStream_t stream)
{
    constexpr size_t ring_bytes = (size_t)4 * NSLOT * (D > 128 ? 2 * DM_SLOT_BYTES : DM_SLOT_BYTES);
    constexpr size_t most = ring_bytes + 4 * (DEAL_MAX_VALUES / D) * sizeof(float2) + 4 * DEAL_MAX_VALUES * sizeof(float);
    static_assert(most <= 160 * 1024, "a compute unit's LDS");
    const size_t lds = ring_bytes + 4 * (DEAL_MAX_VALUES / D) * sizeof(float2) + (size_t)4 * p.G * p.Sq * D * sizeof(float);
    auto kern = sdpa_decode_deal_kernel<T, D, NSLOT>;
    // the dynamic-LDS limit of this instance is raised once per device, not per launch
    static std::atomic<uint64_t> prepared{0};
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess) dev = 0;
    const uint64_t bit = 1ull << (dev & 63);
    if (!(prepared.load(std::memory_order_acquire) & bit)) {
        hipError_t e = hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)most);
        if (e != hipSuccess) return e;
        prepared.fetch_or(bit, std::memory_order_release);
    }
    hipLaunchKernelGGL(kern, dim3(p.deal), dim3(256), lds, stream, p);
    return hipGetLastError();
}
template <typename T>
static hipError_t launch_decode_deal_d(const SdpaParams& p, hipStream_t stream)
{
    const bool two = p.deal > device_cus();      // two workgroups per compute unit, of two slots per wavefront each
    if (p.Dp == 256) return launch_decode_deal_t<T, 256, 2>(p, stream);
    if (p.Dp == 128) return two ? launch_decode_deal_t<T, 128, 2>(p, stream) : launch_decode_deal_t<T, 128, 4>(p, stream);
    return two ? launch_decode_deal_t<T, 64, 2>(p, stream) : launch_decode_deal_t<T, 64, 4>(p, stream);
}

// Host has validated what launch_sdpa_decode_mfma asks for; no mask, query heads of a group x query positions x p.Dp up to 1024.
hipError_t launch_sdpa_decode_deal(const SdpaParams& p, int dtype, hipStream_t stream)
{
    const hipError_t e = dtype == 1 ? launch_decode_deal_d<f16_t>(p, stream) : launch_decode_deal_d<bf16_t>(p, stream);
    return e != hipSuccess ? e : launch_sdpa_combine(p, dtype, stream);
}

}  // namespace incin_rocm
