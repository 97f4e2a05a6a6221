// bf16 / f16 attention forward on the gfx950 matrix cores where the keys of a head fit into LDS at once: up to 256 keys at head
// dimensions up to 64, up to 128 at head dimensions up to 128 (encoders and vision models with many short sequences, cross
// attention over a short text).  The function of the reference CPU composition
// (crates/incin-backends/src/cpu/ops/shape_ops.rs:1245-1269), optional causal flag, per-batch key and query lengths, MHA and GQA, no mask
// tensor; the operand layouts are those of sdpa_prefill_mfma.hip.
//
// Such a launch is bound by memory: 64 x 12 heads x 197 x 64 are 78 MB of Q, K, V and O for 6 us of matrix instructions.  The
// kernel for long sequences walks the keys in tiles of 64 behind a barrier each, with the next tile's copies one tile ahead: its
// workgroups live for two to four tiles and wait for memory five times in a row.  Here everything a workgroup reads is asked
// for at once - all K and V rows by global -> LDS copies, its first Q rows beside them - and awaited once; the one barrier is
// the one behind that.  Then every wavefront works alone: 32 query rows at a time (all heads of a group in turn), the scores of
// all keys that the rows see in registers (16 per 32 keys: no online softmax, the maximum is exact), exponentials between the
// products; the next rows' Q fetched meanwhile.  Heads of up to 32 or 64 rows and keys come four or two to a workgroup, a
// wavefront or two each, so that no wavefront idles.
//
// Measured against that kernel (f16 / bf16; us a call, calls back to back): 64 x 12 heads x 197 x 64 28.8 -> 25.1 (3.1 TB/s), 256 x 12 x 197 111 -> 90,
// 256 x 16 x 64 39.4 -> 26.3 (5.1 TB/s), 256 x 12 x 17 28.0 -> 8.7, 119 x 16 x 43 x 128 29.6 -> 18.9, 64 x 32 / 8 x 128 x 128 causal 45.9 -> 35.7,
// 32 x 12 x 224 causal 17.4 -> 14.5, 8 x 32 x 4096 rows over 77 keys 105 -> 73; behind it by up to a fifth in the launches that
// tiles_are_ahead names, which stay with it.
#include <algorithm>
#include <type_traits>

#include "sdpa_mfma_common.h"

namespace incin_rocm {

// NBM: blocks of 32 keys that the scores of an item may take (registers); `nb` of them are what this launch's keys need (LDS).
// WPP wavefronts of a workgroup share a (batch, KV head) pair, 4 / WPP pairs a workgroup; with WPP = 4 `chunks` workgroups share
// a pair's 32-row items.
template <typename T, int D, int NBM, int WPP>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2, 2))) void sdpa_prefill_short_kernel(SdpaParams p, int nb, int chunks)
{
#if defined(__HIP_DEVICE_COMPILE__)
    typedef typename Mma<T>::vec8 vec8;
    typedef PfLayout<D> L;
    constexpr int NSTEP = D / 16, NDB = D / 32, NQH = D / 64, R = 4;
    constexpr int BLK = 32 * L::ROWB, LPB = BLK / 1024 / WPP;      // bytes of a block of 32 keys; wavefront-wide 1 KiB copies of it per wavefront
    extern __shared__ __attribute__((aligned(1024))) char smem[];      // 4 KiB per wavefront for rows in and out; per pair: K, V

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int sub = wave / WPP, wsub = wave % WPP;      // which pair of the workgroup, which of its wavefronts
    const int ql = lane & 31, g = lane >> 5;
    const int Sq = p.Sq, Skv = p.Skv, coff = Skv - Sq;
    // a pair's workgroups on one XCD, whose L2 then serves its K and V rows to all of them
    const int pairs = p.B * p.Hkv;
    int pair, chunk = 0;
    if (WPP < 4) pair = blockIdx.x * (4 / WPP) + sub;
    else if ((pairs & 7) == 0) {
        const int slot = blockIdx.x >> 3;
        chunk = slot % chunks;
        pair = (slot / chunks) * 8 + (blockIdx.x & 7);
    } else {
        chunk = blockIdx.x % chunks;
        pair = blockIdx.x / chunks;
    }
    const bool real = WPP == 4 || pair < pairs;      // (the last workgroup's pairs beyond the last one: nothing to do but the barrier)
    pair = min(pair, pairs - 1);
    const int hkv = pair % p.Hkv, b = pair / p.Hkv;
    const int kv_len = p.kv_lens ? clampi(p.kv_lens[b], 0, Skv) : Skv;
    const int rows_b = p.q_lens ? clampi(p.q_lens[b], 0, Sq) : Sq;
    // items of 32 rows: blocks of a head, then the group's next head; this wavefront's are item0, item0 + step, ...
    const int nblk = (rows_b + 31) >> 5, items = real ? nblk * p.G : 0;
    const int item0 = chunk * WPP + wsub, step = WPP * chunks;
    if (WPP == 4 && chunk * WPP >= items) return;      // (uniform)

    const T* kp = (const T*)p.k + (int64_t)b * p.k_sb + (int64_t)hkv * p.k_sh;
    const T* vp = (const T*)p.v + (int64_t)b * p.v_sb + (int64_t)hkv * p.v_sh;
    char* const stage = smem + wave * 4096;
    char* const kbuf = smem + 4 * 4096 + sub * 2 * nb * BLK;
    char* const vbuf = kbuf + nb * BLK;

    auto row0_of = [&](int item) { return (item % nblk) * 32; };
    auto q_of = [&](int item) { return (const T*)p.q + (int64_t)b * p.q_sb + (int64_t)(hkv * p.G + item / nblk) * p.q_sh; };
    uint4v qraw[NQH][4];
    if (item0 < items) fetch_q_rows(qraw, q_of(item0), row0_of(item0), Sq, p.q_ss, p.D, lane);
    if (items > 0) {
        int k_voff[LPB], v_voff[LPB];
#pragma unroll
        for (int c = 0; c < LPB; ++c) {
            const int pos = (wsub * LPB + c) * 64 + lane, row = pos / L::CPR, slot = pos % L::CPR;
            k_voff[c] = dma_chunk_offset(row, (int)p.k_ss * 2, slot ^ L::fk(row), p.D * 2);
            v_voff[c] = dma_chunk_offset(row, (int)p.v_ss * 2, slot ^ L::fv(row), p.Dv * 2);
        }
        // all blocks the sequence has keys in (rows beyond its last key arrive as zeros)
        auto copy = [&](const T* base, int64_t stride, int width, char* dst, const int (&voff)[LPB]) __attribute__((always_inline)) {
#pragma unroll
            for (int k = 0; k < NBM; ++k)
                if (k * 32 < kv_len) {
                    const int64_t rem = (int64_t)(kv_len - k * 32 - 1) * stride * 2 + width * 2;
                    const uint4v r = dma_descriptor(base + (int64_t)k * 32 * stride, (int)(rem > 0x7fffffffLL ? 0x7fffffffLL : rem));
#pragma unroll
                    for (int c = 0; c < LPB; ++c) dma_copy16(r, lds_address(dst) + k * BLK + (wsub * LPB + c) * 1024, voff[c]);
                }
        };
        copy(kp, p.k_ss, p.D, kbuf, k_voff);
        copy(vp, p.v_ss, p.Dv, vbuf, v_voff);
    }

    // operand addresses: K row ql of a block, chunk 2 s + g; V transposed, column block db, half h of 16 rows
    int k_addr[NSTEP], v_addr[NDB][2];
#pragma unroll
    for (int s = 0; s < NSTEP; ++s) k_addr[s] = ql * L::ROWB + (((2 * s + g) ^ L::fk(ql)) << 4);
    {
        const int n = lane & 15, dh = (lane >> 4) & 1;
#pragma unroll
        for (int db = 0; db < NDB; ++db)
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const int r = 8 * h + 4 * g + (n >> 2), c = 4 * db + 2 * dh + ((n & 3) >> 1);
                v_addr[db][h] = r * L::ROWB + ((c ^ L::fv(r)) << 4) + (n & 1) * 8;
            }
    }
    const float c2 = p.scale * 1.4426950408889634f;

    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    if (WPP > 1) __syncthreads();

    for (int item = item0; item < items; item += step) {
        const int row0 = row0_of(item), my_i = row0 + ql;
        const int hq = hkv * p.G + item / nblk;
        vec8 qreg[NSTEP];
        stage_q_rows(qreg, qraw, stage, lane);
#pragma unroll
        for (int s = 0; s < NSTEP; ++s)
#pragma unroll
            for (int e = 0; e < 8; ++e) qreg[s][e] = (T)((float)qreg[s][e] * c2);
        if (item + step < items) fetch_q_rows(qraw, q_of(item + step), row0_of(item + step), Sq, p.q_ss, p.D, lane);
        // this lane's key count, the item's smallest and largest
        const int lim = p.causal ? clampi(my_i + coff + 1, 0, kv_len) : kv_len;
        const int lim_min = p.causal ? clampi(row0 + coff + 1, 0, kv_len) : kv_len;
        const int lim_max = p.causal ? clampi(min(row0 + 31, rows_b - 1) + coff + 1, 0, kv_len) : kv_len;

        floatx16 o_acc[NDB];
#pragma unroll
        for (int db = 0; db < NDB; ++db)
#pragma unroll
            for (int r = 0; r < 16; ++r) o_acc[db][r] = 0.0f;
        float m = -INFINITY, l_tot = 0.0f;
        // An item whose rows see keys in the first NB blocks: straight-line code for each count, so that operands are read ahead
        // and vector work sits between matrix instructions across the blocks.
        auto attend = [&](auto NB_) __attribute__((always_inline)) {
            constexpr int NB = decltype(NB_)::value;
            // ---- S^T = K Q^T, all keys (LDS operands R matrix instructions ahead) ----
            floatx16 sc[NB];
            {
                vec8 ring[R];
                auto fetch = [&](int i) __attribute__((always_inline)) { ring[i % R] = *(const vec8*)(kbuf + (i / NSTEP) * BLK + k_addr[i % NSTEP]); };
#pragma unroll
                for (int i = 0; i < R; ++i) fetch(i);
#pragma unroll
                for (int k = 0; k < NB; ++k)
#pragma unroll
                    for (int r = 0; r < 16; ++r) sc[k][r] = 0.0f;
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int i = 0; i < NB * NSTEP; ++i) {
                    sc[i / NSTEP] = Mma<T>::run(ring[i % R], qreg[i % NSTEP], sc[i / NSTEP]);
                    if (i + R < NB * NSTEP) fetch(i + R);
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
            // register r of block k is key 32 k + 8 (r / 4) + 4 g + r % 4
            const int rel = lim - 4 * g;
#pragma unroll
            for (int k = 0; k < NB; ++k)
                if (lim_min < 32 * (k + 1)) {      // (uniform) some row of the item does not see all of the block
#pragma unroll
                    for (int r = 0; r < 16; ++r)
                        if (32 * k + 8 * (r / 4) + (r % 4) >= rel) sc[k][r] = -INFINITY;
                }
            m = sc[0][0];
#pragma unroll
            for (int k = 0; k < NB; ++k)
#pragma unroll
                for (int r = 0; r < 16; ++r) m = fmaxf(m, sc[k][r]);
            m = xor32_max(m);
            const float m_use = m == -INFINITY ? 0.0f : m;

            // ---- P^T block by block, each between the products of the one before: O^T += V^T P^T ----
            float rsum = 0.0f;
            uint4v pb[2][2];      // [block parity][half of 16 keys]
            auto soft = [&](int k, int r) __attribute__((always_inline)) {      // registers r, r + 1
                const unsigned w = pinned(pack2<T>(__builtin_amdgcn_exp2f(sc[k][r] - m_use), __builtin_amdgcn_exp2f(sc[k][r + 1] - m_use)));
                pb[k % 2][r / 8][(r % 8) / 2] = w;
                rsum = Mma<T>::add2(__builtin_bit_cast(typename Mma<T>::vec2, w), rsum);
            };
            constexpr int NPV = 2 * NDB;      // matrix instructions of a block
            vec8 ring[R];
            auto fetch = [&](int i) __attribute__((always_inline)) {      // i = (block, half, column block)
                const int k = i / NPV, h = (i / NDB) % 2, db = i % NDB;
                short8v av;
                av.lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((short4v __attribute__((address_space(3)))*)(vbuf + v_addr[db][0] + k * BLK + h * 16 * L::ROWB));
                av.hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((short4v __attribute__((address_space(3)))*)(vbuf + v_addr[db][1] + k * BLK + h * 16 * L::ROWB));
                ring[i % R] = __builtin_bit_cast(vec8, av);
            };
#pragma unroll
            for (int i = 0; i < R; ++i) fetch(i);
#pragma unroll
            for (int r = 0; r < 16; r += 2) soft(0, r);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int i = 0; i < NB * NPV; ++i) {
                const int k = i / NPV, m2 = i % NPV;
                o_acc[i % NDB] = Mma<T>::run(ring[i % R], __builtin_bit_cast(vec8, pb[k % 2][m2 / NDB]), o_acc[i % NDB]);
                if (i + R < NB * NPV) fetch(i + R);
                if (k + 1 < NB) {
#pragma unroll
                    for (int r = m2 * (16 / NPV); r < (m2 + 1) * (16 / NPV); r += 2) soft(k + 1, r);
                }
                __builtin_amdgcn_sched_barrier(0);
            }
            l_tot = xor32_sum(rsum);
        };
        switch ((lim_max + 31) >> 5) {
            case 0: break;
            case 1: attend(std::integral_constant<int, 1>{}); break;
            case 2: if constexpr (NBM >= 2) attend(std::integral_constant<int, 2>{}); break;
            case 3: if constexpr (NBM >= 3) attend(std::integral_constant<int, 3>{}); break;
            case 4: if constexpr (NBM >= 4) attend(std::integral_constant<int, 4>{}); break;
            case 5: if constexpr (NBM >= 5) attend(std::integral_constant<int, 5>{}); break;
            case 6: if constexpr (NBM >= 6) attend(std::integral_constant<int, 6>{}); break;
            case 7: if constexpr (NBM >= 7) attend(std::integral_constant<int, 7>{}); break;
            default: if constexpr (NBM >= 8) attend(std::integral_constant<int, 8>{}); break;
        }
        const float inv = l_tot == 0.0f ? __builtin_nanf("") : 1.0f / l_tot;      // no visible key: NaN, as the reference
        if (p.lse && g == 0 && my_i < rows_b)
            p.lse[((int64_t)b * p.Hq + hq) * Sq + my_i] = l_tot == 0.0f ? -INFINITY : (m + __builtin_log2f(l_tot)) * 0.6931471805599453f;
        store_o_rows(o_acc, inv, stage, (T*)p.o + (int64_t)b * p.o_sb + (int64_t)hq * p.o_sh, row0, rows_b, p.o_ss, p.Dv, lane);
    }
#endif
}

template <typename T, int D, int NBM, int WPP>
static hipError_t launch_short(const SdpaParams& p, int nb, int64_t pairs, int chunks, hipStream_t stream)
{
    constexpr int PPW = 4 / WPP;      // pairs per workgroup
    const size_t lds = 4 * 4096 + (size_t)PPW * 2 * nb * 32 * PfLayout<D>::ROWB;
    auto* kernel = sdpa_prefill_short_kernel<T, D, NBM, WPP>;
    if (lds > 65536) {      // (more dynamic LDS than a kernel may ask for by default; set once per device and instance)
        static std::atomic<unsigned long long> done{0};
        int dev = 0;
        hipError_t e = hipGetDevice(&dev);
        if (e != hipSuccess) return e;
        if (dev >= 64 || !(done.load(std::memory_order_relaxed) >> dev & 1)) {
            e = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, 4 * 4096 + PPW * 2 * NBM * 32 * PfLayout<D>::ROWB);
            if (e != hipSuccess) return e;
            if (dev < 64) done.fetch_or(1ull << dev, std::memory_order_relaxed);
        }
    }
    hipLaunchKernelGGL(kernel, dim3((unsigned)((pairs + PPW - 1) / PPW * chunks)), dim3(256), lds, stream, p, nb, chunks);
    return hipGetLastError();
}
template <typename T>
static hipError_t launch_short_t(const SdpaParams& p, int64_t pairs, int64_t items, int chunks, hipStream_t stream)
{
    const int nb = (p.Skv + 31) / 32;
    if (p.Dp == 128) {
        if (nb == 1 && items == 1) return launch_short<T, 128, 1, 1>(p, nb, pairs, 1, stream);
        if (nb <= 2) return items <= 2 ? launch_short<T, 128, 2, 2>(p, nb, pairs, 1, stream) : launch_short<T, 128, 2, 4>(p, nb, pairs, chunks, stream);
        return launch_short<T, 128, 4, 4>(p, nb, pairs, chunks, stream);
    }
    if (nb == 1 && items == 1) return launch_short<T, 64, 1, 1>(p, nb, pairs, 1, stream);
    if (nb <= 2) return items <= 2 ? launch_short<T, 64, 2, 2>(p, nb, pairs, 1, stream) : launch_short<T, 64, 2, 4>(p, nb, pairs, chunks, stream);
    if (nb <= 4) return launch_short<T, 64, 4, 4>(p, nb, pairs, chunks, stream);
    return launch_short<T, 64, 8, 4>(p, nb, pairs, chunks, stream);
}

// Workgroups per pair: as many as give every compute unit two, at most one item per wavefront; more only read K and V more often
// (in us, by chunks: 8 x 12 heads x 197 keys 7.8 with 2, 10.5 with 1; 8 x 16 x 4096 rows over 77 keys at D = 128 66 / 62 / 57 / 66 / 108 with
// 32 / 8 / 4 / 2 / 1; 64 x 12 x 197 27.8 with 2, 25 with 1).
static int64_t short_chunks(int64_t pairs, int64_t items) { return std::min((items + 3) / 4, std::max<int64_t>(1, (2 * (int64_t)device_cus() + pairs - 1) / pairs)); }

// Which of the launches whose keys fit come here: all but those that the kernel that walks tiles of 64 keys is ahead on.  That one's
// workgroups are lighter - more of them on a compute unit - and where its last tile is nearly full and no wavefront here has a
// second item whose Q rows arrive under the first, nothing is left to gain (us, tiles / here, bf16, no mask):
//   D <= 64, 185 - 192 or 225 - 256 keys, one item per wavefront: 8 x 16 x 192 6.2 / 6.5, 20 x 16 x 192 11.9 / 12.7, 16 x 16 x 256 9.4 / 9.9, 8 x
//     32 / 8 x 192 8.2 / 8.8; or a last round of workgroups at most a quarter full: 36 x 16 x 256 22.1 / 23.5, 66 x 16 x 256 36.1 / 37.0 (but
//     32 x 16 x 256 19.3 / 17.4, 42 x 16 x 192 20.4 / 19.2, 20 x 16 x 161 13.3 / 13.0; with a causal mask 16 x 16 x 256 9.8 / 9.3);
//   D <= 64, more than 160 keys, at most 128 rows, more than a round: 64 x 16 x 64 rows over 256 keys 17.6 / 21.4, over 200 18.0 / 19.4 (over 160
//     16.6 / 16.1);
//   D > 64, 97 - 128 keys, at most 128 rows, more than a round: 64 x 16 x 128 25.0 / 26.2, 48 x 16 20.7 / 21.6, causal 20.7 / 21.3; level from seven
//     workgroups per compute unit on (128 x 16 46.9 / 46.3), and D <= 96, whose products are the fewer there, from one to ten: 64 x 16 x
//     128 x 96 22.3 / 24.0, 18 x 16 8.7 / 9.2 (160 x 16 50.9 / 51.0; 64 x 16 x 100 x 80 19.3 / 19.2); 49 - 64 keys under 97 - 128 rows 19.2 / 20.4.
static bool tiles_are_ahead(const SdpaParams& p)
{
    const int64_t cus = device_cus(), pairs = (int64_t)p.B * p.Hkv, items = ((int64_t)(p.Sq + 31) / 32) * p.G;
    if (3 * p.G * ((p.Sq + 127) / 128) > 4 * ((items + 3) / 4)) return false;      // (its blocks of 128 rows of one head would be half empty)
    if (p.Dp == 64) {
        if (p.causal || p.Skv <= 160) return false;
        if (items <= 4 && pairs > 2 * cus) return true;
        if (!(p.Skv > 224 || (p.Skv > 184 && p.Skv <= 192))) return false;
        const int64_t chunks = short_chunks(pairs, items), round = 2 * cus, blocks = pairs * chunks, last = blocks % round;
        return 4 * chunks >= items || (blocks > round && blocks < 3 * round && last > 0 && 4 * last <= round);
    }
    if (items > 4) return false;
    const bool wide = p.D > 96 || p.Dv > 96;
    if (pairs <= (wide || p.causal ? 2 : 1) * cus || pairs >= (wide ? 7 : 10) * cus) return false;
    if (p.Skv > (p.causal ? 112 : wide ? 96 : 100)) return p.Sq > 32;
    return !p.causal && p.Skv > 48 && p.Skv <= 64 && p.Sq > 96 && pairs > 2 * cus;
}
bool prefill_short_fits(const SdpaParams& p)
{
    return !p.mask && p.num_splits <= 1 && p.Skv >= 1 && p.Skv <= (p.Dp == 64 ? 256 : 128) && p.Dp <= 128 && !tiles_are_ahead(p);
}

// Host has validated what sdpa_prefill_mfma.hip asks for; the keys fit (prefill_short_fits).
hipError_t launch_sdpa_prefill_short(const SdpaParams& p, int dtype, hipStream_t stream)
{
    const int64_t pairs = (int64_t)p.B * p.Hkv;
    const int64_t items = ((int64_t)(p.Sq + 31) / 32) * p.G;      // 32-row items of a pair
    const int64_t chunks = short_chunks(pairs, items);
    if (pairs * chunks > 0x7fffffffLL) return hipErrorInvalidValue;
    return dtype == 1 ? launch_short_t<f16_t>(p, pairs, items, (int)chunks, stream) : launch_short_t<bf16_t>(p, pairs, items, (int)chunks, stream);
}

}  // namespace incin_rocm
