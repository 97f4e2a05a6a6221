// Kernel-side view of one attention launch (filled from incin_rocm_sdpa_desc_t by
// the host dispatcher after validation).  Strides are in elements.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace incin_rocm {

struct SdpaParams {
    const void* q;
    const void* k;
    const void* v;
    void* o;
    const void* mask;          // nullable dense additive mask (same dtype as q)
    const int32_t* kv_lens;    // nullable, B entries
    const int32_t* q_lens;     // nullable, B entries: query rows at and beyond are padding (output unspecified)
    float* lse;                // nullable, [B, Hq, Sq]: natural-log softmax normaliser of every row (generic and MFMA prefill kernels)
    int64_t q_sb, q_sh, q_ss;
    int64_t k_sb, k_sh, k_ss;
    int64_t v_sb, v_sh, v_ss;
    int64_t o_sb, o_sh, o_ss;
    int64_t m_sb, m_sh, m_si, m_sj;
    int32_t B, Hq, Hkv, G;     // G = Hq / Hkv
    int32_t Sq, Skv, D, Dv;
    int32_t Dp;                // matrix-core kernels: the head dimension their instance is built for (64 or 128); D and Dv fit in it, zero-padded
    float scale;
    int32_t causal;
    int32_t interleave;        // matrix-core prefill and backward kernels: (batch, KV head) pairs per group of the work list, set by their launchers
    int32_t groups;            // the same: those groups per list
    int32_t deal_groups;       // the same: how the list reaches the 8 XCDs (work_order)
    // split-KV only
    int32_t num_splits;
    int32_t split_len;         // keys per split (multiple of the kernel's key tile)
    int32_t split_turn;        // largest shift of work_split (a power of two minus one; 0: none)
    int32_t split_even;        // splits are equal shares of a batch entry's keys, not of the capacity (split_keys)
    int32_t deal;              // workgroups that the blocks of all sequences are dealt to in equal shares (decode_deal.h; 0: by splits as above)
    float* ws_acc;             // [B, Hq, Sq, num_splits, Dp] f32 partial numerators (Dp == Dv for the vector-ALU kernel); dealt: [deal, 2, G * Sq, Dp]
    float* ws_ml;              // [B, Hq, Sq, num_splits, 2]  running max (f32 natural-log domain, 16-bit log2) and denominator; dealt: [deal, 2, G * Sq, 2]
    // matrix-core prefill kernels with a dense mask: one byte per block of 32 query rows x 32 keys (0 mixed, 1 all zero,
    // 2 all -inf), written by mask_classify_kernel ahead of the attention kernel, in the caller's workspace;
    // [mask batch entries][mask heads][ceil(Sq / 32)][ceil(Skv / 32)], an extent of 1 where the mask is broadcast
    const uint8_t* mask_flags;
    // and, for the 16-bit prefill kernel, one int per mask row ([mask batch entries][mask heads][Sq, or 1 where the rows are
    // broadcast]): n if the row is n zeros followed by -inf to its end - a causal mask, key padding, both - else -1, written by
    // mask_row_limits_kernel.  A workgroup whose rows all have one needs no mask values, only the limits.  Null: not provided.
    const int32_t* mask_lims;
    int32_t lims_rows;         // rows per block of the launch that takes the blocks whose rows all have a limit (128 or 256; set by the launcher)
    int32_t mask_vec;          // 16-bit MFMA kernel: the mask's rows allow 8-byte loads of 4 consecutive keys
    int32_t mask_chunks;       // 16-bit MFMA prefill kernel: the mask's rows can be copied into LDS 16 bytes (8 keys) at a time
};

typedef __bf16 bf16_t;
typedef _Float16 f16_t;

template <typename T> __device__ __forceinline__ float to_f32(T x) { return (float)x; }
template <typename T> __device__ __forceinline__ T from_f32(float x) { return (T)x; }

// Number of keys a query row may look at, before kv_lens: causal alignment puts
// the last query on the last key (query i sees keys j <= i + Skv - Sq).
__device__ __forceinline__ int causal_limit(int i, int Sq, int Skv) { return i + (Skv - Sq) + 1; }

__device__ __forceinline__ int clampi(int x, int lo, int hi) { return x < lo ? lo : (x > hi ? hi : x); }

// Blocks that one launch may have: its work-items along an axis stay below 2^32.  Kernels whose items are small, or that hold those of two or
// three gradients in one launch, pass that with very many small heads, and are then launched twice or
// more (in multiples of 8: a block stays on the XCD it would have been on).
constexpr int64_t max_blocks(int threads) { return (1ll << 32) / threads - 8; }

// Where the block flags of (batch b, query head hq) start, and the flags per row of blocks.
__device__ __forceinline__ const uint8_t* mask_flags_of(const SdpaParams& p, int b, int hq)
{
    const int nkb = (p.Skv + 31) / 32, nrb = (p.Sq + 31) / 32;
    const int Hm = p.m_sh ? p.Hq : 1;
    const int64_t bh = (int64_t)(p.m_sb ? b : 0) * Hm + (p.m_sh ? hq : 0);
    return p.mask_flags + bh * nrb * nkb;
}

// Where the row limits of (batch b, query head hq) start.
__device__ __forceinline__ const int32_t* mask_lims_of(const SdpaParams& p, int b, int hq)
{
    const int Hm = p.m_sh ? p.Hq : 1;
    const int64_t bh = (int64_t)(p.m_sb ? b : 0) * Hm + (p.m_sh ? hq : 0);
    return p.mask_lims + bh * (p.m_si ? p.Sq : 1);
}

// Which split of the keys a workgroup of a split-KV launch takes (grid: x splits, y and z groups; group is the (batch, KV head)
// pair): x, shifted from group to group by up to split_turn where the launcher asks for that.
// Workgroups reach the 8 XCDs round-robin in dispatch order, so an even number of splits by itself gives an XCD the
// same few splits of every group; with key counts the last splits of short sequences are empty, and the XCDs that hold them run
// out of work.  There split_turn is d - 1 with d = 2, 4 or 8 the power of two in the
// number of splits; g + g / 2 + g / 4 takes every such value whatever g is modulo 2, 4 or 8.  Counts spread from an eighth of the
// capacity to all of it, us before and after: 33 sequences x 8 KV heads x 4096 x 64 (8 splits) 39.7 -> 29.6, 24 31.2 -> 25.4, 16 x 2 x 32768 x
// 128 (8) 68.3 -> 59.4, 8 x 8 x 8192 x 128 (8) 39.1 -> 34.8, f32 8 x 8 x 4096 39.7 -> 36.3, 64 x 1 x 60000 (4) 196 -> 182; 4 sequences level, 2 or 3
// have little to balance (17.0 / 17.5) and are left alone.  (The host decides: worked out by every workgroup, the rule cost the
// launches that it leaves alone 0.2 - 0.5 us - 8 x 1 x 60000 44.7 without it, 45.3 so, 44.7 now; 8 x 12 x 2048 x 256 50.7 / 51.0 / 50.8.)
inline int split_turn_of(bool key_counts, int B, int num_splits)
{
    const int d = num_splits & -num_splits;
    return key_counts && B >= 4 && num_splits > 1 ? (d < 8 ? d : 8) - 1 : 0;
}
// Which keys of a batch entry with kv_len of them a split holds: split_len of the capacity's, or - split_even_of says where - an equal share of
// those there are, in whole blocks of `unit` keys.
struct KeyRange { int begin, end; };
__device__ __forceinline__ KeyRange split_keys(const SdpaParams& p, int split, int kv_len, int unit)
{
    KeyRange r;
    if (p.split_even) {
        const int blocks = (kv_len + unit - 1) / unit, each = blocks / p.num_splits, more = blocks - each * p.num_splits;
        r.begin = (each * split + min(split, more)) * unit;      // (the first `more` splits take one block more)
        r.end = min(r.begin + (each + (split < more ? 1 : 0)) * unit, kv_len);
    } else {
        r.begin = split * p.split_len;
        r.end = min(r.begin + p.split_len, kv_len);
    }
    return r;
}
// Equal shares where one round of workgroups is the whole launch (`one_round`), so that its longest is what the launch takes, and the
// splits are short (`split_bytes` of K: 256 KiB at most), so that a workgroup is bound by its own latencies and not by the memory system - there
// splits of one length are the better ones: those of short sequences that are empty leave their bandwidth to the others, and all
// end together.  From 8 sequences on the shift above balances as well.  Bf16, us, splits of the capacity / equal shares: 32 on 8 heads x 4 sequences of 3000 - 16000
// keys 34.0 / 29.8, 2 of 4096 - 32768 at D = 64 20.8 / 17.3, 3 x 4 x 832 - 2386 11.8 / 10.4, 6 x 8 x 1650 - 2037 19.8 / 18.6, f32 1 x 2 x 2058 18.4 / 14.7, one of 407 at D = 256 17.5 /
// 15.4; but 8 x 8 x 1024 - 8192 31.8 / 32.2, 16 x 8 x 512 - 4096 31.8 / 32.9, 4 x 8 x 7000 - 60000 (7500 a split) 95 / 101, 2 x 2 x 10000 - 29999 at D = 256 27.2 / 27.5.
inline int split_even_of(bool key_counts, int B, int num_splits, bool one_round, int64_t split_bytes, int Dp)
{
    return key_counts && num_splits > 1 && one_round && split_bytes <= (256 << 10) && B < (Dp > 128 ? 2 : 8);
}
__device__ __forceinline__ int work_split(const SdpaParams& p, int group)
{
    const int x = blockIdx.x;
    if (p.split_turn == 0) return x;
    const int y = x + ((group + (group >> 1) + (group >> 2)) & p.split_turn);
    return y >= p.num_splits ? y - p.num_splits : y;
}

}  // namespace incin_rocm
