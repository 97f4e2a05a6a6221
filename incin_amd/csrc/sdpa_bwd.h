// Launch parameters of the attention backward kernels (sdpa_bwd_mfma.hip, sdpa_bwd_f32.hip, sdpa_bwd_generic.hip), shared with the C ABI layer.
#pragma once
#include <hip/hip_runtime.h>

#include "sdpa_params.h"

namespace incin_rocm {

struct SdpaBwdParams {
    SdpaParams f;                  // the forward's operands and masks; f.o = the forward's output, f.lse = its normalisers
    const void* d_o;               // upstream gradient, [B, Hq, Sq, D] by strides
    void* d_q;
    void* d_k;
    void* d_v;
    float* neg_l2;                 // workspace, [B, Hq, Sq]: -L_i log2(e) (the normalisers, negated, in log2 units)
    float* neg_delta;              // workspace, [B, Hq, Sq]: -D_i = -(dO_i . O_i)
    int32_t dots_in_dq;            // 16-bit matrix-core kernels up to 128: the dQ kernel computes the two rows above (it runs first), else a kernel of its own
    int64_t do_sb, do_sh, do_ss;
    int64_t dq_sb, dq_sh, dq_ss;
    int64_t dk_sb, dk_sh, dk_ss;
    int64_t dv_sb, dv_sh, dv_ss;
    // Matrix-core kernels where the longest walk would decide when the launch ends: the key tiles of a dQ workgroup are dealt to
    // parts_q workgroups (f32 only), the query tiles of a dK/dV workgroup to parts_kv (1, 2, 4; 16-bit storage also 8).  The sums meet in
    // planes of the workspace - contiguous f32 copies of the gradient's shape - and a pass behind the kernel adds them in
    // order.  f32: part 0 writes the gradient's rows itself and part k > 0 plane k - 1, which the pass adds to the rows; 16-bit
    // storage: every part writes a plane, and the pass rounds their sum into the rows.
    int32_t parts_q, parts_kv;
    int32_t split;                 // f32: the kernel whose values are three bf16 parts (sdpa_bwd_f32_split.hip) takes the call
    int32_t share;                 // f32: wavefronts of a workgroup that share a block's walk (1, 2 or 4)
    float* part_dq;                // workspace, f32: [parts_q - 1][B, Hq, Sq, D]
    float* part_dk;                // workspace, f32: [parts_kv - 1][B, Hkv, Skv, D]; 16-bit storage: [parts_kv][...]
    float* part_dv;                // workspace, likewise [..][B, Hkv, Skv, Dv]
};

// 16-bit storage up to head dimension 128, the rules that the planner of the workspace and the launcher share.
//   blocks: 128-key blocks of all (batch, KV head) pairs; walk: 64-row query tiles of a block's walk over its group's heads.
//
// Which dK/dV kernel.  Head dimensions up to 96 without a mask tensor: the kernel with one wavefront per 32 keys (the other
// pairs them) wherever there is more than one workgroup per compute unit to cover its latencies or the walks can be dealt to
// more: 8 x 32 heads x 4096, causal, whole call 2.32 -> 1.80 ms, 32 x 12 x 512 144 -> 96 us.  A launch of one query head per KV head
// that gives it less than a workgroup per compute unit, for walks of some length, keeps the paired kernel, whose eight
// wavefronts per 128 keys are twice as many (8 heads x 2048 62 us against 70, 4 x 4096 94 against 106; at 16 tiles 48 against 44).
// From 65 to 96 likewise, from walks of 12 tiles on (paired / narrow: 60 x 12 x 400 at 80 289 / 216 us, 87 x 16 x 98 98 / 83, 8 x 16 x 2553 at 96 causal
// 719 / 605, 8 x 32 x 220 47 / 36, 2 x 32 on 8 x 2000 228 / 207; 2 heads x 5224 139 / 162, 16 x 1000 50 / 56).
inline bool bwd16_narrow(int64_t D, int64_t Dv, bool mask, int64_t G, int64_t blocks, int64_t walk, int64_t cus)
{
    return D <= 96 && Dv <= 96 && !mask && (G > 1 || blocks >= cus || walk < (D <= 64 && Dv <= 64 ? 32 : 12));
}
// Whether the dQ kernel runs on a stream of its own beside the dK/dV kernel.  The fork and the join cost 5 - 7 us, and the call a
// kernel for the row dots, which the dQ kernel computes where it runs first (8 x 16 heads x 256, D = 64: 40 us forked, 21 in
// order; 4 x 16 x 512, D = 128: 69 and 47).  It pays where the dK/dV kernel leaves compute units idle for long enough:
//   paired kernel (one workgroup fills a compute unit): at most half the compute units (8 x 2048, D = 128: 78 forked, 111 in
//   order; 16 x 1024 57 / 67; from 12 tiles of walk on: 12 x 768 48 / 55, 8 x 512 44 / 42); under a causal mask, whose blocks end
//   at different times, up to two rounds of workgroups with walks of 32 tiles (64 when they are dealt) if the dQ launch is at
//   most two rounds too - of 16 tiles up to one and a half rounds, undivided: the second one leaves half of the compute units idle (40 x 1024 84 / 89,
//   48 x 1024 88 / 92, 56 x 1024 113 / 105) - (8 x 8192 457 / 488, 2 x 32 / 8 x 2048 268 / 309, 16 / 4 x 2048 in 4 parts 145 / 126, 64 / 8 x 4096 975 / 891;
//   without a mask 8 x 8192 942 / 823);
//   the other: grouped queries with walks of 32 tiles and at most three key blocks per compute unit (training steps, D = 64: 64 on 8 x 4096 617 / 669, 2 x 64 on 8 x
//   4096 1183 / 1263, 2 x 32 on 8 x 2048 208 / 229, 8 x 32 on 8 x 1024 208 / 213, but 8 x 32 on 8 x 2048 660 / 644); without, under a causal mask, two and a quarter
//   with walks of 44, one and a half of 32 (8 x 8192 368 / 399, 12 x 4096 185 / 197, 2 x 12 x 3000 161 / 164, 2 x 8 x 2048 98 / 104, but 2 x 16 x 2048 119 / 114, 4 x 16 x 2048
//   196 / 183, 2 x 16 x 4096 337 / 317, 8 x 16 x 4096 1218 / 1183; D = 96: 12 x 4096 223 / 263, 4 x 16 x 4096 921 / 882; neither: 32 x 12 x 512 118 / 103, 2 x 16 x 2048 135 / 121).
inline bool bwd16_forks(bool narrow, bool causal, int64_t G, int64_t blocks, int64_t parts, int64_t walk, int64_t dq_blocks, int64_t cus)
{
    const int64_t w = walk / parts;
    if (narrow && G > 1) return w >= 32 && blocks <= 3 * cus;
    if (narrow) return causal && ((w >= 44 && 4 * parts * blocks <= 9 * cus) || (w >= 32 && 2 * parts * blocks <= 3 * cus));
    if (2 * parts * blocks <= cus && w >= 12) return true;
    if (causal && parts == 1 && blocks > cus && 2 * blocks <= 3 * cus && dq_blocks <= 2 * cus && w >= 16) return true;
    return causal && parts * blocks <= 2 * cus && dq_blocks <= 4 * cus && w >= (parts > 1 ? 64 : 32);
}

hipError_t launch_sdpa_bwd_mfma(const SdpaBwdParams& bp, int dtype, hipStream_t stream);
hipError_t launch_sdpa_bwd_wide(const SdpaBwdParams& bp, int dtype, hipStream_t stream);
// (of sdpa_bwd_mfma.hip: the row dots, and the sum of the planes of a call with parts_kv > 1 into dK and dV)
hipError_t launch_sdpa_bwd_delta(const SdpaBwdParams& bp, int dtype, hipStream_t stream);
hipError_t launch_sdpa_bwd_sum_planes(const SdpaBwdParams& bp, int dtype, hipStream_t stream);
hipError_t launch_sdpa_bwd_f32(const SdpaBwdParams& bp, hipStream_t stream);
hipError_t launch_sdpa_bwd_f32_split(const SdpaBwdParams& bp, hipStream_t stream);
hipError_t launch_sdpa_bwd_generic(const SdpaBwdParams& bp, int dtype, hipStream_t stream);

}  // namespace incin_rocm
