// Classifies a dense additive mask by blocks of 32 query rows x 32 keys, ahead of a matrix-core attention launch:
//   0  mixed     the block's values have to be added to the scores
//   1  zeros     every value is 0: the block needs no mask at all
//   2  hidden    every value is -inf: no key of the block is visible to any of its rows, the block is skipped
// The reference's operator knows one mask form, an additive tensor (crates/incin-backends/src/cpu/ops/shape_ops.rs:
// 1262-1266), and its callers build the causal mask as full(-inf).triu(1): with the flags, such a tensor costs about
// what the causal flag costs - blocks above the diagonal are skipped, blocks below it run the unmasked path.
// One workgroup per strip of 32 rows x 256 keys (8 blocks): a thread takes 8 consecutive keys of 4 rows - 16-byte
// loads for masks with unit key stride, element-wise loads otherwise and at the end of a row - and the votes of a
// block meet in LDS; rows beyond Sq and keys beyond Skv do not vote.
#include "sdpa_mfma_common.h"

namespace incin_rocm {

// Eight consecutive values of a mask's row in one load, wherever the row starts: the type asks for no more than an element's alignment, and
// the compiler takes 16-byte loads for it, which the memory path allows at any address.  (By elements where rows were not multiples of 32 bytes:
// whole call, f32, a bias per head, 8 heads x 1001 x 1001 134 -> 123 us, bf16 12 x 801 x 801 98 -> 85, 32 x 900 x 900 64 -> 60.)
template <typename T> struct Mask8 { typedef T type __attribute__((ext_vector_type(8), aligned(sizeof(T)))); };
// The values of keys j0 .. j0 + 7 that a row has, as elements from .. 7 of what is returned; key j0 exists.  VEC (unit key stride, eight keys
// or more): at the end of the row the eight before it, so that nothing is read one element after the other there.
template <typename T> struct RowPart {
    T x[8];
    int first_key, from;      // element e is key first_key + e; the first `from` belong to whoever has the eight keys before
};
template <typename T, bool VEC> __device__ __forceinline__ RowPart<T> row_part(const T* row, int64_t m_sj, int j0, int Skv)
{
    RowPart<T> r;
    if constexpr (VEC) {
        r.first_key = min(j0, Skv - 8);
        r.from = j0 - r.first_key;
        const typename Mask8<T>::type v = *(const typename Mask8<T>::type*)(row + r.first_key);
#pragma unroll
        for (int e = 0; e < 8; ++e) r.x[e] = v[e];
    } else {
        // (key by key; the n that there are take the last n places, key j0 fills the others)
        const int n = min(8, Skv - j0);
        r.first_key = j0 + n - 8;
        r.from = 8 - n;
#pragma unroll
        for (int e = 0; e < 8; ++e) r.x[e] = row[(int64_t)max(r.first_key + e, j0) * m_sj];
    }
    return r;
}
// Whoever votes writes the same: a plain store.  (With an atomic, which goes lane by lane, the pass over whole rows was bound by its votes: bf16, a mask per
// head, whole call, 64 x 12 x 197 214 -> 149 us, 32 x 12 x 512 155 -> 130, 8 x 8 x 1024 79 -> 67; 64 MB of causal and key-padding masks, 8 x 16 x 2048, 138 -> 133.)
__device__ __forceinline__ void vote(int* v) { __hip_atomic_store(v, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP); }

// (one workgroup of 256 threads: block row rb of (mask batch entry, mask head) bh, the strip's 8 blocks)
template <typename T, bool VEC>
__device__ __forceinline__ void classify_strip(const T* mask, int64_t m_sb, int64_t m_sh, int64_t m_si, int64_t m_sj,
                                               int Hm, int Sq, int Skv, int nkb, int nrb, uint8_t* flags, int strip, int rb, int bh)
{
    __shared__ int votes[8][2];
    const int b = bh / Hm, h = bh % Hm;
    const T* base = mask + (int64_t)b * m_sb + (int64_t)h * m_sh;
    const int c8 = threadIdx.x & 31, r0 = threadIdx.x >> 5;       // 8 keys starting at strip * 256 + c8 * 8; rows r0, r0 + 8, ..
    if (threadIdx.x < 16) votes[threadIdx.x >> 1][threadIdx.x & 1] = 0;
    __syncthreads();
    const int j0 = strip * 256 + c8 * 8;
    if (j0 < Skv) {
        RowPart<T> part[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) part[u] = row_part<T, VEC>(base + (int64_t)min(rb * 32 + r0 + 8 * u, Sq - 1) * m_si, m_sj, j0, Skv);      // (for rows that do not exist the last one again)
        int not_zero = 0, not_hidden = 0;
#pragma unroll
        for (int u = 0; u < 4; ++u)
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const float f = to_f32(part[u].x[e]);
                not_zero |= e >= part[u].from && !(f == 0.0f);
                not_hidden |= e >= part[u].from && !(f == -INFINITY);
            }
        if (not_zero) vote(&votes[c8 >> 2][0]);
        if (not_hidden) vote(&votes[c8 >> 2][1]);
    }
    __syncthreads();
    if (threadIdx.x < 8) {
        const int kb = strip * 8 + threadIdx.x;
        if (kb < nkb) flags[((int64_t)bh * nrb + rb) * nkb + kb] = !votes[threadIdx.x][0] ? 1 : (!votes[threadIdx.x][1] ? 2 : 0);
    }
}

template <typename T, bool VEC>
__global__ __launch_bounds__(256) void mask_classify_kernel(const T* mask, int64_t m_sb, int64_t m_sh, int64_t m_si, int64_t m_sj,
                                                           int Hm, int Sq, int Skv, int nkb, uint8_t* flags, const int32_t* lims, int rows_m)
{
    const int strip = blockIdx.x, rb = blockIdx.y, bh = blockIdx.z;
    if (lims != nullptr) {
        // Row limits are known (mask_row_limits_kernel ran before): the attention launches read the flags only of blocks of 128
        // or 256 rows in which some row has no limit.  If every row of the 256 around these 32 has one, nobody will ask.
        const int blk0 = (rb * 32 / 256) * 256, blk1 = min(blk0 + 256, Sq);
        const int32_t* l = lims + (int64_t)bh * rows_m;
        bool ok = true;
        for (int i = blk0 + (int)threadIdx.x; i < blk1; i += 256) ok = ok && l[rows_m > 1 ? i : 0] >= 0;
        if (__syncthreads_and(ok)) return;
    }
    classify_strip<T, VEC>(mask, m_sb, m_sh, m_si, m_sj, Hm, Sq, Skv, nkb, gridDim.y, flags, strip, rb, bh);
}

// Row limits: for every row of the mask, n if the row reads n zeros and then -inf to its end (n = Skv: all zeros, n = 0:
// all -inf), else -1.  What a causal mask, a key-padding mask and their sum look like; a kernel that knows the limit of
// every row it handles compares key numbers with it instead of reading the mask.  One wavefront per row: the first
// position that is not zero and the number of -inf values decide.
template <typename T, bool VEC>
__device__ __forceinline__ void limits_of_rows(const T* mask, int64_t m_sb, int64_t m_sh, int64_t m_si, int64_t m_sj,
                                               int Hm, int rows_m, int Skv, int64_t n_rows, int32_t* lims, unsigned group)
{
    const int lane = threadIdx.x & 63;
    const int64_t r = (int64_t)group * 4 + (threadIdx.x >> 6);       // (mask batch entry, mask head, row)
    if (r >= n_rows) return;
    const int i = (int)(r % rows_m);
    const int64_t bh = r / rows_m;
    const T* row = mask + (bh / Hm) * m_sb + (bh % Hm) * m_sh + (int64_t)i * m_si;
    int first = Skv, ninf = 0;
    if (VEC) {
        for (int j0 = lane * 8; j0 < Skv; j0 += 512) {
            const RowPart<T> part = row_part<T, true>(row, m_sj, j0, Skv);
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const float f = to_f32(part.x[e]);
                if (!(f == 0.0f)) first = min(first, part.first_key + e);
                ninf += f == -INFINITY && e >= part.from;
            }
        }
    } else {
        for (int j = lane; j < Skv; j += 64) {
            const float f = to_f32(row[(int64_t)j * m_sj]);
            if (!(f == 0.0f)) first = min(first, j);
            ninf += f == -INFINITY;
        }
    }
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) {
        first = min(first, __shfl_xor(first, off, 64));
        ninf += __shfl_xor(ninf, off, 64);
    }
    if (lane == 0) lims[r] = ninf == Skv - first ? first : -1;
}
template <typename T, bool VEC>
__global__ __launch_bounds__(256) void mask_row_limits_kernel(const T* mask, int64_t m_sb, int64_t m_sh, int64_t m_si, int64_t m_sj,
                                                             int Hm, int rows_m, int Skv, int64_t n_rows, int32_t* lims)
{
    limits_of_rows<T, VEC>(mask, m_sb, m_sh, m_si, m_sj, Hm, rows_m, Skv, n_rows, lims, blockIdx.x);
}

// Limits and flags side by side in one launch: workgroups 0 .. n_strips - 1 classify a strip each (all of them: no limits to go by),
// the others take four rows each.
template <typename T, bool VEC>
__global__ __launch_bounds__(256) void mask_both_kernel(const T* mask, int64_t m_sb, int64_t m_sh, int64_t m_si, int64_t m_sj,
                                                       int Hm, int Sq, int Skv, int nkb, int nrb, uint8_t* flags, int32_t* lims, int rows_m, int64_t n_rows, unsigned n_strips)
{
    if (blockIdx.x >= n_strips) {
        limits_of_rows<T, VEC>(mask, m_sb, m_sh, m_si, m_sj, Hm, rows_m, Skv, n_rows, lims, blockIdx.x - n_strips);
        return;
    }
    const int across = (nkb + 7) / 8, strip = blockIdx.x % across, row = blockIdx.x / across;
    classify_strip<T, VEC>(mask, m_sb, m_sh, m_si, m_sj, Hm, Sq, Skv, nkb, nrb, flags, strip, row % nrb, row / nrb);
}

// Both in one pass over the mask: a workgroup of sixteen wavefronts takes 32 whole rows, two per wavefront, and has the limits of
// the rows and the flags of their blocks at the end.  Row by row as above (first position that is not zero, number of -inf values),
// the votes of a stretch of 4096 keys in LDS.
template <typename T, bool VEC>
__global__ __launch_bounds__(1024) void mask_scan_kernel(const T* mask, int64_t m_sb, int64_t m_sh, int64_t m_si, int64_t m_sj,
                                                        int Hm, int Sq, int Skv, int nkb, uint8_t* flags, int32_t* lims, int rows_m)
{
    constexpr int STRETCH = 4096;
    __shared__ int votes[STRETCH / 32][2];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int rb = blockIdx.x, bh = blockIdx.y;
    const T* base = mask + (int64_t)(bh / Hm) * m_sb + (int64_t)(bh % Hm) * m_sh;
    int first[2] = {Skv, Skv}, ninf[2] = {0, 0};
    for (int s0 = 0; s0 < Skv; s0 += STRETCH) {
        const int s1 = min(s0 + STRETCH, Skv);
        if (threadIdx.x < 2 * STRETCH / 32) votes[threadIdx.x >> 1][threadIdx.x & 1] = 0;
        __syncthreads();
#pragma unroll 2
        for (int j0 = s0 + lane * 8; j0 < s1; j0 += 512) {
            int not_zero = 0, not_hidden = 0;
#pragma unroll
            for (int r = 0; r < 2; ++r) {
                const int i = rb * 32 + wave + 16 * r;
                if (i >= Sq) continue;
                const T* row = base + (int64_t)i * m_si;
                auto see = [&](float f, int j) __attribute__((always_inline)) {
                    if (!(f == 0.0f)) first[r] = min(first[r], j);
                    ninf[r] += f == -INFINITY;
                    not_zero |= !(f == 0.0f);
                    not_hidden |= !(f == -INFINITY);
                };
                if (VEC && j0 + 7 < Skv) {
                    const typename Mask8<T>::type x = *(const typename Mask8<T>::type*)(row + j0);
#pragma unroll
                    for (int e = 0; e < 8; ++e) see(to_f32(x[e]), j0 + e);
                } else {      // (apart: what row_part leaves to the lane before costs the whole rows 10 - 15 %, this kernel being bound by its vector work)
                    const RowPart<T> part = row_part<T, VEC>(row, m_sj, j0, Skv);
#pragma unroll
                    for (int e = 0; e < 8; ++e)
                        if (e >= part.from) see(to_f32(part.x[e]), part.first_key + e);
                }
            }
            if (not_zero) vote(&votes[(j0 - s0) >> 5][0]);
            if (not_hidden) vote(&votes[(j0 - s0) >> 5][1]);
        }
        __syncthreads();
        const int kb = s0 / 32 + (int)threadIdx.x;
        if (threadIdx.x < STRETCH / 32 && kb < nkb)
            flags[((int64_t)bh * gridDim.x + rb) * nkb + kb] = !votes[threadIdx.x][0] ? 1 : (!votes[threadIdx.x][1] ? 2 : 0);
        __syncthreads();
    }
#pragma unroll
    for (int r = 0; r < 2; ++r) {
#pragma unroll
        for (int off = 32; off >= 1; off >>= 1) {
            first[r] = min(first[r], __shfl_xor(first[r], off, 64));
            ninf[r] += __shfl_xor(ninf[r], off, 64);
        }
        const int i = rb * 32 + wave + 16 * r;
        if (lane == 0 && i < rows_m) lims[(int64_t)bh * rows_m + i] = ninf[r] == Skv - first[r] ? first[r] : -1;      // (rows that are repeated: one of them)
    }
}

// Host has validated the extents; nbh = mask batch entries x mask heads (1 where the mask is broadcast).
hipError_t launch_mask_classify(const SdpaParams& p, int dtype, hipStream_t stream)
{
    const int nkb = (p.Skv + 31) / 32, nrb = (p.Sq + 31) / 32;
    const int Bm = p.m_sb ? p.B : 1, Hm = p.m_sh ? p.Hq : 1;
    if (nkb <= 0 || nrb <= 0) return hipSuccess;
    if (nrb > 65535 || (int64_t)Bm * Hm > 65535) return hipErrorInvalidValue;
    const dim3 grid((nkb + 7) / 8, nrb, Bm * Hm);
    uint8_t* flags = (uint8_t*)p.mask_flags;
    const int esz = dtype == 0 ? 4 : 2;
    const bool vec = p.m_sj == 1 && p.Skv >= 8;      // 8 consecutive elements in one load
    const int rows_m = p.m_si ? p.Sq : 1;
    const int64_t n_rows = (int64_t)Bm * Hm * rows_m, n_strips = (int64_t)((nkb + 7) / 8) * nrb * Bm * Hm;
    // Limits and flags side by side, so the mask read twice, where it is less than 16 MB: a launch and its latency saved.  Whole call at D = 64, us, by two
    // launches / by one: bf16, a causal mask, 1 x 1 x 128 x 128 13.3 / 12.1, 2 x 8 x 300 15.6 / 14.3, 16 x 12 x 256 18.0 / 16.7, 64 x 12 x 197 37.1 / 36.4, 4 x 8 x 1024
    // 23.8 / 22.7; key padding [B, 1, 1, Skv] 15.0 / 14.1, 16.8 / 15.7, 35.1 / 34.7, 23.3 / 22.6 for the last four; a bias per head 2 x 8 x 300 25.1 / 21.8, 4 x 16 x 700 47.0 / 43.6, 4 x 8 x
    // 1024 40.0 / 38.2; f32, a causal mask 2 x 8 x 300 20.4 / 19.2, 4 x 8 x 1024 59.8 / 59.4, a bias per head 2 x 8 x 300 43.1 / 39.9.  Above, masks of limits are behind by it
    // (f32 key padding 4 x 8 x 1024 88.7 / 92.7, bf16 1 x 8 x 4096 causal 57 / 61).
    if (p.mask_lims && (int64_t)Bm * Hm * p.Sq * p.Skv * esz < 16 << 20) {
        const dim3 bgrid((unsigned)(n_strips + (n_rows + 3) / 4));
#define BOTH(T, V) hipLaunchKernelGGL((mask_both_kernel<T, V>), bgrid, dim3(256), 0, stream, (const T*)p.mask, p.m_sb, p.m_sh, p.m_si, p.m_sj, Hm, p.Sq, p.Skv, nkb, nrb, flags, (int32_t*)p.mask_lims, rows_m, n_rows, (unsigned)n_strips)
        switch (dtype) {
            case 0: if (vec) BOTH(float, true); else BOTH(float, false); break;
            case 1: if (vec) BOTH(f16_t, true); else BOTH(f16_t, false); break;
            default: if (vec) BOTH(bf16_t, true); else BOTH(bf16_t, false); break;
        }
#undef BOTH
        return hipGetLastError();
    }
    // From there on limits and flags in one pass where its workgroups - one per 32 rows of the mask - are as many as compute units; else two
    // kernels, whose second reads nothing where all rows have limits.  Whole call, us, two / one: bf16, a bias per head, 8 x 8 x 1024 40.8 / 37.0, 1 x 8 x 4096 162 / 151, 8 x 16 x 2048 at D = 128
    // 233 / 217; a mask per head and sequence, 64 x 12 x 197 145 / 149, 32 x 12 x 512 158 / 127, 8 x 8 x 1024 87 / 66; causal and padding per sequence, 32 x 12 x 512 44.6 / 43.3, 8 x 16 x
    // 2048 133 / 133; f32, 1 x 8 x 4096, a bias 660 / 599, a band 280 / 217.  Fewer workgroups: one causal mask, bf16, 1 x 8 x 4096 57 / 62, 8 x 16 x 2048 154 / 156.  Not where all query rows have
    // the same mask row, as with key padding handed over as [B, 1, 1, Skv]: its limits are those of a few rows, the one pass would read each of them 32 times a workgroup (bf16, 16 x 16 x 4096
    // at D = 64 667 / 734, 8 x 16 x 2048 at D = 128 176 / 182, 32 x 12 x 512 42.1 / 43.9).
    if (p.mask_lims && p.m_si != 0 && (int64_t)nrb * Bm * Hm >= device_cus()) {
#define SCAN(T, V) hipLaunchKernelGGL((mask_scan_kernel<T, V>), dim3(nrb, Bm * Hm), dim3(1024), 0, stream, (const T*)p.mask, p.m_sb, p.m_sh, p.m_si, p.m_sj, Hm, p.Sq, p.Skv, nkb, flags, (int32_t*)p.mask_lims, rows_m)
        switch (dtype) {
            case 0: if (vec) SCAN(float, true); else SCAN(float, false); break;
            case 1: if (vec) SCAN(f16_t, true); else SCAN(f16_t, false); break;
            default: if (vec) SCAN(bf16_t, true); else SCAN(bf16_t, false); break;
        }
#undef SCAN
        return hipGetLastError();
    }
    if (p.mask_lims) {       // the limits first: the flags of blocks whose rows all have one are not needed
        const dim3 lgrid((unsigned)((n_rows + 3) / 4));
#define LIMITS(T, V) hipLaunchKernelGGL((mask_row_limits_kernel<T, V>), lgrid, dim3(256), 0, stream, (const T*)p.mask, p.m_sb, p.m_sh, p.m_si, p.m_sj, Hm, rows_m, p.Skv, n_rows, (int32_t*)p.mask_lims)
        switch (dtype) {
            case 0: if (vec) LIMITS(float, true); else LIMITS(float, false); break;
            case 1: if (vec) LIMITS(f16_t, true); else LIMITS(f16_t, false); break;
            default: if (vec) LIMITS(bf16_t, true); else LIMITS(bf16_t, false); break;
        }
#undef LIMITS
    }
#define CLASSIFY(T, V) hipLaunchKernelGGL((mask_classify_kernel<T, V>), grid, dim3(256), 0, stream, (const T*)p.mask, p.m_sb, p.m_sh, p.m_si, p.m_sj, Hm, p.Sq, p.Skv, nkb, flags, p.mask_lims, rows_m)
    switch (dtype) {
        case 0: if (vec) CLASSIFY(float, true); else CLASSIFY(float, false); break;
        case 1: if (vec) CLASSIFY(f16_t, true); else CLASSIFY(f16_t, false); break;
        default: if (vec) CLASSIFY(bf16_t, true); else CLASSIFY(bf16_t, false); break;
    }
#undef CLASSIFY
    return hipGetLastError();
}

// The row limits of a mask given by itself: shape [A0, A1, rows, Skv] with element strides (0 where an axis is repeated),
// one int per (a0, a1, row) in that order.  Behind incin_rocm_mask_row_limits.
hipError_t launch_mask_row_limits(const void* mask, int dtype, const int64_t shape[4], const int64_t strides[4], int32_t* lims, hipStream_t stream)
{
    const int64_t n_rows = shape[0] * shape[1] * shape[2];
    if (n_rows <= 0) return hipSuccess;
    if ((n_rows + 3) / 4 > 0x7fffffffLL) return hipErrorInvalidValue;
    const dim3 grid((unsigned)((n_rows + 3) / 4));
    const bool vec = strides[3] == 1 && shape[3] >= 8;
#define LIMITS(T, V) hipLaunchKernelGGL((mask_row_limits_kernel<T, V>), grid, dim3(256), 0, stream, (const T*)mask, strides[0], strides[1], strides[2], strides[3], (int)shape[1], (int)shape[2], (int)shape[3], n_rows, lims)
    switch (dtype) {
        case 0: if (vec) LIMITS(float, true); else LIMITS(float, false); break;
        case 1: if (vec) LIMITS(f16_t, true); else LIMITS(f16_t, false); break;
        default: if (vec) LIMITS(bf16_t, true); else LIMITS(bf16_t, false); break;
    }
#undef LIMITS
    return hipGetLastError();
}

}  // namespace incin_rocm
