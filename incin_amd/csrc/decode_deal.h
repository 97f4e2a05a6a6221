// Split-KV launches whose sequences differ in length (key counts on the device): the keys of all of them, dealt to the workgroups of
// one round in equal shares.
//
// A launch has a column per KV head, and the same sequences one after the other in each, counted in units of the keys that the four
// wavefronts of a workgroup take in one turn (a sequence without keys counts one: somebody has to write its rows).  Of W workgroups
// and T units in all, the first min(W, T) have a share, T / W units in a row each and the first T mod W of them one more, sequence by
// sequence.  A sequence that lies inside one share is finished by that workgroup; of the others, a share holds at most one that ends in it and
// one that goes on behind it: two places for partial results per workgroup, which the combine kernel (sdpa_decode.hip) adds up in order.  Nothing here is
// known to the host but W: key counts may change between the replays of a recorded launch.
#pragma once
#include "sdpa_params.h"

namespace incin_rocm {

constexpr int DEAL_MAX_BATCH = 256;       // four sequences per lane of a wavefront
constexpr int DEAL_MAX_VALUES = 1024;     // rows of a KV head x head dimension (of the instance)

// Keys per unit: a block of 32 keys (64 at D = 64) for each of the four wavefronts
template <typename T, int D> constexpr int deal_unit() { return D == 64 ? 256 : 128; }

// The sequences of a column: lane l of a wavefront holds those numbered l * per .. + per - 1.
struct DealColumn {
    int per, units[4], before, total;      // units of each, of all before the lane's first, of all
};
template <int UNIT> __device__ __forceinline__ int deal_units(const SdpaParams& p, int b)
{
    const int len = p.kv_lens ? clampi(p.kv_lens[b], 0, p.Skv) : p.Skv;
    return max(1, (len + UNIT - 1) / UNIT);
}
template <int UNIT> __device__ __forceinline__ DealColumn deal_column(const SdpaParams& p)
{
    const int lane = threadIdx.x & 63;
    DealColumn c;
    c.per = (p.B + 63) >> 6;
    int sum = 0;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        const int b = lane * c.per + k;
        c.units[k] = k < c.per && b < p.B ? deal_units<UNIT>(p, b) : 0;
        sum += c.units[k];
    }
    int incl = sum;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        const int x = __shfl_up(incl, off, 64);
        if (lane >= off) incl += x;
    }
    c.before = incl - sum;
    c.total = __builtin_amdgcn_readlane(incl, 63);
    return c;
}
// The sequence that unit `pos` (below total) belongs to, and its first unit.
__device__ __forceinline__ void deal_find(const DealColumn& c, int pos, int* b, int* first)
{
    const unsigned long long at = __builtin_amdgcn_ballot_w64(pos >= c.before && c.units[0] > 0);
    const int l = 63 - __builtin_clzll(at);      // the last lane with sequences that starts at or before pos
    int f = __builtin_amdgcn_readlane(c.before, l), k = 0;
#pragma unroll
    for (int i = 0; i < 3; ++i) {
        const int u = __builtin_amdgcn_readlane(c.units[i], l);
        if (k == i && u > 0 && pos >= f + u) { f += u; ++k; }
    }
    *b = l * c.per + k;
    *first = f;
}
// First unit and units of sequence b.
__device__ __forceinline__ void deal_place(const DealColumn& c, int b, int* first, int* units)
{
    const int l = b / c.per, k = b - l * c.per;
    int f = __builtin_amdgcn_readlane(c.before, l), u = 0;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int x = __builtin_amdgcn_readlane(c.units[i], l);
        if (i < k) f += x;
        if (i == k) u = x;
    }
    *first = f;
    *units = u;
}
// The shares: of `total` units in all, workgroup w's is [begin(w), begin(w + 1)); owner(u) holds unit u.
struct DealShares {
    int count, each, more;      // workgroups with a share; units of each, the first `more` one more
    __device__ __forceinline__ DealShares(int total, int workgroups)
    {
        count = min(workgroups, total);
        each = total / count;
        more = total - each * count;
    }
    __device__ __forceinline__ int begin(int w) const { return w * each + min(w, more); }
    __device__ __forceinline__ int owner(int unit) const
    {
        const int long_ones = more * (each + 1);
        return unit < long_ones ? unit / (each + 1) : more + (unit - long_ones) / each;
    }
};
// Which place a workgroup's partial results of a row go to: rows_per_place rows each.
__device__ __forceinline__ int64_t deal_slot(int w, bool goes_on, int rows_per_place, int row) { return ((int64_t)w * 2 + (goes_on ? 1 : 0)) * rows_per_place + row; }
inline size_t deal_workspace_bytes(int workgroups, int rows_per_place, int Dp) { return (size_t)workgroups * 2 * rows_per_place * (Dp + 2) * sizeof(float); }

}  // namespace incin_rocm
