// Device side of the segment table (layout: grouped_gemm.hpp, namespace segtab): the part that the
// stand-alone kernel of segment_table.hip and the routing kernels share.
#pragma once
#include "grouped_gemm.hpp"

namespace fmoe {
namespace segtab {

constexpr int kThreads = 1024;        // the workgroup that builds a table
constexpr int kSmallExperts = 1024;   // most experts of small_table(): one per thread
constexpr int kRankExperts = 64;     // most experts that are ordered by counting

// LDS of small_table(): the three prefixes and the waves' sums
struct SmallLds {
    int64_t row_sum[kThreads / kWave];
    int32_t wave_sum[2][kThreads / kWave], wave_live[kThreads / kWave];
    int32_t seg[kSmallExperts + 1];
    __attribute__((aligned(8))) int32_t pfx[2][kSmallExperts + 1];   // (afterwards the exchange buffer of sort_descending)
    __attribute__((aligned(16))) int32_t rows[kSmallExperts];
};

// The value of the lane whose number differs in bit J, by the cheapest exchange: within rows of 16 lanes in the vector pipe, of 32
// by a swizzle with a constant pattern, else by address.
template <int J> __device__ __forceinline__ unsigned int lane_xor(unsigned int v) {
    if (J == 1) return __builtin_amdgcn_update_dpp(0, v, 0xb1, 0xf, 0xf, true);     // quad_perm 1 0 3 2
    if (J == 2) return __builtin_amdgcn_update_dpp(0, v, 0x4e, 0xf, 0xf, true);     // quad_perm 2 3 0 1
    if (J == 4)   // bits 0 to 2, then 0 and 1 back: row_half_mirror, quad_perm 3 2 1 0
        return __builtin_amdgcn_update_dpp(0, __builtin_amdgcn_update_dpp(0, v, 0x141, 0xf, 0xf, true), 0x1b, 0xf, 0xf, true);
    if (J == 8) return __builtin_amdgcn_update_dpp(0, v, 0x128, 0xf, 0xf, true);    // row_ror 8
    if (J == 16) return __builtin_amdgcn_ds_swizzle(v, 0x401f);                     // and 31, or 0, xor 16
    return __shfl_xor(v, J, kWave);
}
template <int J> __device__ __forceinline__ unsigned long long lane_xor(unsigned long long v) {
    return ((unsigned long long)lane_xor<J>((unsigned int)(v >> 32)) << 32) | lane_xor<J>((unsigned int)v);
}

// Sorts the workgroup's keys, one per thread, among its first n threads (a power of two of at least 64): thread i ends with the
// i-th largest.  A bitonic network; partners in the same wave exchange by lane, others through buf [kThreads].
template <typename Key> __device__ __forceinline__ Key sort_descending(Key key, int n, Key *buf) {
    const int i = threadIdx.x;
    for (int k = 2; k <= n; k <<= 1) {
        auto take = [&](Key other, int j) {
            const bool keep_larger = ((i & j) == 0) == ((i & k) == 0);
            key = (key > other) == keep_larger ? key : other;
        };
        for (int j = k >> 1; j >= kWave; j >>= 1) {
            buf[i] = key;
            __syncthreads();
            const Key other = buf[i ^ j];
            __syncthreads();
            take(other, j);
        }
        if (k > 32) take(lane_xor<32>(key), 32);
        if (k > 16) take(lane_xor<16>(key), 16);
        if (k > 8) take(lane_xor<8>(key), 8);
        if (k > 4) take(lane_xor<4>(key), 4);
        if (k > 2) take(lane_xor<2>(key), 2);
        take(lane_xor<1>(key), 1);
    }
    return key;
}

// Thread e's place in the list of the experts by descending rows (of equal ones the lower expert first): the expert that belongs
// there.  A key is an expert's rows above its number; 32 bits hold both up to 2^22 rows, half the exchanges of 64.
template <typename Key> __device__ __forceinline__ int expert_in_order(int rows, int n_expert, Key *buf) {
    constexpr int kBits = 10;   // kSmallExperts
    const int e = threadIdx.x;
    int n = kWave;
    while (n < n_expert) n <<= 1;
    // (threads without an expert sort last: their keys have the highest numbers)
    const Key mine = ((Key)(e < n_expert ? rows : 0) << kBits) | (Key)((1 << kBits) - 1 - e);
    return (1 << kBits) - 1 - (int)(sort_descending(mine, n, buf) & ((1 << kBits) - 1));
}

// Prefix sum (with the lane's own value) over the wave, all lanes taking part: within rows of 16 lanes, then over the rows
__device__ __forceinline__ int32_t wave_prefix(int32_t v) {
    v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xf, 0xf, true);    // row_shr 1, 2, 4, 8
    v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xf, 0xf, true);
    v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xf, 0xf, true);
    v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xf, 0xf, true);
    v += __builtin_amdgcn_update_dpp(0, v, 0x142, 0xa, 0xf, false);   // row_bcast 15 into rows 1 and 3
    v += __builtin_amdgcn_update_dpp(0, v, 0x143, 0xc, 0xf, false);   // row_bcast 31 into rows 2 and 3
    return v;
}
// The sum of the first `wave` of at most 16 sums in LDS, all lanes taking part: read together and added by lanes, where a walk over them was a
// chain of up to fifteen LDS latencies.
__device__ __forceinline__ int32_t sums_before(const int32_t *sums, int wave) {
    static_assert(kThreads / kWave <= 16, "a row of lanes holds the sums");
    const int lane = threadIdx.x & (kWave - 1);
    int32_t v = lane < wave ? sums[lane] : 0;
    v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xf, 0xf, true);    // row_shr 1, 2, 4, 8
    v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xf, 0xf, true);
    v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xf, 0xf, true);
    v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xf, 0xf, true);
    return __builtin_amdgcn_readlane(v, 15);
}

// The whole table for at most kSmallExperts experts by one workgroup of kThreads threads, thread e
// holding expert e's row count (others: anything).  The counts are clamped so that their sum never
// exceeds rows_cap.  The prefixes stay in LDS, where the row tiles find their expert by binary
// search: read back from memory, the ten dependent loads of that search were most of the table's
// 9.7 us at 8 experts.  kExact: the counts are the caller's own, none is negative, their sum is at most rows_cap and `upto` is their
// prefix sum with this thread's own.
template <bool kExact>
__device__ __forceinline__ void small_table(int64_t count, int n_expert, int rows_cap, int32_t *__restrict__ tab, SmallLds &lds,
                                            int32_t upto = 0) {
    const int e = threadIdx.x, lane = e & (kWave - 1), wave = e / kWave;
    int32_t lo, hi;
    if constexpr (kExact) {
        hi = upto;
        lo = e < n_expert ? upto - (int32_t)count : upto;
    } else {
        int64_t c64 = e < n_expert ? count : 0;
        c64 = c64 < 0 ? 0 : (c64 > rows_cap ? rows_cap : c64);
        int64_t v = c64;
    #pragma unroll
        for (int off = 1; off < kWave; off <<= 1) {
            const int64_t up = __shfl_up(v, off, kWave);
            if (lane >= off) v += up;
        }
        if (lane == kWave - 1) lds.row_sum[wave] = v;
        __syncthreads();
        for (int w = 0; w < wave; ++w) v += lds.row_sum[w];
        const int64_t before = v - c64;
        lo = (int32_t)(before > rows_cap ? rows_cap : before);
        hi = (int32_t)(v > rows_cap ? rows_cap : v);
    }
    const int32_t rows = hi - lo;
    const int32_t t[2] = {(rows + 255) / 256, (rows + 127) / 128};
    int32_t tv[2];
#pragma unroll
    for (int k = 0; k < 2; ++k) {
        tv[k] = wave_prefix(t[k]);
        if (lane == kWave - 1) lds.wave_sum[k][wave] = tv[k];
    }
    const int live = __popcll(__ballot(rows > 0));
    if (lane == 0) lds.wave_live[wave] = live;
    __syncthreads();
#pragma unroll
    for (int k = 0; k < 2; ++k) tv[k] += sums_before(lds.wave_sum[k], wave);
    int32_t *seg = tab + seg_off(), *pfx256 = tab + pfx256_off(n_expert), *pfx128 = tab + pfx128_off(n_expert);
    const int map256 = (int)map256_off(n_expert), map128 = (int)map128_off(rows_cap, n_expert);
    lds.rows[e] = e < n_expert ? rows : -1;
    if (e < n_expert) {
        lds.seg[e] = seg[e] = lo;
        lds.pfx[0][e] = pfx256[e] = tv[0] - t[0];
        lds.pfx[1][e] = pfx128[e] = tv[1] - t[1];
    }
    if (e == n_expert - 1) {
        lds.seg[n_expert] = seg[n_expert] = hi;
        lds.pfx[0][n_expert] = pfx256[n_expert] = tv[0];
        lds.pfx[1][n_expert] = pfx128[n_expert] = tv[1];
        tab[0] = n_expert;
        tab[kRows] = hi;
        tab[kTiles256] = tv[0];
        tab[kTiles128] = tv[1];
        tab[kMap256] = map256;
        tab[kMap128] = map128;
        tab[kRowsCap] = rows_cap;
        int all_live = 0;
#pragma unroll
        for (int w = 0; w < kThreads / kWave; ++w) all_live += lds.wave_live[w];
        tab[kLive] = all_live;
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < 2; ++k) {
        const int block_rows = k == 0 ? 256 : 128;
        const int32_t *pfx = lds.pfx[k];
        int32_t *map = tab + (k == 0 ? map256 : map128);
        const int tiles = pfx[n_expert];
        for (int i = threadIdx.x; i < tiles; i += kThreads) {
            int a = 0, b = n_expert;  // pfx[a] <= i < pfx[b]
            while (b - a > 1) {
                const int mid = (a + b) >> 1;
                if (pfx[mid] <= i) a = mid; else b = mid;
            }
            const int first = lds.seg[a] + (i - pfx[a]) * block_rows, left = lds.seg[a + 1] - first;
            int4 entry;
            entry.x = a;
            entry.y = first;
            entry.z = left < block_rows ? left : block_rows;
            entry.w = 0;
            *(int4 *)(map + 4 * (int64_t)i) = entry;
        }
    }
    // The experts by descending rows.  Up to kRankExperts an expert's place is counted, the number of experts that come
    // before it; beyond, where the square of their number tells, the experts are sorted.  The whole table, counted and
    // sorted: up to 65 experts 7.6 us either way, 128: 8.6 / 7.6, 192: 10.3 / 8.1, 256: 11.8 / 8.1, 512: 19.6 / 9.1, 1024: 44.6 / 10.6
    // (exchanges by address and 64-bit keys: 256: 10.3, 512: 12.0, 1024: 14.3).
    int4 *order = (int4 *)(tab + order_off(rows_cap, n_expert));
    if (n_expert > kRankExperts) {
        __syncthreads();   // the maps are done with lds.pfx
        const int ex = rows_cap < (1 << 22) ? expert_in_order<unsigned int>(rows, n_expert, (unsigned int *)&lds.pfx[0][0])
                                            : expert_in_order<unsigned long long>(rows, n_expert, (unsigned long long *)&lds.pfx[0][0]);
        if (e < n_expert) order[e] = make_int4(ex, lds.seg[ex], lds.rows[ex], 0);
    } else if (e < n_expert) {
        int place = 0;
        for (int f = 0; f < n_expert; f += 4) {
            const int4 r = *(const int4 *)(lds.rows + f);
            place += (r.x > rows || (r.x == rows && f < e)) + (r.y > rows || (r.y == rows && f + 1 < e)) +
                     (r.z > rows || (r.z == rows && f + 2 < e)) + (r.w > rows || (r.w == rows && f + 3 < e));
        }
        order[place] = make_int4(e, lo, rows, 0);
    }
}

}  // namespace segtab
}  // namespace fmoe
