// Grouped forward product Y[seg_e] = act(X[seg_e] . W_e^T + b_e) for few rows per expert, 16- and 32-bit types over a device
// segment table (gfx950): decoding steps, where every weight is read once and meets a handful of rows.
//
// Bound by the weights' way from memory, so nothing is staged: a wave loads a block of 16 rows of 64 bytes of weights with one 16-byte
// load per lane straight into the registers of a 16 x 16 x 32 MFMA (float32: of four 16 x 16 x 4), and the rows the same way (from L2, where they stay).
// A workgroup of four waves has 16 columns of one row tile; the waves take the contraction in turns of one unit,
// so that together they read whole lines of each weight row, with the next unit's loads under way before the products of
// the current one, and add up their accumulators through LDS in a fixed order.  With 16 waves per compute unit
// that is more than 100 KiB in flight on each, against 64 of the tiles of gemm_kernel.hpp, whose slabs of
// 128 rows are mostly padding here; no contraction has to be split over launches to fill the chip.
// Where it is used, and what it measured: use_skinny() in grouped_gemm.hip.
#include "gemm_skinny.hpp"

namespace fmoe {
namespace gemm {
namespace {

constexpr int kSkThreads = 256, kSkWaves = 4, kSkMaxBlocks = 4;   // most blocks of 16 rows of a wave

// one 16 x 16 block over 64 bytes of contraction; acc as for the 16 x 16 x 32 form
template <typename T> __device__ __forceinline__ void mma_step(f32x4 &acc, const u32x4 &w, const u32x4 &x) { Elem<T>::mma(acc, w, x); }
template <> __device__ __forceinline__ void mma_step<float>(f32x4 &acc, const u32x4 &w, const u32x4 &x) {
    // product j takes element j of every lane's four: contraction elements j, 4 + j, 8 + j and 12 + j of the step
#pragma unroll
    for (int j = 0; j < 4; ++j)
        acc = __builtin_amdgcn_mfma_f32_16x16x4f32(__uint_as_float(w[j]), __uint_as_float(x[j]), acc, 0, 0, 0);
}

template <typename T>
__global__ __launch_bounds__(kSkThreads, 4) void grouped_gemm_skinny_kernel(const SkinnyParams prm) {
#if defined(__HIP_DEVICE_COMPILE__)  // the host pass only needs the launch stub
    constexpr int EB = (int)sizeof(T), CE = 16 / EB, kStep = 64 / EB;   // elements per lane's load and per step
    typedef std::conditional_t<sizeof(T) == 2, u32x2, u32x4> Vec4;        // four elements
    constexpr uint32_t kOutOfRange = 0x80000000u;
    constexpr int kRsrcFlags = 0x00020000;   // raw buffer, 32-bit data format
    typedef const int32_t __attribute__((address_space(4))) *DevTab;    // read-only, uniform: scalar loads
    typedef int i32x4 __attribute__((ext_vector_type(4)));
    typedef const i32x4 __attribute__((address_space(4))) *DevTab4;
    __shared__ f32x4 part[kSkWaves - 1][kSkMaxBlocks][64];

    const DevTab dtab = (DevTab)(uintptr_t)prm.dev_tab;
    const int tile = __builtin_amdgcn_readfirstlane(blockIdx.x / prm.tiles_n);
    if (tile >= dtab[segtab::kTiles128]) return;   // the launch was sized for the most row tiles there can be
    const int n0 = (blockIdx.x - tile * prm.tiles_n) * kSkinnyCols;
    const i32x4 entry = *(DevTab4)(dtab + prm.map_off + 4 * tile);   // {expert, first row, rows (at most 128)}
    const int expert = entry[0], first = entry[1], rows = entry[2], K = prm.k_extent;
    const int t = threadIdx.x, lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const int lb = lane & 15, hq = lane >> 4;

    // weights: rows past the last column lie past the end of the resource and read as zero
    const T *W = (const T *)prm.w + ((int64_t)expert * prm.n_cols + n0) * K;
    const int w_bytes = min(kSkinnyCols, prm.n_cols - n0) * K * EB;
    const __amdgpu_buffer_rsrc_t w_rs = __builtin_amdgcn_make_buffer_rsrc(const_cast<T *>(W), 0, w_bytes, kRsrcFlags);
    const uint32_t w_off = (uint32_t)(lb * K * EB + hq * 16);
    const bool gather = prm.row_index != nullptr;
    const T *X = (const T *)prm.x + (gather ? (int64_t)0 : (int64_t)first * K);
    const int x_bytes = gather ? (int)(prm.x_total_rows * K * EB) : rows * K * EB;
    const __amdgpu_buffer_rsrc_t x_rs = __builtin_amdgcn_make_buffer_rsrc(const_cast<T *>(X), 0, x_bytes, kRsrcFlags);

    // RB blocks of 16 rows from row r0 of the tile on; STEPS contraction steps of 64 bytes to a unit
    auto pass = [&](auto rb_tag, auto steps_tag, int r0) {
        constexpr int RB = decltype(rb_tag)::value, STEPS = decltype(steps_tag)::value;
        uint32_t x_off[RB];
#pragma unroll
        for (int y = 0; y < RB; ++y) {
            const int row = r0 + 16 * y + lb;
            int64_t src = row < rows ? row : -1;
            if (gather && row < rows) {
                const int64_t idx = prm.row_index[first + row];
                src = -1;
                if (idx >= 0 && idx <= (int64_t)INT32_MAX)
                    src = prm.div_shift < 0 ? idx : (int64_t)(__umulhi((uint32_t)idx, prm.div_mul) >> prm.div_shift);
                if (src >= prm.x_total_rows) src = -1;
            }
            x_off[y] = src >= 0 ? (uint32_t)(src * K * EB + hq * 16) : kOutOfRange;
        }
        f32x4 acc[RB];
#pragma unroll
        for (int y = 0; y < RB; ++y) acc[y] = f32x4{0.f, 0.f, 0.f, 0.f};
        struct Unit { u32x4 w[STEPS], x[STEPS][RB]; };
        auto load = [&](Unit &u, int unit) {
#pragma unroll
            for (int s = 0; s < STEPS; ++s) {
                const int k = (unit * STEPS + s) * kStep;
                // sign bit set where this lane's elements lie past the contraction (and for every unit past it)
                const uint32_t past = (uint32_t)(K - 1 - k - hq * CE) & kOutOfRange;
                u.w[s] = __builtin_amdgcn_raw_buffer_load_b128(w_rs, (int)((w_off + k * EB) | past), 0, 0);
#pragma unroll
                for (int y = 0; y < RB; ++y)
                    u.x[s][y] = __builtin_amdgcn_raw_buffer_load_b128(x_rs, (int)((x_off[y] + k * EB) | past), 0, 0);
            }
        };
        auto multiply = [&](const Unit &u) {
#pragma unroll
            for (int s = 0; s < STEPS; ++s)
#pragma unroll
                for (int y = 0; y < RB; ++y) mma_step<T>(acc[y], u.w[s], u.x[s][y]);
        };
        const int n_units = (K + kStep * STEPS - 1) / (kStep * STEPS);
        Unit a, b;
        int unit = wave;
        load(a, unit);
        while (unit < n_units) {
            load(b, unit + kSkWaves);
            multiply(a);
            unit += kSkWaves;
            if (unit >= n_units) break;
            load(a, unit + kSkWaves);
            multiply(b);
            unit += kSkWaves;
        }
        // the waves' sums in ascending order of the wave
        __syncthreads();
        if (wave > 0) {
#pragma unroll
            for (int y = 0; y < RB; ++y) part[wave - 1][y][lane] = acc[y];
        }
        __syncthreads();
        if (wave > 0) return;   // (from this pass)
        // acc[y][i] is C(row 16 y + lb, column 4 hq + i)
        const int col = n0 + 4 * hq;
        alignas(16) T b4[4] = {};
        if (prm.bias != nullptr && col < prm.n_cols)
            *(Vec4 *)b4 = *(const Vec4 *)((const T *)prm.bias + (int64_t)expert * prm.n_cols + col);
#pragma unroll
        for (int y = 0; y < RB; ++y) {
            f32x4 v = acc[y];
#pragma unroll
            for (int w = 0; w < kSkWaves - 1; ++w) v += part[w][y][lane];
            const int row = r0 + 16 * y + lb;
            if (row >= rows || col >= prm.n_cols) continue;
            alignas(16) T pre[4], res[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const float p = v[i] + (float)b4[i];
                pre[i] = (T)p;
                res[i] = (T)apply_act<sizeof(T) == 2>(p, prm.activation);
            }
            const int64_t at = (int64_t)(first + row) * prm.n_cols + col;
            if (prm.aux != nullptr) *(Vec4 *)((T *)prm.aux + at) = *(const Vec4 *)pre;
            *(Vec4 *)((T *)prm.y + at) = *(const Vec4 *)res;
        }
    };
    typedef std::integral_constant<int, 1> One;
    typedef std::integral_constant<int, 2> Two;
    typedef std::integral_constant<int, 4> Four;
    // (blocks of rows, and contraction steps of a unit: two units have to fit 128 registers)
    if (rows <= 16) {
        pass(One{}, Four{}, 0);
    } else if (rows <= 32) {
        pass(Two{}, std::integral_constant<int, 3>{}, 0);
    } else {
        for (int r0 = 0; r0 < rows; r0 += 64) pass(Four{}, One{}, r0);
    }
#endif
}

}  // namespace

int launch_skinny(const SkinnyParams &prm, int dtype, int64_t row_tiles, hipStream_t stream) {
    const int64_t grid = row_tiles * prm.tiles_n;
    if (grid > (int64_t)INT32_MAX) return fail(FMOE_ELIMIT, "grouped GEMM: grid of %lld workgroups", (long long)grid);
    FMOE_REQUIRE(dtype == FMOE_BF16 || dtype == FMOE_F16 || dtype == FMOE_F32, "grouped GEMM: dtype %d is not a 16- or 32-bit float type", dtype);
    if (dtype == FMOE_F32) grouped_gemm_skinny_kernel<float><<<(unsigned)grid, kSkThreads, 0, stream>>>(prm);
    else if (dtype == FMOE_BF16) grouped_gemm_skinny_kernel<__bf16><<<(unsigned)grid, kSkThreads, 0, stream>>>(prm);
    else grouped_gemm_skinny_kernel<_Float16><<<(unsigned)grid, kSkThreads, 0, stream>>>(prm);
    FMOE_LAUNCH_CHECK();
    return FMOE_OK;
}

}  // namespace gemm
}  // namespace fmoe
