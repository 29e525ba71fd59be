// Grouped GEMM over ragged expert segments for 16-bit types whose feature sizes or pointers are off the
// 16-byte grid (gfx950), on the 16 x 16 x 32 MFMA.
//
// The aligned kernels bring slabs straight from memory into LDS, which needs 16-byte chunks on 16-byte boundaries.
// Here a chunk of eight elements comes in through registers with one 16-byte load from wherever it begins (global
// loads take any alignment) and goes to the same LDS image as in gemm_kernel.hpp, so that the fragment reads
// and products are the same.  Where the contraction or the row of a [contraction][index] operand ends inside a chunk, the
// chunk that ends with it is read and moved down; rows past a tile's end repeat its last row and are not stored.
//
// 128 x 128 tiles (64 x 64 per wave), 64 x 128 where those would leave compute units without one; two slabs of
// LDS, the next slab's chunks are requested before the products of the current one.  Bound by the latency of those
// loads up to a few hundred rows per expert (1.2 us a slab) and by their way through registers above (8192 rows, 2047 x 4093:
// 600 to 680 TFLOP/s).  Measured against the element-wise kernel it replaced: see the dispatch in grouped_gemm.hip.
#include "gemm_kernel.hpp"

namespace fmoe {
namespace {
using namespace gemm;

constexpr int kUaThreads = 256, kUaBN = 128, kUaBK = 64;

template <typename T> __device__ __forceinline__ u32x4 load_unaligned(const T *p) {
    u32x4 v;
    __builtin_memcpy(&v, p, 16);
    return v;
}
// The first n of the eight elements at p, zeros after them.  8 <= n: all of them.  0 < n < 8: with `back`, the eight
// elements that end with them (the caller knows that as many precede them in their row), moved down; else one by one.
// n <= 0: nothing is read at p, but with `back` eight elements at `safe`.
template <typename T> __device__ __forceinline__ u32x4 load_part(const T *p, const T *safe, int n, bool back) {
    if (back) {
        const int s = 8 - max(0, min(n, 8));   // elements to move down
        const u32x4 v = load_unaligned(n > 0 ? p - s : safe);
        const u32x4 a = s & 4 ? u32x4{v[2], v[3], 0u, 0u} : v;
        const u32x4 b = s & 2 ? u32x4{a[1], a[2], a[3], 0u} : a;
        const u32x4 c = s & 1 ? u32x4{__builtin_amdgcn_alignbit(b[1], b[0], 16), __builtin_amdgcn_alignbit(b[2], b[1], 16),
                                      __builtin_amdgcn_alignbit(b[3], b[2], 16), b[3] >> 16} : b;
        return n > 0 ? c : u32x4{0u, 0u, 0u, 0u};
    }
    if (n >= 8) return load_unaligned(p);
    alignas(16) uint16_t e[8] = {};
    const uint16_t *src = (const uint16_t *)p;
#pragma unroll
    for (int j = 0; j < 7; ++j)
        if (j < n) e[j] = src[j];
    return __builtin_bit_cast(u32x4, e);
}

// PSHAPE / QSHAPE: kKC = [index][contraction] in memory, kMC = [contraction][index].
template <typename T, int BM, int PSHAPE, int QSHAPE, int RAGGED>
__global__ __launch_bounds__(kUaThreads) void grouped_gemm_unaligned_kernel(const GemmParams prm) {
#if defined(__HIP_DEVICE_COMPILE__)  // the host pass only needs the launch stub
    static_assert(QSHAPE == kKC || BM == 128, "the swizzle of a [contraction][index] slab needs rows of 256 bytes");
    constexpr int BN = kUaBN, BK = kUaBK, TI = 4, TJ = BM / 32;
    constexpr int NP = BN * 8 / kUaThreads, NQ = BM * 8 / kUaThreads;   // chunks per thread and slab
    constexpr int P_BYTES = BN * 128, Q_BYTES = BM * 128, STAGE = P_BYTES + Q_BYTES;
    constexpr bool kBiasGrad = RAGGED == kRaggedK;
    __shared__ __attribute__((aligned(16))) unsigned char smem[2 * STAGE];

    const int t = threadIdx.x, lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const int wm = wave >> 1, wn = wave & 1, lb = lane & 15, hq = lane >> 4;

    // -- which tile: a contiguous eighth of the logical order per XCD, kGroupM row tiles per column tile
    // (over a device table the launch is sized for the most tiles there can be)
    typedef const int32_t __attribute__((address_space(4))) *DevTab;    // read-only, uniform: scalar loads
    const DevTab dtab = (DevTab)(uintptr_t)prm.dev_tab;
    const bool dev = prm.dev_tab != nullptr;
    int tm_total = prm.tiles_m, total_tiles = prm.total_tiles;
    if (RAGGED == kRaggedRows) {
        tm_total = dev ? dtab[segtab::kTiles128] * (128 / BM) : prm.tab.tile[prm.tab.n];
        total_tiles = tm_total * prm.tiles_n;
    }
    const int per_xcd = (total_tiles + 7) >> 3;
    const int L = (blockIdx.x & 7) * per_xcd + (blockIdx.x >> 3);
    if ((int)(blockIdx.x >> 3) >= per_xcd || L >= total_tiles) return;
    int ei = 0, rem = L;
    if (RAGGED == kRaggedK) {
        ei = L / (prm.tiles_m * prm.tiles_n);
        rem = L - ei * (prm.tiles_m * prm.tiles_n);
    }
    const int grp = rem / (kGroupM * prm.tiles_n), in_grp = rem - grp * kGroupM * prm.tiles_n;
    const int gsz = min(kGroupM, tm_total - grp * kGroupM);
    const int nt = in_grp / gsz, mt = grp * kGroupM + in_grp - nt * gsz;
    int seg_lo, seg_hi, row0 = 0;   // (ragged rows over a device table: of this very tile)
    if (RAGGED == kRaggedRows && dev) {
        typedef int i32x4 __attribute__((ext_vector_type(4)));
        typedef const i32x4 __attribute__((address_space(4))) *DevTab4;
        constexpr int kPerEntry = 128 / BM;   // (tiles of 64 rows: the halves of the map's 128; the second may have no rows)
        const i32x4 entry = *(DevTab4)(dtab + prm.dev_map_off + 4 * (mt / kPerEntry));
        ei = entry[0];
        seg_hi = entry[1] + entry[2];
        row0 = seg_lo = entry[1] + (mt % kPerEntry) * BM;
        if (seg_lo >= seg_hi) return;
    } else if (RAGGED == kRaggedRows) {
        int lo = 0, hi = prm.tab.n;  // tile[lo] <= mt < tile[hi]
        while (hi - lo > 1) {
            const int mid = (lo + hi) >> 1;
            if (prm.tab.tile[mid] <= mt) lo = mid; else hi = mid;
        }
        ei = lo;
        seg_lo = prm.tab.seg[ei];
        seg_hi = prm.tab.seg[ei + 1];
        row0 = seg_lo + (mt - prm.tab.tile[ei]) * BM;
    } else {
        seg_lo = dev ? dtab[segtab::kHeader + ei] : prm.tab.seg[ei];
        seg_hi = dev ? dtab[segtab::kHeader + ei + 1] : prm.tab.seg[ei + 1];
    }
    const int expert = prm.tab.first_expert + ei;
    const int n0 = nt * BN, p_valid = min(BN, prm.n_cols - n0);
    int K, q_valid, m0 = 0;
    const T *P, *Q;
    int64_t c_off;
    if (RAGGED == kRaggedRows) {
        q_valid = min(BM, seg_hi - row0);
        K = prm.k_extent;
        P = (const T *)prm.P + (int64_t)expert * prm.p_expert_stride + (PSHAPE == kKC ? (int64_t)n0 * prm.ldp : (int64_t)n0);
        Q = (const T *)prm.Q + (int64_t)row0 * prm.ldq;
        c_off = (int64_t)row0 * prm.ldc + n0;
    } else {
        m0 = mt * BM;
        q_valid = min(BM, prm.n_rows - m0);
        K = seg_hi - seg_lo;
        P = (const T *)prm.P + (int64_t)seg_lo * prm.ldp + n0;
        Q = (const T *)prm.Q + (int64_t)seg_lo * prm.ldq + m0;
        c_off = (int64_t)expert * prm.c_expert_stride + (int64_t)m0 * prm.ldc + n0;
    }

    // An expert without rows: its tiles write zeros over equal parts of its gradient, which is dense (as a tile of no
    // slabs, stored 16 bytes at a time off the grid: 1 row over 500 experts of 1483 x 70, 91 us, like this 23).
    if (RAGGED == kRaggedK && K == 0 && !(prm.accumulate_first && ei == 0)) {
        const int64_t size = (int64_t)prm.n_rows * prm.n_cols, per = (size + prm.tiles_m * prm.tiles_n - 1) / (prm.tiles_m * prm.tiles_n);
        const int64_t lo = min(rem * per, size), hi = min(lo + per, size);
        T *gw = (T *)prm.C + (int64_t)expert * prm.c_expert_stride;
        const int64_t body = min(lo + (int64_t)((16 - ((uintptr_t)(gw + lo) & 15)) & 15) / 2, hi), vecs = (hi - body) / 8;
        for (int64_t i = lo + t; i < body; i += kUaThreads) gw[i] = (T)0.f;
        for (int64_t v = t; v < vecs; v += kUaThreads) ((u32x4 *)(gw + body))[v] = u32x4{0u, 0u, 0u, 0u};
        for (int64_t i = body + 8 * vecs + t; i < hi; i += kUaThreads) gw[i] = (T)0.f;
        if (rem == 0 && prm.bias_grad != nullptr)
            for (int r = t; r < prm.n_rows; r += kUaThreads) ((T *)prm.bias_grad)[(int64_t)expert * prm.n_rows + r] = (T)0.f;
        return;
    }

    // -- memory -> registers -> LDS: thread t has chunk it * 256 + t of the slab
    auto chunk_index = [&](int shape, int it) { return shape == kKC ? (it * kUaThreads + t) >> 3 : (it * kUaThreads + t) >> 4; };
    // (its offsets from the slab's first element do not change: rows and chunks past a tile's end repeat the last one)
    int64_t p_off[NP], q_off[NQ];
    auto set_offsets = [&](int shape, int64_t *off, int n, int64_t ld, int valid) {
#pragma unroll
        for (int it = 0; it < n; ++it) {
            const int r = chunk_index(shape, it);
            off[it] = shape == kKC ? (int64_t)min(r, valid - 1) * ld + (t & 7) * 8 : (int64_t)r * ld + min((t & 15) * 8, (valid - 1) & ~7);
        }
    };
    set_offsets(PSHAPE, p_off, NP, prm.ldp, p_valid);
    set_offsets(QSHAPE, q_off, NQ, prm.ldq, q_valid);
    auto fetch = [&](int shape, u32x4 *dst, int n, const T *base, const int64_t *off, int64_t ld, int valid, int extent,
                     int row_elems, int k0) {
        const T *slab = base + (shape == kKC ? (int64_t)k0 : (int64_t)k0 * ld);
        // A chunk that runs past the end of its [contraction][index] row brings in what is not stored: the first
        // elements of the row below, of which there is one unless this is the last slab.  (Nothing touches what these
        // loads return before the products of the slab before; the other branch waits for its loads at once.)
        if (k0 + BK <= K && (shape == kKC || valid == extent || (k0 + BK < K && row_elems >= 8))) {
#pragma unroll
            for (int it = 0; it < n; ++it) dst[it] = load_unaligned(slab + off[it]);
        } else {
            const bool back = (shape == kKC ? K : row_elems) >= 8;
            const T *safe = shape == kKC ? base : base + min(0, valid - 8);
#pragma unroll
            for (int it = 0; it < n; ++it) {
                const int r = chunk_index(shape, it);
                const int left = shape == kKC ? K - k0 - (t & 7) * 8 : (k0 + r < K ? valid - min((t & 15) * 8, (valid - 1) & ~7) : 0);
                dst[it] = load_part(slab + off[it], safe, left, back);
            }
        }
    };
    auto put = [&](int shape, const u32x4 *src, int n, unsigned char *to) {
        for (int it = 0; it < n; ++it) {
            const int r = chunk_index(shape, it);
            const int at = shape == kKC ? r * 128 + (((t & 7) ^ swz(r)) << 4) : r * 256 + (((t & 15) ^ mc_swz<T>(r)) << 4);
            *(u32x4 *)(to + at) = src[it];
        }
    };
    // -- fragments, as in gemm_kernel.hpp: block j of step ks
    auto frag = [&](int shape, const unsigned char *buf, int j, int ks) -> u32x4 {
        if (shape == kKC) return *(const u32x4 *)(buf + (16 * j + lb) * 128 + (((4 * ks + hq) ^ swz(lb)) << 4));
        typedef short s16x4 __attribute__((ext_vector_type(4)));
        typedef __attribute__((address_space(3))) s16x4 *lds_s16x4_ptr;
        const int kb = ks * 32 + hq * 8 + (lb >> 2);
        const unsigned char *at = buf + kb * 256 + (((2 * j + ((lb >> 1) & 1)) ^ mc_swz<T>(kb)) << 4) + (lb & 1) * 8;
        const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4_ptr)(at));
        const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4_ptr)(at + 1024));
        const u32x2 l2 = __builtin_bit_cast(u32x2, lo), h2 = __builtin_bit_cast(u32x2, hi);
        return u32x4{l2[0], l2[1], h2[0], h2[1]};
    };

    // Block row y of a wave.  Ragged rows: every other one, so that both pairs of waves have some of an expert's few
    // rows and the epilogue ends at the last of them.
    auto row_block = [&](int y) { return RAGGED == kRaggedRows ? 2 * y + wm : TJ * wm + y; };

    f32x4 acc[TI][TJ], bacc[kBiasGrad ? TJ : 1];
#pragma unroll
    for (int x = 0; x < TI; ++x)
#pragma unroll
        for (int y = 0; y < TJ; ++y) acc[x][y] = f32x4{0.f, 0.f, 0.f, 0.f};
    if (kBiasGrad) {
#pragma unroll
        for (int y = 0; y < TJ; ++y) bacc[y] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
    const bool want_bias = kBiasGrad && prm.bias_grad != nullptr && n0 == 0 && wn == 0;
    const uint32_t one2 = std::is_same<T, __bf16>::value ? 0x3f803f80u : 0x3c003c00u;
    const u32x4 ones = {one2, one2, one2, one2};

    u32x4 pr[NP], qr[NQ];
    const int n_slabs = (K + BK - 1) / BK;
    if (n_slabs > 0) {
        fetch(PSHAPE, pr, NP, P, p_off, prm.ldp, p_valid, BN, prm.n_cols, 0);
        fetch(QSHAPE, qr, NQ, Q, q_off, prm.ldq, q_valid, BM, prm.n_rows, 0);
    }
    for (int s = 0; s < n_slabs; ++s) {
        unsigned char *buf = smem + (s & 1) * STAGE;
        put(PSHAPE, pr, NP, buf);
        put(QSHAPE, qr, NQ, buf + P_BYTES);
        // (one barrier a slab: the other buffer, written next, was last read before it)
        __syncthreads();
        if (s + 1 < n_slabs) {
            fetch(PSHAPE, pr, NP, P, p_off, prm.ldp, p_valid, BN, prm.n_cols, (s + 1) * BK);
            fetch(QSHAPE, qr, NQ, Q, q_off, prm.ldq, q_valid, BM, prm.n_rows, (s + 1) * BK);
        }
#pragma unroll
        for (int ks = 0; ks < 2; ++ks) {
            u32x4 pf[TI], qf[TJ];
#pragma unroll
            for (int x = 0; x < TI; ++x) pf[x] = frag(PSHAPE, buf, wn * TI + x, ks);
#pragma unroll
            for (int y = 0; y < TJ; ++y) qf[y] = frag(QSHAPE, buf + P_BYTES, row_block(y), ks);
#pragma unroll
            for (int x = 0; x < TI; ++x)
#pragma unroll
                for (int y = 0; y < TJ; ++y) Elem<T>::mma(acc[x][y], pf[x], qf[y]);
            if (kBiasGrad && want_bias) {
#pragma unroll
                for (int y = 0; y < TJ; ++y) Elem<T>::mma(bacc[y], ones, qf[y]);
            }
        }
    }
    __syncthreads();

    // -- epilogue: acc[x][y][i] is C(row 16 row_block(y) + lb, column 64 wn + 16 x + 4 hq + i); sixteen rows at a
    // time through 2 KiB of LDS per wave and out as 128-byte row pieces
    unsigned char *stg = smem + wave * 2048;
    T *C = (T *)prm.C + c_off, *aux = prm.aux ? (T *)prm.aux + c_off : nullptr;
    const bool accumulate = RAGGED == kRaggedK && prm.accumulate_first && ei == 0;
    const T *bias = prm.bias ? (const T *)prm.bias + (int64_t)expert * prm.bias_expert_stride + n0 : nullptr;
    // (read once: in the loop, behind stores that might reach it as far as the compiler can tell, every use waited for those.  Forward
    // with GELU, 8192 rows, 8 experts of 2047 x 4093: 275 -> 225 us; with the epilogue's end at an expert's last rows
    // 556 rows, 64 of 38 x 1990: 50 -> 23)
    float bias_of[TI][4];
#pragma unroll
    for (int x = 0; x < TI; ++x)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int col = 64 * wn + 16 * x + 4 * hq + i;
            bias_of[x][i] = bias != nullptr && col < p_valid ? (float)bias[col] : 0.f;
        }
    auto wave_sync = [&]() {
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
        __builtin_amdgcn_wave_barrier();
    };
    auto store_rows = [&](T *to, int y) {
        wave_sync();
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const int r = i * 8 + (lane >> 3), c = lane & 7;
            const u32x4 v = *(const u32x4 *)(stg + r * 128 + ((c ^ (r & 7)) << 4));
            const int row = 16 * row_block(y) + r, col = 64 * wn + c * 8;
            if (row < q_valid && col < p_valid) {
                T *p = to + (int64_t)row * prm.ldc + col;
                if (col + 8 <= p_valid) {
                    __builtin_memcpy(p, &v, 16);
                } else {
                    const T *e = (const T *)&v;
#pragma unroll
                    for (int j = 0; j < 7; ++j)
                        if (col + j < p_valid) p[j] = e[j];
                }
            }
        }
        wave_sync();
    };
#pragma unroll
    for (int y = 0; y < TJ; ++y) {
        if (16 * row_block(y) >= q_valid) break;
        const int row = 16 * row_block(y) + lb;
#pragma unroll
        for (int kind = 1; kind >= 0; --kind) {   // 1: the pre-activation, 0: the result
            if (kind == 1 && (prm.epilogue != kEpiBiasAct || aux == nullptr)) continue;
#pragma unroll
            for (int x = 0; x < TI; ++x) {
                alignas(8) T res[4];
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const int col = 64 * wn + 16 * x + 4 * hq + i;
                    const bool in = row < q_valid && col < p_valid;
                    float v = acc[x][y][i] + bias_of[x][i];
                    if (kind == 0 && prm.epilogue == kEpiBiasAct) v = apply_act<false>(v, prm.activation);
                    if (prm.epilogue == kEpiDAct) v *= act_grad<false>(in ? (float)aux[(int64_t)row * prm.ldc + col] : 0.f, prm.activation);
                    if (accumulate) v += in ? (float)C[(int64_t)row * prm.ldc + col] : 0.f;
                    res[i] = (T)v;
                }
                *(u32x2 *)(stg + lb * 128 + (((2 * x + (hq >> 1)) ^ (lb & 7)) << 4) + (hq & 1) * 8) = *(const u32x2 *)res;
            }
            store_rows(kind == 1 ? aux : C, y);
        }
        if (kBiasGrad && want_bias && hq == 0 && row < q_valid) {
            T *dst = (T *)prm.bias_grad + (int64_t)expert * prm.n_rows + m0 + row;
            *dst = (T)(bacc[y][0] + (accumulate ? (float)*dst : 0.f));
        }
    }
#endif
}

template <typename T, int BM, int PS, int QS, int RG>
int launch_unaligned_tiles(GemmParams &prm, int epilogue, hipStream_t stream) {
    prm.epilogue = epilogue;
    prm.tiles_n = (int)ceil_div(prm.n_cols, kUaBN);
    prm.tiles_m = RG == kRaggedRows ? 0 : (int)ceil_div(prm.n_rows, BM);
    int64_t row_tiles = (int64_t)prm.tab.n * prm.tiles_m;
    if (RG == kRaggedRows && prm.dev_tab != nullptr) {
        row_tiles = segtab::cap_tiles(prm.dev_rows_cap, prm.tab.n, 128) * (128 / BM);
        prm.dev_map_off = (int32_t)segtab::map128_off(prm.dev_rows_cap, prm.tab.n);
    } else if (RG == kRaggedRows) {
        row_tiles = prm.tab.tile[prm.tab.n];
    }
    const int64_t total = row_tiles * prm.tiles_n;
    if (total > (int64_t)INT32_MAX - 8) return fail(FMOE_ELIMIT, "grouped GEMM: %lld tiles exceed the grid limit", (long long)total);
    if (total == 0) return FMOE_OK;
    prm.total_tiles = (int)total;
    ProfileScope prof(prm.profile_class, prm.profile_work, stream);
    grouped_gemm_unaligned_kernel<T, BM, PS, QS, RG><<<(unsigned)((total + 7) / 8 * 8), kUaThreads, 0, stream>>>(prm);
    FMOE_LAUNCH_CHECK();
    return FMOE_OK;
}

template <typename T> int launch_unaligned_typed(GemmParams &prm, int product, int epilogue, hipStream_t stream) {
    const bool low = prm.block_m == 64;
    switch (product) {
        case 0:
            return low ? launch_unaligned_tiles<T, 64, kKC, kKC, kRaggedRows>(prm, epilogue, stream)
                       : launch_unaligned_tiles<T, 128, kKC, kKC, kRaggedRows>(prm, epilogue, stream);
        case 1:
            return low ? launch_unaligned_tiles<T, 64, kMC, kKC, kRaggedRows>(prm, epilogue, stream)
                       : launch_unaligned_tiles<T, 128, kMC, kKC, kRaggedRows>(prm, epilogue, stream);
    }
    return launch_unaligned_tiles<T, 128, kMC, kMC, kRaggedK>(prm, epilogue, stream);
}

}  // namespace

// product: 0 forward, 1 data gradient, 2 weight gradient (with the bias gradient).  Ragged rows: prm.block_m (64 or 128)
// is the tile height, for which prm.tab was filled in (a device table serves both).
int launch_mfma_unaligned(gemm::GemmParams &prm, int dtype, int product, int epilogue, hipStream_t stream) {
    if (dtype == FMOE_BF16) return launch_unaligned_typed<__bf16>(prm, product, epilogue, stream);
    if (dtype == FMOE_F16) return launch_unaligned_typed<_Float16>(prm, product, epilogue, stream);
    return fail(FMOE_EINVAL, "grouped GEMM: dtype %d is not a 16-bit float type", dtype);
}

}  // namespace fmoe
