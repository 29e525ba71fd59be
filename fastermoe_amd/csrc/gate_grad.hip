// Backward of the gate's linear layer from the gradient of the selected scores (gfx950).
//
// The gate names top_k experts per token and its scores are their logits x . w_e + b_e
// (fmoe/gates/naive_gate.py:26-42), so the gradient of the logits has top_k entries per token.  As autograd runs
// it, those entries are written into a dense [tokens, experts] matrix and go through two library products a few columns wide, two
// reductions for the bias and one more pass over the input gradient to add the gate's part:
//   grad_x[t] = experts' part + sum_j g[t,j] w[idx[t,j]]      grad_w[e] = sum over (t,j) with idx = e of g[t,j] x[t]
// Here the gate's part of the first is a sum of top_k rows of w per token (a caller that has the experts' part as rows, as the layer's
// backward does, gets both sums in one pass), and the second is one pass over x with the matrix cores.
#include "gate_grad.hpp"
#include "profile.hpp"
#include "vec16.hpp"

#include <type_traits>

namespace fmoe {
namespace {

constexpr int kBlock = 256;
constexpr int kWavesPerBlock = kBlock / kWave;
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));

// ---- input gradient: reduce_slots plus the gate's part ---------------------------------------
// A wave owns P pieces of 64 vectors (1 KiB) of one token's row and takes its slots K at a time, with all K P loads of rows and of w in
// flight together: the slots' experts (and rows) are a dependent load before them, scalar ones as they are the same for the wave, and w's
// rows come from the caches.  The layer's backward hands in the experts' rows, the gate's own node asks for its part alone (rows null).
// us for the gate's part with P = 1 / 2 / 4 and all slots at a time (and with the rows, against reduce_slots alone): bf16, 32768 tokens of
// 4096, 8 experts, top-2: 73 / 62 / 69 (147 / 141 / 150, 133), 16384 of 2048, 64 experts, top-1: 15.0 / 12.3 / 12.8
// (27.9 / 25.5 / 26.7, 23.5), 16384 of 4096, top-4: 55 / 54 / 64; float32, 32768 of 4096, top-2: 115 / 87 / 81, top-4 at 16384:
// 87 / 71 / 84.  As a library product over the dense gradient the first took 99.
// Tokens or rows too few for that many waves take P = 1.
// More than two slots: 16-bit types two at a time, so that seven or eight waves fit a SIMD where the loads of all slots and pieces at once leave four
// (top-8, 8192 tokens of 2048, 256 experts: 71.7 -> 56.4 us, 32768 of 512: 72.0 -> 58.2; top-4, 16384 of 4096: 120.5 -> 113.4, 8192 of
// 1024: 17.8 either way; launches that leave the chip waves to spare wait twice, 64 tokens of 2048, top-8: 5.7 -> 6.1; the order of the sums
// is the same).  float32 as many as there are, whose rows are twice the bytes for the same sums (8192 of
// 2048, top-8: 103.4, two at a time 107.3).
// ANY (16-bit types): rows of any length, read 16 bytes at a time wherever they lie; row_vecs counts the last, partial piece.
template <typename T, int K, int P, bool ANY>
__global__ __launch_bounds__(kBlock) void reduce_slots_gate_kernel(
    const u32x4 *__restrict__ rows, const int64_t *__restrict__ slot_to_row, const T *__restrict__ grad_score,
    const int64_t *__restrict__ topk_idx, const u32x4 *__restrict__ w, u32x4 *__restrict__ out, int64_t n_tokens, int top_k,
    int64_t n_rows, int n_expert, int row_vecs, int groups_per_row, int row_elems) {
    // vector v of row r
    auto load = [&](const u32x4 *base, int64_t r, int v, auto once) {
        if constexpr (ANY) {
            return load_some((const T *)base + r * row_elems + v * 8, row_elems - v * 8);
        } else {
            const u32x4 *at = &base[r * row_vecs + v];
            if constexpr (decltype(once)::value) return __builtin_nontemporal_load(at); else return *at;
        }
    };
    const int lane = threadIdx.x & (kWave - 1);
    // one token per wave: its slots' rows, experts and gradients are scalar loads
    const uint32_t group = __builtin_amdgcn_readfirstlane(blockIdx.x * kWavesPerBlock + threadIdx.x / kWave);
    const int64_t t = __builtin_amdgcn_readfirstlane(group / (uint32_t)groups_per_row);
    if (t >= n_tokens) return;
    const int v0 = (int)(group - (uint32_t)t * (uint32_t)groups_per_row) * (P * kWave) + lane;
    float acc[P][8] = {}, gate[P][8] = {};
    for (int j0 = 0; j0 < top_k; j0 += K) {
        u32x4 val[P][K], wv[P][K];
        float g[K];
#pragma unroll
        for (int j = 0; j < K; ++j) {
            const bool has = j0 + j < top_k;
            const int64_t s = t * top_k + (has ? j0 + j : 0);
            const int64_t src = has && slot_to_row ? slot_to_row[s] : -1, e = topk_idx[s];
            const bool live = src >= 0 && src < n_rows, named = has && e >= 0 && e < n_expert;
            g[j] = named ? (float)grad_score[s] : 0.f;
#pragma unroll
            for (int p = 0; p < P; ++p) {
                const int v = v0 + p * kWave;
                val[p][j] = live && v < row_vecs ? load(rows, src, v, std::true_type{}) : u32x4{0, 0, 0, 0};
                wv[p][j] = named && v < row_vecs ? load(w, e, v, std::false_type{}) : u32x4{0, 0, 0, 0};
            }
        }
#pragma unroll
        for (int j = 0; j < K; ++j)
#pragma unroll
            for (int p = 0; p < P; ++p) {
                float f[8];
                Vec<T>::unpack(val[p][j], f);
#pragma unroll
                for (int i = 0; i < Vec<T>::N; ++i) acc[p][i] += f[i];
                Vec<T>::unpack(wv[p][j], f);
#pragma unroll
                for (int i = 0; i < Vec<T>::N; ++i) gate[p][i] += g[j] * f[i];
            }
    }
#pragma unroll
    for (int p = 0; p < P; ++p) {
        const int v = v0 + p * kWave;
        if (v >= row_vecs) continue;
#pragma unroll
        for (int i = 0; i < Vec<T>::N; ++i) acc[p][i] += gate[p][i];
        if constexpr (ANY) store_some((T *)out + t * row_elems + v * 8, Vec<T>::pack(acc[p]), row_elems - v * 8);
        else __builtin_nontemporal_store(Vec<T>::pack(acc[p]), &out[t * row_vecs + v]);
    }
}

template <typename T, int K, bool ANY>
int launch_reduce_gate(const void *rows, const int64_t *slot_to_row, const void *grad_score, const int64_t *topk_idx, const void *w,
                       void *out, int64_t n_tokens, int64_t top_k, int64_t n_rows, int64_t n_expert, int64_t row_elems,
                       hipStream_t st) {
    const int64_t row_vecs = ceil_div(row_elems * (int64_t)sizeof(T), 16);
    constexpr int kPieces = K >= 8 ? 1 : K == 4 || sizeof(T) == 2 ? 2 : 4;   // (K 4 and 8: float32)
#define FMOE_RG(P)                                                                                                                    \
    {                                                                                                                                 \
        const int64_t groups = ceil_div(row_vecs, (P) * kWave), blocks = ceil_div(n_tokens * groups, kWavesPerBlock);                  \
        if (blocks > INT32_MAX / kWavesPerBlock) return fail(FMOE_ELIMIT, "fmoe_reduce_slots_gate: grid too large");                   \
        reduce_slots_gate_kernel<T, K, P, ANY><<<(int)blocks, kBlock, 0, st>>>((const u32x4 *)rows, slot_to_row, (const T *)grad_score,     \
                                                                         topk_idx, (const u32x4 *)w, (u32x4 *)out, n_tokens,          \
                                                                         (int)top_k, n_rows, (int)n_expert, (int)row_vecs,            \
                                                                         (int)groups, (int)row_elems);                                \
    }
    if (kPieces > 1 && row_vecs >= kPieces * kWave && n_tokens * row_vecs >= (int64_t)kPieces * kWave * 4096) FMOE_RG(kPieces)
    else FMOE_RG(1)
#undef FMOE_RG
    FMOE_LAUNCH_CHECK();
    return FMOE_OK;
}

// ---- weight gradient --------------------------------------------------------------------------
// grad_w = G^T x with G [tokens, experts] holding top_k entries per token.  A workgroup takes kCols columns of x and a
// range of tokens, kTok at a time: the tokens' entries of G are scattered into an LDS tile [expert][token] that is zero
// otherwise, the columns go to LDS as they lie, and the four waves multiply (every wave all experts, 32 columns), with x and the
// entries of the next tokens on their way.  The sums over
// the token ranges go to memory in float32 and are added in the order of the ranges by a second kernel.
// Bound by reading x once: 32768 tokens of 4096 and 8 experts 45 us (5.9 TB/s; 198 as a library product over the dense G), 16384 x 2048
// and 64 experts 26 (139), 8192 x 2048 and 256 experts, where the chain of steps bounds it, 46 (70).
constexpr int kCols = 128;
template <typename T> constexpr int tokens_per_step() { return sizeof(T) == 2 ? 64 : 32; }
template <typename T> constexpr int g_stride() { return tokens_per_step<T>() + 16 / (int)sizeof(T); }   // elements per expert

template <typename T, int EB, bool ANY>   // EB: blocks of 16 experts; ANY (16-bit types): rows of x of any length
__global__ __launch_bounds__(kBlock) void gate_wgrad_kernel(const T *__restrict__ grad_score, const int64_t *__restrict__ topk_idx,
                                                            const T *__restrict__ x, float *__restrict__ part_w,
                                                            float *__restrict__ part_b, int n_tokens, int d, int n_expert, int top_k,
                                                            int tokens_per_range) {
    constexpr int kTok = tokens_per_step<T>(), kGS = g_stride<T>();
    constexpr int CE = 16 / (int)sizeof(T), CPR = kCols / CE;            // chunks per row of the tile
    constexpr int kLoads = kTok * CPR / kBlock;                          // 16-byte chunks per thread
    extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
    unsigned char *xt = lds;                                             // [kTok][kCols], 16-bit: chunks swizzled
    T *gt = (T *)(lds + kTok * kCols * sizeof(T));                       // [16 EB][kGS]
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6, lb = lane & 15, hq = lane >> 4;
    const int c0 = blockIdx.x * kCols;
    const int lo = blockIdx.y * tokens_per_range, hi = min(n_tokens, lo + tokens_per_range);
    // The bias gradient, in the workgroups of the first columns.  16-bit types: one more column of products in the first
    // wave.  float32: the rows of the LDS tile are added in double, as a chain of products over a long range is further from the
    // exact sum than what it replaces (32768 tokens that all name 4 experts, relative error 1.0e-6; as one more
    // pass of torch's sum over the dense gradient 7.7e-8; added like this 2.9e-8); lane and wave are expert and part of the tokens.
    constexpr bool kWideBias = sizeof(T) == 4;
    constexpr int kBiasExperts = EB <= 4 ? 64 : EB * 16, kBiasParts = kBlock / kBiasExperts, kBiasTok = kTok / kBiasParts;
    const bool bias_wg = part_b != nullptr && blockIdx.x == 0, with_bias = !kWideBias && bias_wg && wave == 0;
    const int bias_e = t % kBiasExperts, bias_part = t / kBiasExperts;
    double bias_sum = 0.;

    for (int i = t; i < EB * 16 * kGS; i += kBlock) gt[i] = (T)0.f;
    f32x4 acc[EB][2], bacc[EB];
#pragma unroll
    for (int e = 0; e < EB; ++e) {
        acc[e][0] = acc[e][1] = bacc[e] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
    // chunk c of token row k is stored at c ^ swizzle(k) (16-bit types, for the transposing reads)
    auto swizzle = [](int k) { return sizeof(T) == 2 ? ((k & 3) << 2) | (((k >> 3) & 1) << 1) : 0; };
    u32x4 ahead[kLoads];
    auto load_x = [&](int t0) {
#pragma unroll
        for (int i = 0; i < kLoads; ++i) {
            const int q = i * kBlock + t, k = q / CPR, c = q % CPR;
            const T *at = x + (int64_t)(t0 + k) * d + c0 + c * CE;
            const bool in = t0 + k < hi && c0 + c * CE < d;
            if constexpr (ANY) ahead[i] = in ? load_some(at, d - (c0 + c * CE)) : u32x4{0, 0, 0, 0};
            else ahead[i] = in ? *(const u32x4 *)at : u32x4{0, 0, 0, 0};
        }
    };
    // this step's first kHeld entries per thread are loaded a step ahead and kept until they are cleared again
    constexpr int kHeld = 2;
    int held_e[kHeld], next_e[kHeld];
    T held_g[kHeld], next_g[kHeld];
    auto load_g = [&](int t0) {
#pragma unroll
        for (int h = 0; h < kHeld; ++h) {
            const int i = h * kBlock + t;
            const int64_t s = (int64_t)t0 * top_k + i;
            next_e[h] = -1;
            if (i < kTok * top_k && s < (int64_t)hi * top_k) {
                const int64_t e = topk_idx[s];
                if (e >= 0 && e < n_expert) next_e[h] = (int)e;
                next_g[h] = grad_score[s];
            }
        }
    };
    auto scatter_g = [&](int t0, bool clear) {
#pragma unroll
        for (int h = 0; h < kHeld; ++h)
            if (held_e[h] >= 0) gt[held_e[h] * kGS + (h * kBlock + t) / top_k] = clear ? (T)0.f : held_g[h];
        for (int i = kHeld * kBlock + t; i < kTok * top_k; i += kBlock) {
            const int k = i / top_k;
            if (t0 + k >= hi) break;
            const int64_t s = (int64_t)t0 * top_k + i;
            const int64_t e = topk_idx[s];
            if (e >= 0 && e < n_expert) gt[e * kGS + k] = clear ? (T)0.f : grad_score[s];
        }
    };
    load_g(lo);
    load_x(lo);
    __syncthreads();
    for (int t0 = lo; t0 < hi; t0 += kTok) {
#pragma unroll
        for (int i = 0; i < kLoads; ++i) {
            const int q = i * kBlock + t, k = q / CPR, c = q % CPR;
            *(u32x4 *)(xt + (k * CPR + (c ^ swizzle(k))) * 16) = ahead[i];
        }
#pragma unroll
        for (int h = 0; h < kHeld; ++h) {
            held_e[h] = next_e[h];
            held_g[h] = next_g[h];
        }
        scatter_g(t0, false);
        __syncthreads();
        if (t0 + kTok < hi) {
            load_x(t0 + kTok);
            load_g(t0 + kTok);
        }
        if constexpr (sizeof(T) == 2) {
            const uint32_t one2 = std::is_same<T, __bf16>::value ? 0x3f803f80u : 0x3c003c00u;
            const u32x4 ones = {one2, one2, one2, one2};
            auto mma = [](f32x4 &c, const u32x4 &a, const u32x4 &b) {
                if constexpr (std::is_same<T, __bf16>::value)
                    c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
                else
                    c = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
            };
#pragma unroll
            for (int ks = 0; ks < kTok / 32; ++ks) {
                u32x4 b[2];
#pragma unroll
                for (int cb = 0; cb < 2; ++cb) {
                    // the transposing read hands lane (lb, hq) column lb of its block at tokens 8 hq .. 8 hq + 7 (two reads of four)
                    typedef short s16x4 __attribute__((ext_vector_type(4)));
                    typedef __attribute__((address_space(3))) s16x4 *lds_s16x4_ptr;
                    const int col = wave * 32 + cb * 16 + 4 * (lb & 3), k = ks * 32 + hq * 8 + (lb >> 2);
                    const unsigned char *at = xt + (k * CPR + ((col >> 3) ^ swizzle(k))) * 16 + (col & 7) * 2;
                    const s16x4 a0 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4_ptr)(at));
                    const s16x4 a1 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4_ptr)(at + 4 * CPR * 16));
                    const u32x2 l2 = __builtin_bit_cast(u32x2, a0), h2 = __builtin_bit_cast(u32x2, a1);
                    b[cb] = u32x4{l2[0], l2[1], h2[0], h2[1]};
                }
#pragma unroll
                for (int e = 0; e < EB; ++e) {
                    const u32x4 a = *(const u32x4 *)(gt + (e * 16 + lb) * kGS + ks * 32 + hq * 8);
                    mma(acc[e][0], a, b[0]);
                    mma(acc[e][1], a, b[1]);
                    if (with_bias) mma(bacc[e], a, ones);
                }
            }
        } else {
            const float *xf = (const float *)xt, *gf = (const float *)gt;
#pragma unroll
            for (int ks = 0; ks < kTok / 4; ++ks) {
                const int k = ks * 4 + hq;
                const float b0 = xf[k * kCols + wave * 32 + lb], b1 = xf[k * kCols + wave * 32 + 16 + lb];
#pragma unroll
                for (int e = 0; e < EB; ++e) {
                    const float a = gf[(e * 16 + lb) * kGS + k];
                    acc[e][0] = __builtin_amdgcn_mfma_f32_16x16x4f32(a, b0, acc[e][0], 0, 0, 0);
                    acc[e][1] = __builtin_amdgcn_mfma_f32_16x16x4f32(a, b1, acc[e][1], 0, 0, 0);
                }
            }
            if (bias_wg && bias_e < EB * 16) {
#pragma unroll
                for (int k = 0; k < kBiasTok; k += 4) {
                    const f32x4 v = *(const f32x4 *)(gf + bias_e * kGS + bias_part * kBiasTok + k);
                    bias_sum += ((double)v[0] + (double)v[1]) + ((double)v[2] + (double)v[3]);
                }
            }
        }
        __syncthreads();
        scatter_g(t0, true);   // the entries of these tokens are zero again before the next ones are scattered
        __syncthreads();
    }
    // lane (lb, hq) holds experts 4 hq .. 4 hq + 3 of every expert block at column lb of its column blocks
#pragma unroll
    for (int e = 0; e < EB; ++e)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int ex = e * 16 + 4 * hq + i;
            if (ex >= n_expert) continue;
            float *dst = part_w + ((int64_t)blockIdx.y * n_expert + ex) * d;
#pragma unroll
            for (int cb = 0; cb < 2; ++cb) {
                const int c = c0 + wave * 32 + cb * 16 + lb;
                if (c < d) dst[c] = acc[e][cb][i];
            }
            if (with_bias && lb == 0) part_b[(int64_t)blockIdx.y * n_expert + ex] = bacc[e][i];
        }
    if (kWideBias && bias_wg) {   // (uniform over the workgroup; the tiles were last read before the barrier that ends the loop)
        double *sums = (double *)lds;   // [kBiasParts][kBiasExperts]
        sums[t] = bias_sum;
        __syncthreads();
        if (t < kBiasExperts && t < n_expert) {
#pragma unroll
            for (int q = 1; q < kBiasParts; ++q) bias_sum += sums[q * kBiasExperts + t];
            part_b[(int64_t)blockIdx.y * n_expert + t] = (float)bias_sum;
        }
    }
}

// adds the ranges' sums in ascending order (float32 results: in double): elements [0, n_w) are grad_w's, the n_b after
// them grad_b's
template <typename T>
__global__ __launch_bounds__(kBlock) void gate_wgrad_reduce_kernel(const float *__restrict__ part_w, const float *__restrict__ part_b,
                                                                   T *__restrict__ grad_w, T *__restrict__ grad_b, int64_t n_w,
                                                                   int n_b, int ranges) {
    const int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x;
    if (i >= n_w + n_b) return;
    const float *src = i < n_w ? part_w + i : part_b + (i - n_w);
    const int64_t step = i < n_w ? n_w : n_b;
    typename std::conditional<sizeof(T) == 4, double, float>::type sum = 0;
    for (int r0 = 0; r0 < ranges; r0 += 8) {
        float v[8];
#pragma unroll
        for (int r = 0; r < 8; ++r) v[r] = src[(int64_t)min(r0 + r, ranges - 1) * step];
        // (the eight loads are out before the first is waited for: with the conversion to double at each, or a condition around
        // it, they go one by one, 19 us instead of 5 for 64 ranges)
#pragma unroll
        for (int r = 0; r < 8; ++r) asm volatile("" : "+v"(v[r]));
#pragma unroll
        for (int r = 0; r < 8; ++r) sum += r0 + r < ranges ? v[r] : 0.f;
    }
    if (i < n_w) grad_w[i] = (T)sum;
    else grad_b[i - n_w] = (T)sum;
}

constexpr int kMaxGateExpert = 256;

// token ranges of the weight gradient: about 512 workgroups in all (two per CU; 16384 x 2048 and 64 experts take 26 us with 512, 33 with
// 1024 and 45 with 2048, for the sums that have to be added), each of at least 64 tokens, and no more float32 sums than half of
// what is read (8192 x 2048 and 256 experts: 46 us, 63 with twice and 65 with half of that)
int wgrad_ranges(int64_t n_tokens, int64_t d, int64_t n_expert) {
    const int64_t cols = ceil_div(d, kCols);
    int64_t r = ceil_div(512, cols);
    if (r > ceil_div(n_tokens, 64)) r = ceil_div(n_tokens, 64);
    if (r > n_tokens / (2 * n_expert)) r = n_tokens / (2 * n_expert);
    return (int)(r < 1 ? 1 : r);
}

template <typename T, bool ANY>
int launch_wgrad(const void *grad_score, const int64_t *topk_idx, const void *x, void *grad_w, void *grad_b, int64_t n_tokens,
                 int64_t d, int64_t n_expert, int64_t top_k, float *ws, hipStream_t st) {
    const int ranges = wgrad_ranges(n_tokens, d, n_expert);
    const int64_t step = tokens_per_step<T>();
    const int per_range = (int)(ceil_div(ceil_div(n_tokens, ranges), step) * step);
    float *part_w = ws, *part_b = grad_b ? ws + (int64_t)ranges * n_expert * d : nullptr;
    const dim3 grid((unsigned)ceil_div(d, kCols), (unsigned)ranges);
    const int eb = n_expert <= 16 ? 1 : n_expert <= 32 ? 2 : n_expert <= 64 ? 4 : n_expert <= 128 ? 8 : 16;
    const size_t lds = (tokens_per_step<T>() * kCols + eb * 16 * g_stride<T>()) * sizeof(T);
#define FMOE_GW(EB)                                                                                                          \
    gate_wgrad_kernel<T, EB, ANY><<<grid, kBlock, lds, st>>>((const T *)grad_score, topk_idx, (const T *)x, part_w, part_b,        \
                                                        (int)n_tokens, (int)d, (int)n_expert, (int)top_k, per_range)
    switch (eb) {
        case 1: FMOE_GW(1); break;
        case 2: FMOE_GW(2); break;
        case 4: FMOE_GW(4); break;
        case 8: FMOE_GW(8); break;
        default: FMOE_GW(16); break;
    }
#undef FMOE_GW
    FMOE_LAUNCH_CHECK();
    const int64_t n_w = n_expert * d, n_b = grad_b ? n_expert : 0;
    gate_wgrad_reduce_kernel<T><<<(unsigned)ceil_div(n_w + n_b, kBlock), kBlock, 0, st>>>(part_w, part_b, (T *)grad_w, (T *)grad_b, n_w,
                                                                                         (int)n_b, ranges);
    FMOE_LAUNCH_CHECK();
    return FMOE_OK;
}

}  // namespace

bool gate_grad_any_grid(int64_t d_model, int64_t n_expert, int64_t top_k, int dtype) {
    return fmoe_gate_grad_supported(d_model, n_expert, top_k, dtype) == 1 ||
           (dtype_bytes(dtype) == 2 && n_expert >= 1 && n_expert <= kMaxGateExpert && top_k >= 1 && top_k <= n_expert && d_model >= 1 &&
            d_model < (1 << 24));
}

int gate_weight_grad(const void *grad_score, const int64_t *topk_idx, const void *x, void *grad_w, void *grad_b, int64_t n_tokens,
                     int64_t d_model, int64_t n_expert, int64_t top_k, int dtype, void *workspace, int64_t workspace_bytes, hipStream_t st) {
    if (!gate_grad_any_grid(d_model, n_expert, top_k, dtype))
        return fail(FMOE_ELIMIT, "fmoe_gate_weight_grad: d_model=%lld n_expert=%lld top_k=%lld dtype=%d is not taken", (long long)d_model,
                    (long long)n_expert, (long long)top_k, dtype);
    FMOE_REQUIRE(n_tokens >= 1 && n_tokens * top_k <= (int64_t)INT32_MAX, "fmoe_gate_weight_grad: n_tokens=%lld", (long long)n_tokens);
    FMOE_REQUIRE(grad_score && topk_idx && x && grad_w && aligned16(x), "fmoe_gate_weight_grad: NULL or misaligned pointer");
    const int64_t need = fmoe_gate_weight_grad_workspace_bytes(n_tokens, d_model, n_expert);
    if (workspace == nullptr || workspace_bytes < need)
        return fail(FMOE_EWORKSPACE, "fmoe_gate_weight_grad: needs %lld bytes of workspace, got %lld", (long long)need,
                    (long long)workspace_bytes);
    FMOE_REQUIRE((reinterpret_cast<uintptr_t>(workspace) & 3u) == 0, "fmoe_gate_weight_grad: the workspace must be 4-byte aligned");
    float *ws = (float *)workspace;
    const bool any = (d_model * dtype_bytes(dtype)) % 16 != 0;
#define FMOE_GWL(T, ANY) return launch_wgrad<T, ANY>(grad_score, topk_idx, x, grad_w, grad_b, n_tokens, d_model, n_expert, top_k, ws, st)
    if (dtype == FMOE_F32) FMOE_GWL(float, false);
    if (dtype == FMOE_BF16) {
        if (any) FMOE_GWL(__bf16, true);
        FMOE_GWL(__bf16, false);
    }
    if (any) FMOE_GWL(_Float16, true);
    FMOE_GWL(_Float16, false);
#undef FMOE_GWL
}

int reduce_slots_gate(const void *rows, const int64_t *slot_to_row, const void *grad_score, const int64_t *topk_idx, const void *w, void *out,
                      int64_t n_tokens, int64_t top_k, int64_t n_rows, int64_t n_expert, int64_t row_elems, int dtype, bool any_grid, hipStream_t st) {
    FMOE_REQUIRE(dtype == FMOE_F32 || dtype == FMOE_BF16 || dtype == FMOE_F16, "fmoe_reduce_slots_gate: dtype %d", dtype);
    FMOE_REQUIRE(n_tokens >= 0 && top_k >= 1 && n_rows >= 0 && n_expert >= 1 && row_elems >= 0, "fmoe_reduce_slots_gate: bad sizes");
    if (n_tokens == 0 || row_elems == 0) return FMOE_OK;
    if (n_tokens > (int64_t)INT32_MAX || top_k > 65536 || row_elems > (int64_t)(1 << 28) || n_expert > (int64_t)(1 << 24))
        return fail(FMOE_ELIMIT, "fmoe_reduce_slots_gate: sizes beyond the supported range");
    FMOE_REQUIRE(grad_score && topk_idx && w && out && (rows || n_rows == 0 || slot_to_row == nullptr), "fmoe_reduce_slots_gate: NULL pointer");
    const bool any = (row_elems * dtype_bytes(dtype)) % 16 != 0;
    FMOE_REQUIRE((!any || (any_grid && dtype != FMOE_F32)) && aligned16(rows) && aligned16(w) && aligned16(out),
                 "fmoe_reduce_slots_gate: misaligned pointer, or rows that are no whole 16-byte chunks");
    // (bytes: the experts' rows and the result; the gate's part alone: its weight, once, and the result)
    ProfileScope prof(kProfReduceSlots, (double)(slot_to_row ? (top_k + 1) * n_tokens : n_tokens + n_expert) * row_elems * dtype_bytes(dtype), st);
#define FMOE_RGT(T, K, ANY)                                                                                                       \
    return launch_reduce_gate<T, K, ANY>(rows, slot_to_row, grad_score, topk_idx, w, out, n_tokens, top_k, n_rows, n_expert, row_elems, st)
#define FMOE_RGK(T, ANY)                                                                                                          \
    {                                                                                                                             \
        if (top_k == 1) FMOE_RGT(T, 1, ANY);                                                                                      \
        FMOE_RGT(T, 2, ANY);                                                                                                      \
    }
    if (dtype == FMOE_F32) {
        if (top_k > 4) FMOE_RGT(float, 8, false);
        if (top_k > 2) FMOE_RGT(float, 4, false);
        FMOE_RGK(float, false)
    }
    if (dtype == FMOE_BF16) {
        if (any) FMOE_RGK(__bf16, true)
        FMOE_RGK(__bf16, false)
    }
    if (any) FMOE_RGK(_Float16, true)
    FMOE_RGK(_Float16, false)
#undef FMOE_RGK
#undef FMOE_RGT
}

}  // namespace fmoe

using namespace fmoe;

extern "C" int fmoe_gate_grad_supported(int64_t d_model, int64_t n_expert, int64_t top_k, int dtype) {
    if (dtype != FMOE_F32 && dtype != FMOE_BF16 && dtype != FMOE_F16) return 0;
    return (n_expert >= 1 && n_expert <= kMaxGateExpert && top_k >= 1 && top_k <= n_expert && d_model >= 1 && d_model < (1 << 24) &&
            (d_model * dtype_bytes(dtype)) % 16 == 0) ? 1 : 0;
}

extern "C" int64_t fmoe_gate_weight_grad_workspace_bytes(int64_t n_tokens, int64_t d_model, int64_t n_expert) {
    if (n_tokens < 1 || d_model < 1 || n_expert < 1) return 0;
    return (int64_t)wgrad_ranges(n_tokens, d_model, n_expert) * n_expert * (d_model + 1) * (int64_t)sizeof(float);
}

extern "C" int fmoe_gate_weight_grad(const void *grad_score, const int64_t *topk_idx, const void *x, void *grad_w, void *grad_b,
                                     int64_t n_tokens, int64_t d_model, int64_t n_expert, int64_t top_k, int dtype, void *workspace,
                                     int64_t workspace_bytes, void *stream) {
    if (!fmoe_gate_grad_supported(d_model, n_expert, top_k, dtype))
        return fail(FMOE_ELIMIT, "fmoe_gate_weight_grad: d_model=%lld n_expert=%lld top_k=%lld dtype=%d is not taken", (long long)d_model,
                    (long long)n_expert, (long long)top_k, dtype);
    return gate_weight_grad(grad_score, topk_idx, x, grad_w, grad_b, n_tokens, d_model, n_expert, top_k, dtype, workspace, workspace_bytes,
                            (hipStream_t)stream);
}

extern "C" int fmoe_gate_grad_any_supported(int64_t d_model, int64_t n_expert, int64_t top_k, int dtype) {
    return gate_grad_any_grid(d_model, n_expert, top_k, dtype) ? 1 : 0;
}

extern "C" int fmoe_gate_weight_grad_any(const void *grad_score, const int64_t *topk_idx, const void *x, void *grad_w, void *grad_b,
                                         int64_t n_tokens, int64_t d_model, int64_t n_expert, int64_t top_k, int dtype, void *workspace,
                                         int64_t workspace_bytes, void *stream) {
    return gate_weight_grad(grad_score, topk_idx, x, grad_w, grad_b, n_tokens, d_model, n_expert, top_k, dtype, workspace, workspace_bytes,
                            (hipStream_t)stream);
}

extern "C" int fmoe_reduce_slots_gate_any(const void *rows, const int64_t *slot_to_row, const void *grad_score, const int64_t *topk_idx,
                                          const void *w, void *out, int64_t n_tokens, int64_t top_k, int64_t n_rows, int64_t n_expert,
                                          int64_t row_elems, int dtype, void *stream) {
    return reduce_slots_gate(rows, slot_to_row, grad_score, topk_idx, w, out, n_tokens, top_k, n_rows, n_expert, row_elems, dtype, true,
                             (hipStream_t)stream);
}

extern "C" int fmoe_reduce_slots_gate(const void *rows, const int64_t *slot_to_row, const void *grad_score, const int64_t *topk_idx,
                                      const void *w, void *out, int64_t n_tokens, int64_t top_k, int64_t n_rows, int64_t n_expert,
                                      int64_t row_elems, int dtype, void *stream) {
    return reduce_slots_gate(rows, slot_to_row, grad_score, topk_idx, w, out, n_tokens, top_k, n_rows, n_expert, row_elems, dtype, false,
                             (hipStream_t)stream);
}
