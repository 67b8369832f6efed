// Matrix prefill of a bf16 decoder stack.  The reference prefills a prompt one position per
// worker step and leaves a matrix prefill as an open question (docs/development.md:331); this
// one runs up to kChunkRows positions through each layer at once.  Its arithmetic is the
// reference's full causal block (decoder_reference.py:273-312, recompute_prefix) with every
// rounding point of the decode path (docs/architecture.md:284-312), so that the cache rows it
// writes are the ones a position-by-position prefill writes, up to the FP32 summation order of
// the dot products:
//
//   u = bf16(bf16(x * rsqrt(mean(x^2) + eps)) * attn_norm)      norm_rows
//   q, k, v = bf16(W u)                                          GEMM (MFMA, FP32 sums)
//   q, k rotated as the worker rotates them; K, V rows -> cache  rope_rows
//   s = bf16(bf16(q . k) * (1 / sqrt(dh)));                       attention_tiles (causal: M the
//   P = bf16(exp(s - M) / S); attention = bf16(sum P v)          row's maximum, S its FP32 exp-sum)
//   r = bf16(bf16(Wo attention) + x)                             GEMM with the residual
//   z = RMSNorm(r) with ffn_norm                                 norm_rows
//   p = bf16(bf16(silu(bf16(Wgate z))) * bf16(Wup z))            one GEMM over both matrices
//   y = bf16(bf16(Wdown p) + r)                                  GEMM with the residual
//
// A GEMM too small for the chip splits K; the kernel after it adds the parts (norm_rows, rope_rows).
//
// The GEMMs are this library's MFMA kernel rather than a library's: rocBLAS, linked into this
// library, conflicted with the different rocBLAS build PyTorch ships, and a process that loaded
// this library before importing torch crashed.
#include "prefill.hpp"

#include <algorithm>
#include <type_traits>
#include <string>

#include "device_common.hpp"
#include "prefill_gemm.hpp"
#include "worker_config.hpp"

namespace tiles {
namespace {

using Bf = Num<true>;
constexpr int kRowThreads = 256;
constexpr int kTile = 64;  // key positions per attention tile

__device__ inline float bf(uint16_t bits) { return bf16_bits_to_float(bits); }
__device__ inline uint16_t bits16(float v) { return static_cast<uint16_t>(float_to_bf16_bits(v)); }

// The rows a GEMM left: bf16 rows (splits 1), or the FP32 sums of its parts of K, `plane` elements
// apart.
struct GemmRows {
    const uint16_t* rows;
    const float* partial;
    int splits;
    size_t plane;
};

// Eight adjacent values of a GEMM's rows from element `at`, rounded to bf16.  The number of parts is
// a template argument so that their loads are in flight together.
template <int kSplits>
__device__ inline void load_rows8(const GemmRows& g, size_t at, float (&v)[8])
{
    if constexpr (kSplits == 1) {
        const u32x4 bits = *reinterpret_cast<const u32x4*>(g.rows + at);
#pragma unroll
        for (int e = 0; e < 8; ++e)
            v[e] = Bf::elem(bits, e);
    } else {
        f32x4 part[kSplits][2];
#pragma unroll
        for (int p = 0; p < kSplits; ++p) {
            const f32x4* from = reinterpret_cast<const f32x4*>(g.partial + p * g.plane + at);
            part[p][0] = from[0];
            part[p][1] = from[1];
        }
#pragma unroll
        for (int p = 1; p < kSplits; ++p) {
            part[0][0] += part[p][0];
            part[0][1] += part[p][1];
        }
#pragma unroll
        for (int e = 0; e < 8; ++e)
            v[e] = Bf::round(part[0][e / 4][e % 4]);
    }
}

constexpr int kMostSplits = 8;
// f(std::integral_constant<int, splits>{}).
template <int kSplits = 1, typename F>
void with_splits(int splits, const F& f)
{
    if (splits == kSplits)
        f(std::integral_constant<int, kSplits>{});
    else if constexpr (kSplits < kMostSplits)
        with_splits<kSplits + 1>(splits, f);
}

// x[r] = the embedding row of tokens[r], 16 bytes a thread.
__global__ void __launch_bounds__(kRowThreads) gather_rows(const uint16_t* embedding, const ti_token_id* tokens, int d,
                                                           uint16_t* x)
{
    const u32x4* src = reinterpret_cast<const u32x4*>(embedding + static_cast<size_t>(tokens[blockIdx.x]) * d);
    u32x4* dst = reinterpret_cast<u32x4*>(x + static_cast<size_t>(blockIdx.x) * d);
    for (int i = threadIdx.x; i < d / 8; i += kRowThreads)
        dst[i] = src[i];
}

// out[r] = bf16(bf16(x[r] * inv_rms) * scale), inv_rms = 1 / sqrt(mean(x[r]^2) + eps) in FP32, as the
// worker's rms_apply computes it.  Of a GEMM that left parts (kSplits > 1), x[r] is
// bf16(bf16(sum) + residual[r]) and also goes to sum_out.  One block a row, 16 bytes a load, the row
// in registers between its two passes: at 4,096 rows of 2,048 from memory 8.6 us (2 bytes a load,
// the row read twice: 14.3), at 36 rows the latency of its loads.
template <int kSplits>
__global__ void __launch_bounds__(kRowThreads) norm_rows(GemmRows sums, const uint16_t* x, const uint16_t* scale, int d, float eps,
                                                         uint16_t* sum_out, uint16_t* out)
{
    constexpr int kMost = kMaxHidden / 8 / kRowThreads;  // 16-byte vectors of a row a thread holds
    __shared__ float partial[kRowThreads / 64];
    const size_t first = static_cast<size_t>(blockIdx.x) * d;
    float v[kMost][8];
    float squares = 0.0f;
#pragma unroll
    for (int i = 0; i < kMost; ++i) {
        const int n = (i * kRowThreads + threadIdx.x) * 8;
        if (n < d) {
            const u32x4 bits = *reinterpret_cast<const u32x4*>(x + first + n);
            float sum[8];
            if constexpr (kSplits > 1)
                load_rows8<kSplits>(sums, first + n, sum);
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                v[i][e] = kSplits > 1 ? Bf::round(sum[e] + Bf::elem(bits, e)) : Bf::elem(bits, e);
                squares = fmaf(v[i][e], v[i][e], squares);
            }
            if constexpr (kSplits > 1)
                *reinterpret_cast<u32x4*>(sum_out + first + n) = pack_bf16(v[i]);
        }
    }
    const float wave_sum = group_sum<64>(squares);
    if ((threadIdx.x & 63) == 63)
        partial[threadIdx.x / 64] = wave_sum;
    __syncthreads();
    float total = 0.0f;
#pragma unroll
    for (int w = 0; w < kRowThreads / 64; ++w)
        total += partial[w];
    const float inv = 1.0f / sqrtf(total / static_cast<float>(d) + eps);
#pragma unroll
    for (int i = 0; i < kMost; ++i) {
        const int n = (i * kRowThreads + threadIdx.x) * 8;
        if (n < d) {
            const u32x4 bits = *reinterpret_cast<const u32x4*>(scale + n);
#pragma unroll
            for (int e = 0; e < 8; ++e)
                v[i][e] = Bf::round(v[i][e] * inv) * Bf::elem(bits, e);
            *reinterpret_cast<u32x4*>(out + first + n) = pack_bf16(v[i]);
        }
    }
}

// Row r of the Q/K/V product ([q heads | k heads | v heads]; nq 0: [k heads | v heads]) at position
// `position + r`: the query and key heads rotated (split halves; cos and sin of position * frequency
// rounded to bf16, each product rounded, then the difference or sum), the query heads to q_rot, the
// key and value heads to the cache row of the position.  A block computes its position's cos and sin
// once and rotates 8 pairs a thread: 13.3 us for 4,096 rows of 40 heads (20.1 with cos and sin computed
// for every pair and 2 bytes a load).
template <int DH, int kSplits>
__global__ void __launch_bounds__(kRowThreads) rope_rows(GemmRows qkv, int position, const float* frequencies, int nq, int nkv,
                                                         uint16_t* q_rot, uint16_t* key_cache, uint16_t* value_cache)
{
    constexpr int kHalf = DH / 2, kVectors = kHalf / 8;
    __shared__ float cosine[kHalf], sine[kHalf];
    const int r = blockIdx.x, pos = position + r;
    const size_t first = static_cast<size_t>(r) * (nq + 2 * nkv) * DH;
    if (threadIdx.x < kHalf) {
        const float angle = static_cast<float>(pos) * frequencies[threadIdx.x];
        cosine[threadIdx.x] = Bf::round(cosf(angle));
        sine[threadIdx.x] = Bf::round(sinf(angle));
    }
    __syncthreads();
    const int rotated = (nq + nkv) * kVectors, all = rotated + nkv * DH / 8;
    for (int index = threadIdx.x; index < all; index += kRowThreads) {
        if (index >= rotated) {
            const int at = (index - rotated) * 8;
            float v[8];
            load_rows8<kSplits>(qkv, first + (nq + nkv) * DH + at, v);
            *reinterpret_cast<u32x4*>(value_cache + static_cast<size_t>(pos) * nkv * DH + at) = pack_bf16(v);
            continue;
        }
        const int head = index / kVectors, pair = (index - head * kVectors) * 8;
        float a[8], b[8], lo[8], hi[8];
        load_rows8<kSplits>(qkv, first + head * DH + pair, a);
        load_rows8<kSplits>(qkv, first + head * DH + pair + kHalf, b);
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const float c = cosine[pair + e], s = sine[pair + e];
            lo[e] = Bf::round(a[e] * c) - Bf::round(b[e] * s);
            hi[e] = Bf::round(b[e] * c) + Bf::round(a[e] * s);
        }
        uint16_t* dst = head < nq ? q_rot + (static_cast<size_t>(r) * nq + head) * DH
                                  : key_cache + (static_cast<size_t>(pos) * nkv + head - nq) * DH;
        *reinterpret_cast<u32x4*>(dst + pair) = pack_bf16(lo);
        *reinterpret_cast<u32x4*>(dst + pair + kHalf) = pack_bf16(hi);
    }
}

// Causal attention on the matrix cores, for 64 rows (positions position + r0 ..) and every
// query head of K/V head blockIdx.y: wave w takes rows r0 + 16 w .. + 15.  Scores are
// computed transposed, S^T = K Q^T with v_mfma_f32_16x16x32_bf16 (A: 16 key rows, B: the 16
// query rows of one head), so that lane l holds query l % 16 against keys 4 (l / 16) + i of each
// 16-key subtile.  Each score is bf16(bf16(dot) * scale) (the decode worker's score_of), keys past
// the query's position are masked (tiles past the block's first row only; rows past the chunk
// compute finite values nobody stores).  Pass 1 keeps each lane's running maximum and exp-sum per
// head, rescaled when the maximum grows, and merges the four lanes of a query at the end (exact
// maximum M, FP32 S).  Pass 2 recomputes the scores, rounds P = exp(s - M) / S to bf16 in
// registers and takes P V on the matrix cores with P as the A operand straight from the score
// layout: a 32-key step's k-elements 8 g .. 8 g + 7 of lane group g are keys 4 g .. 4 g + 3 and
// 16 + 4 g .. + 3 of the step (the sum over keys does not depend on their order), and two
// transposing LDS reads of the V rows supply the same keys.  The block stages each 64-key tile's
// K rows (and, in pass 2, V rows) in LDS once for its four waves, as stored, while the next
// tile's rows load into registers.
// The output is rounded once.  Keys past the block's last position are clamped to it when loaded
// and masked.
constexpr int kAttnThreads = 256;
constexpr int kAttnRows = 64;  // query positions per block: 16 per wave

// Two waves per SIMD for head_dim 64 (256 registers a lane at most; unbounded, the compiler
// took 276 and ran one); 128 needs more than 256 in either case.
template <int DH>
__global__ void __launch_bounds__(kAttnThreads) __attribute__((amdgpu_waves_per_eu(DH == 64 ? 2 : 1)))
attention_tiles(const uint16_t* q_rot, int position, int rows, int nq, int nkv,
                                                                const uint16_t* key_cache, const uint16_t* value_cache,
                                                                float scale, uint16_t* out)
{
    constexpr int KS = DH / 32;                              // 32-dim steps of a score
    constexpr int NT = DH / 16;                              // 16-dim output tiles
    constexpr int kVStride = DH + 8;                         // bf16 per staged V row
    constexpr int kKStride = DH + 8;                         // bf16 per staged K row
    constexpr int kVectors = DH / 8;                         // 16-byte vectors of a K or V row
    constexpr int kLoads = kTile * kVectors / kAttnThreads;  // vectors per thread per tile
    static_assert(kTile * kVectors % kAttnThreads == 0, "whole vectors per thread");
    __shared__ __attribute__((aligned(16))) uint16_t vs[kTile * kVStride];
    __shared__ __attribute__((aligned(16))) uint16_t ks[kTile * kKStride];
    // Causal blocks differ in work by their row block (block x reads x + 1 key tiles at position
    // 0).  Every block is resident at once, two per CU, and the dispatcher gives blocks L and L + H
    // (H = half the grid) the same CU; launched in row-block order those two were alike, and the
    // CUs holding two of the last row blocks set the kernel's time.  So block L takes the L-th
    // heaviest (row block, head) and block L + H the L-th lightest: the two add up to one
    // average pair.  Any assignment covers every (row block, head) once.
    const int row_blocks = gridDim.x, items = gridDim.x * gridDim.y, half = (items + 1) / 2;
    const int linear = blockIdx.x + gridDim.x * blockIdx.y;
    const int heaviest = linear < half ? linear : items - 1 - (linear - half);  // index in descending weight
    const int h = heaviest % nkv, group = nq / nkv;
    const int lane = threadIdx.x & 63, wave = threadIdx.x / 64;
    const int col = lane & 15, g4 = lane >> 4;
    const int r0 = (row_blocks - 1 - heaviest / nkv) * kAttnRows;
    const int last_row = min(r0 + kAttnRows, rows) - 1;
    const int last_key = position + last_row;  // the block's last key: every load stays at or below it
    const int tiles = last_key / kTile + 1;
    const int full_tiles = (position + r0 + 1) / kTile;  // tiles every row of the block sees whole
    const int qrow = r0 + 16 * wave + col;     // this lane's query row (B operand, output column)
    const int qpos = position + qrow;

    // B operands of the scores: query row qrow of each head, dims 32 k + 8 g4 .. + 7.
    u32x4 qb[kMaxGroup][KS];
#pragma unroll
    for (int g = 0; g < kMaxGroup; ++g)
#pragma unroll
        for (int k = 0; k < KS; ++k) {
            const bool live = g < group && qrow < rows;
            const size_t at = (static_cast<size_t>(live ? qrow : 0) * nq + h * group + (live ? g : 0)) * DH + 32 * k + 8 * g4;
            qb[g][k] = live ? *reinterpret_cast<const u32x4*>(q_rot + at) : u32x4{0u, 0u, 0u, 0u};
        }
    // This thread's vectors of tile kt's rows (K or V cache), keys clamped to the last key.
    auto load_rows = [&](const uint16_t* cache, int kt, u32x4 (&r)[kLoads]) {
#pragma unroll
        for (int i = 0; i < kLoads; ++i) {
            const int index = threadIdx.x + i * kAttnThreads, t = index / kVectors, v = index - t * kVectors;
            const int key = min(kt * kTile + t, last_key);
            r[i] = *reinterpret_cast<const u32x4*>(cache + (static_cast<size_t>(key) * nkv + h) * DH + 8 * v);
        }
    };
    auto stage_k = [&](const u32x4 (&r)[kLoads]) {
#pragma unroll
        for (int i = 0; i < kLoads; ++i) {
            const int index = threadIdx.x + i * kAttnThreads, t = index / kVectors, v = index - t * kVectors;
            *reinterpret_cast<u32x4*>(ks + t * kKStride + 8 * v) = r[i];
        }
    };
    auto stage_v = [&](const u32x4 (&r)[kLoads]) {
#pragma unroll
        for (int i = 0; i < kLoads; ++i) {
            const int index = threadIdx.x + i * kAttnThreads, t = index / kVectors, v = index - t * kVectors;
            *reinterpret_cast<u32x4*>(vs + t * kVStride + 8 * v) = r[i];
        }
    };
    // B operand of P V for dims 16 n .. + 15 over keys 4 g4 .. + 3 and 16 + 4 g4 .. + 3 of the
    // 32-key step: two transposing reads (ds_read_b64_tr_b16) of the V rows as stored.  Within a
    // 16-lane group lane j names key row 4 e + .. (e = j / 4) and dims 16 n + 4 (j % 4) .. + 3;
    // lane `col` receives dim 16 n + col of the four rows.
    auto v_operand = [&](int step, int n) {
        u32x4 out;
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            typedef short v4s __attribute__((ext_vector_type(4)));
            const int row = 32 * step + 16 * h + 4 * g4 + (col >> 2);
            const v4s v = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                (__attribute__((address_space(3))) v4s*)(vs + row * kVStride + 16 * n + 4 * (col & 3)));
            const uint2 pair = __builtin_bit_cast(uint2, v);
            out[2 * h] = pair.x;
            out[2 * h + 1] = pair.y;
        }
        return out;
    };
    // Scores of subtile j of the staged tile kt for every head: s[g][i] at key 64 kt + 16 j + 4 g4 + i.
    auto scores = [&](auto masked, int kt, int j, float (&s)[kMaxGroup][4]) {
        u32x4 ka[KS];
#pragma unroll
        for (int k = 0; k < KS; ++k)
            ka[k] = *reinterpret_cast<const u32x4*>(ks + (16 * j + col) * kKStride + 32 * k + 8 * g4);
#pragma unroll
        for (int g = 0; g < kMaxGroup; ++g) {
            f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int k = 0; k < KS; ++k)
                acc = mfma_16x16x32_bf16(ka[k], qb[g][k], acc);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                // With head_dim 64 the scale is 2^-3: the product of a bf16 value and it is a bf16
                // value already (short of the subnormal range), so the second rounding is the identity.
                const float score = DH == 64 ? Bf::round(acc[i]) * 0.125f : Bf::round(Bf::round(acc[i]) * scale);
                if constexpr (decltype(masked)::value)
                    s[g][i] = kt * kTile + 16 * j + 4 * g4 + i <= qpos ? score : -INFINITY;
                else
                    s[g][i] = score;
            }
        }
    };

    // Pass 1: this lane's running maximum and exp-sum per head, over its keys.
    float m[kMaxGroup], total[kMaxGroup];
#pragma unroll
    for (int g = 0; g < kMaxGroup; ++g) {
        m[g] = -INFINITY;
        total[g] = 0.0f;
    }
    u32x4 kr[kLoads], vr[kLoads];
    auto pass1_tile = [&](auto masked, int kt) {
        __syncthreads();  // the previous tile's K reads are done
        stage_k(kr);
        load_rows(key_cache, kt + 1, kr);  // the next tile (clamped past the last) in flight
        __syncthreads();
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            float s[kMaxGroup][4];
            scores(masked, kt, j, s);
#pragma unroll
            for (int g = 0; g < kMaxGroup; ++g) {
                const float grown = fmaxf(m[g], fmaxf(fmaxf(s[g][0], s[g][1]), fmaxf(s[g][2], s[g][3])));
                if constexpr (decltype(masked)::value)
                    if (grown == -INFINITY)
                        continue;  // every key so far masked
                // total exp(m - grown) + e_0 + ... + e_3, the first two terms as one FMA; the factor
                // (0 for the first subtile's m = -inf) is exactly 1 where the maximum held, and is
                // skipped when it held in every lane of the wave.
                const float first = exp_nonpositive(s[g][0] - grown);
                float sum;
                if (__builtin_amdgcn_ballot_w64(grown != m[g]) != 0)
                    sum = fmaf(total[g], exp_nonpositive(m[g] - grown), first);
                else
                    sum = total[g] + first;
#pragma unroll
                for (int i = 1; i < 4; ++i)
                    sum += exp_nonpositive(s[g][i] - grown);
                total[g] = sum;
                m[g] = grown;
            }
        }
    };
    load_rows(key_cache, 0, kr);
    int kt = 0;
    for (; kt < full_tiles; ++kt)
        pass1_tile(std::false_type{}, kt);
    for (; kt < tiles; ++kt)
        pass1_tile(std::true_type{}, kt);
    // The four lanes of a query (lane groups g4 = 0..3) merge: M exact, S rescaled to it.
#pragma unroll
    for (int g = 0; g < kMaxGroup; ++g)
#pragma unroll
        for (int offset = 16; offset < 64; offset <<= 1) {
            const float om = __shfl_xor(m[g], offset), ot = __shfl_xor(total[g], offset);
            const float grown = fmaxf(m[g], om);
            if (grown != -INFINITY) {
                total[g] = total[g] * exp_nonpositive(m[g] - grown) + ot * exp_nonpositive(om - grown);
                m[g] = grown;
            }
        }
    float inverse[kMaxGroup];  // 1 / S, correctly rounded
#pragma unroll
    for (int g = 0; g < kMaxGroup; ++g)
        inverse[g] = 1.0f / total[g];

    // Pass 2: P = bf16(exp(s - M) / S) as A operands, P V against the staged V rows.
    f32x4 o[kMaxGroup][NT];
#pragma unroll
    for (int g = 0; g < kMaxGroup; ++g)
#pragma unroll
        for (int n = 0; n < NT; ++n)
            o[g][n] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    auto pass2_tile = [&](auto masked, int kt) {
        __syncthreads();  // the previous tile's K and V reads are done
        stage_k(kr);
        stage_v(vr);
        load_rows(key_cache, kt + 1, kr);
        load_rows(value_cache, kt + 1, vr);
        __syncthreads();
#pragma unroll
        for (int step = 0; step < 2; ++step) {  // keys 32 step .. + 31 of the tile
            float s0[kMaxGroup][4], s1[kMaxGroup][4];
            scores(masked, kt, 2 * step, s0);
            scores(masked, kt, 2 * step + 1, s1);
            u32x4 vb[NT];
#pragma unroll
            for (int n = 0; n < NT; ++n)
                vb[n] = v_operand(step, n);
#pragma unroll
            for (int g = 0; g < kMaxGroup; ++g) {
                if (g >= group)
                    continue;
                float p[8];  // exp(s - M), masked keys exp(-inf) = 0; then P
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    p[i] = exp_nonpositive(s0[g][i] - m[g]);
                    p[4 + i] = exp_nonpositive(s1[g][i] - m[g]);
                }
                const float least = fminf(fminf(fminf(p[0], p[1]), fminf(p[2], p[3])), fminf(fminf(p[4], p[5]), fminf(p[6], p[7])));
                if (__builtin_expect(least >= kQuotientFloor, 1)) {
#pragma unroll
                    for (int i = 0; i < 8; ++i)
                        p[i] = divide_by(p[i], total[g], inverse[g]);
                } else {
#pragma unroll
                    for (int i = 0; i < 8; ++i)
                        p[i] = p[i] / total[g];
                }
                // Rounded to bf16 in pairs (v_cvt_pk_bf16_f32).
                auto pair = [](float lo, float hi) { return __builtin_bit_cast(uint32_t, bf16x2{static_cast<__bf16>(lo), static_cast<__bf16>(hi)}); };
                const u32x4 pa = {pair(p[0], p[1]), pair(p[2], p[3]), pair(p[4], p[5]), pair(p[6], p[7])};
#pragma unroll
                for (int n = 0; n < NT; ++n)
                    o[g][n] = mfma_16x16x32_bf16(pa, vb[n], o[g][n]);
            }
        }
    };
    load_rows(key_cache, 0, kr);
    load_rows(value_cache, 0, vr);
    for (kt = 0; kt < full_tiles; ++kt)
        pass2_tile(std::false_type{}, kt);
    for (; kt < tiles; ++kt)
        pass2_tile(std::true_type{}, kt);
    // o[g][n]: lane l holds query rows r0 + 16 wave + 4 g4 + i, dim 16 n + col.
#pragma unroll
    for (int g = 0; g < kMaxGroup; ++g)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int r = r0 + 16 * wave + 4 * g4 + i;
            if (g < group && r < rows)
#pragma unroll
                for (int n = 0; n < NT; ++n)
                    out[(static_cast<size_t>(r) * nq + h * group + g) * DH + 16 * n + col] = bits16(Bf::round(o[g][n][i]));
        }
}

// The tile shapes of the GEMM, and the time in us a 64-wide K step of one takes a CU that runs one
// block of it, and two at a time (measured at Llama-3.2-1B's widths, 36 to 4,096 rows).  The largest
// tile reads the least from L2 per product and wins where its blocks fill the chip; the smaller ones
// fill it with fewer rows and, at 64 rows, stream W at 3.9 TB/s where it is read once.
struct TileShape {
    int bm, bn;
    float alone, paired;  // paired 0: two do not fit a CU's LDS
};
constexpr TileShape kTileShapes[] = {{256, 256, 2.03f, 0.0f}, {128, 128, 0.85f, 1.1f}, {128, 64, 0.52f, 0.74f}, {64, 64, 0.29f, 0.46f}};
constexpr float kBlockStart = 2.4f;         // us a block takes besides its K steps
constexpr float kPartialRate = 3.1e6f;      // bytes per us that partial sums are written and read back at
constexpr int kCus = 256;
constexpr size_t kPartialFloats = 16u << 20;  // 64 MiB of partial sums

struct Tiling {
    int shape, splits;
};

// The tile shape and split of K with the least estimated time: blocks of a CU run one after another,
// or in pairs.  The estimate picks within 2% of the fastest measured choice on average over nine row
// counts from 36 to 4,096 and the four products of a Llama-3.2-1B layer (13% at worst).
Tiling choose_tiling(int m, int columns, int k, bool may_split)
{
    Tiling best{0, 1};
    float least = INFINITY;
    const int steps = k / 64;
    for (int shape = 0; shape < 4; ++shape) {
        const TileShape& t = kTileShapes[shape];
        const long tiles = static_cast<long>((m + t.bm - 1) / t.bm) * ((columns + t.bn - 1) / t.bn);
        for (int splits = 1; splits <= (may_split ? kMostSplits : 1); ++splits) {
            if (splits > 1 && (steps / splits < 4 || static_cast<size_t>(splits) * m * columns > kPartialFloats))
                break;
            const long per_cu = (tiles * splits + kCus - 1) / kCus;
            const int part = (steps + splits - 1) / splits;
            float time = t.paired > 0.0f ? (per_cu / 2) * (part * t.paired + kBlockStart) + (per_cu % 2) * (part * t.alone + kBlockStart)
                                         : per_cu * (part * t.alone + kBlockStart);
            if (splits > 1)
                time += static_cast<float>(splits) * m * columns * sizeof(float) / kPartialRate;
            if (time < least) {
                least = time;
                best = {shape, splits};
            }
        }
    }
    return best;
}

template <int BM, int BN, int WM, int WN, int KS, int STAGES, GemmOut OUT>
void launch_gemm(hipStream_t stream, GemmArgs g)
{
    const int columns = OUT == GemmOut::kSilu ? 2 * g.n : g.n;
    g.m_tiles = (g.m + BM - 1) / BM;
    g.n_tiles = (columns + BN - 1) / BN;
    hipLaunchKernelGGL((gemm_tiles<BM, BN, WM, WN, KS, STAGES, OUT>), dim3(g.m_tiles * g.n_tiles * g.splits),
                       dim3((BM / WM) * (BN / WN) * 64), 0, stream, g);
}

template <GemmOut OUT>
void launch_shape(hipStream_t stream, int shape, const GemmArgs& g)
{
    // kSilu groups four MFMA tiles of columns, so its waves take 64.
    constexpr bool kWide = OUT == GemmOut::kSilu;
    switch (shape) {
    case 0: return launch_gemm<256, 256, 128, 64, 64, 2, OUT>(stream, g);
    case 1: return launch_gemm<128, 128, kWide ? 32 : 64, kWide ? 64 : 32, 64, 2, OUT>(stream, g);
    case 2: return launch_gemm<128, 64, kWide ? 32 : 64, kWide ? 64 : 32, 64, 3, OUT>(stream, g);
    default: return launch_gemm<64, 64, kWide ? 16 : 32, kWide ? 64 : 32, 64, 4, OUT>(stream, g);
    }
}

} // namespace

bool MatrixPrefill::supports(const ti_worker_program_view& p)
{
    const ti_model_shape& s = p.shape;
    const int dh = s.head_dim;
    if (p.weight_dtype != TI_DTYPE_BFLOAT16 || !p.stack.full_stack || (dh != 64 && dh != 128) || s.kv_heads <= 0 ||
        s.query_heads % s.kv_heads != 0 || s.query_heads / s.kv_heads > kMaxGroup)
        return false;
    // Every GEMM of MatrixPrefill::layer, as (K, N): Q/K/V (d, heads x dh), Wo (query width, d),
    // gate/up (d, f), down (f, d).  The GEMM takes K a multiple of 32 and N a multiple of 16; the
    // head widths are multiples of 64 already.  A stack outside these prefills through the worker.
    auto gemm_shape = [](int k, int n) { return k >= 32 && k % 32 == 0 && n >= 16 && n % 16 == 0; };
    const int d = s.hidden_size, f = s.intermediate_size, qw = s.query_heads * dh, kvw = s.kv_heads * dh;
    return gemm_shape(d, qw) && gemm_shape(d, kvw) && gemm_shape(qw, d) && gemm_shape(d, f) && gemm_shape(f, d);
}

MatrixPrefill::MatrixPrefill(const ti_worker_program_view& program) : p_(program) {}

MatrixPrefill::~MatrixPrefill()
{
    if (buffer_)
        (void)hipFree(buffer_);
}

namespace {
struct Views {
    uint16_t *x, *u, *qkv, *q, *attention, *r, *product;
    float* partial;
};
size_t row_elements(const ti_model_shape& s)
{
    const size_t d = s.hidden_size, f = s.intermediate_size;
    const size_t qkv = static_cast<size_t>(s.query_heads + 2 * s.kv_heads) * s.head_dim;
    const size_t q = static_cast<size_t>(s.query_heads) * s.head_dim;
    return 3 * d + qkv + 2 * q + f;  // x, u, r | qkv | q, attention | product
}
Views views(void* buffer, const ti_model_shape& s, size_t rows)
{
    const size_t d = s.hidden_size, q = static_cast<size_t>(s.query_heads) * s.head_dim;
    Views v{};
    v.partial = static_cast<float*>(buffer);
    uint16_t* at = reinterpret_cast<uint16_t*>(v.partial + kPartialFloats);
    auto take = [&](size_t per_row) {
        uint16_t* start = at;
        at += rows * per_row;
        return start;
    };
    v.x = take(d);
    v.u = take(d);
    v.r = take(d);
    v.qkv = take(static_cast<size_t>(s.query_heads + 2 * s.kv_heads) * s.head_dim);
    v.q = take(q);
    v.attention = take(q);
    v.product = take(s.intermediate_size);
    return v;
}

// Enqueues X W^T of x [m][k] and w [n][k] into rows of c, or as partial sums; returns where the
// product is.  With a residual (row stride n), c receives bf16(bf16(sum) + residual) unless the
// sums are partial: the kernel that adds those adds the residual too.
GemmRows gemm(hipStream_t stream, const uint16_t* x, int m, int k, const uint16_t* w, int n, const uint16_t* residual, uint16_t* c,
              int ldc, float* partial)
{
    GemmArgs g{x, w, nullptr, residual, c, partial, m, n, k, ldc, 1, 0, 0};
    if (k % 64 != 0) {  // an FFN width of an odd number of 32s: K in steps of 32
        if (residual)
            launch_gemm<128, 128, 64, 32, 32, 3, GemmOut::kResidual>(stream, g);
        else
            launch_gemm<128, 128, 64, 32, 32, 3, GemmOut::kRows>(stream, g);
        return {c, nullptr, 1, 0};
    }
    const Tiling t = choose_tiling(m, n, k, partial != nullptr);
    g.splits = t.splits;
    if (t.splits > 1) {
        launch_shape<GemmOut::kPartial>(stream, t.shape, g);
        return {nullptr, partial, t.splits, static_cast<size_t>(m) * n};
    }
    if (residual)
        launch_shape<GemmOut::kResidual>(stream, t.shape, g);
    else
        launch_shape<GemmOut::kRows>(stream, t.shape, g);
    return {c, nullptr, 1, 0};
}
} // namespace

int MatrixPrefill::layer(hipStream_t stream, void* kv, int layer, int position, int rows)
{
    const ti_model_shape& s = p_.shape;
    const int d = s.hidden_size, f = s.intermediate_size, dh = s.head_dim, nq = s.query_heads, nkv = s.kv_heads;
    const int qw = nq * dh, kvw = nkv * dh;
    const Views v = views(buffer_, s, kChunkRows);
    const ti_layer_layout& w = p_.layout;
    auto weights = [&](int of) {
        return static_cast<const uint16_t*>(p_.weights) + p_.stack.layer_weights_offset +
               static_cast<size_t>(of) * p_.stack.layer_weight_stride;
    };
    const uint16_t* base = weights(layer);
    uint16_t* cache = static_cast<uint16_t*>(kv) + static_cast<size_t>(layer) * p_.stack.layer_kv_stride;
    const float eps = p_.numeric.rms_norm_eps;
    // out = RMSNorm(x), x first completed (into sum_out) by the residual when the GEMM left parts.
    auto norm = [&](const GemmRows& sums, const uint16_t* residual, uint16_t* sum_out, const uint16_t* scale) {
        with_splits(sums.splits, [&](auto n) {
            hipLaunchKernelGGL(norm_rows<n>, dim3(rows), dim3(kRowThreads), 0, stream, sums, n > 1 ? residual : sum_out, scale, d,
                               eps, sum_out, v.u);
        });
    };

    if (layer == 0)
        norm({v.x, nullptr, 1, 0}, nullptr, v.x, base + w.attn_norm);
    // The prompt's last position goes through the worker, and the positions here are read again only
    // as cache rows: the last layer ends with its K and V.
    const bool last = layer + 1 == p_.stack.layers;
    const int first_row = last ? qw : 0, width = (last ? 0 : qw) + 2 * kvw;
    GemmRows qkv{v.qkv, nullptr, 1, 0};
    // Wq, Wk and Wv are consecutive in the package's layer layout (plan.cpp checks the regions): one
    // GEMM over their rows.
    if (w.Wk == w.Wq + static_cast<uint32_t>(qw) * d && w.Wv == w.Wk + static_cast<uint32_t>(kvw) * d) {
        qkv = gemm(stream, v.u, rows, d, base + w.Wq + static_cast<size_t>(first_row) * d, width, nullptr, v.qkv, width, v.partial);
    } else {
        if (!last)
            gemm(stream, v.u, rows, d, base + w.Wq, qw, nullptr, v.qkv, width, nullptr);
        gemm(stream, v.u, rows, d, base + w.Wk, kvw, nullptr, v.qkv + width - 2 * kvw, width, nullptr);
        gemm(stream, v.u, rows, d, base + w.Wv, kvw, nullptr, v.qkv + width - kvw, width, nullptr);
    }
    const int rotated_queries = last ? 0 : nq;
    auto rope = [&](auto head_dim) {
        with_splits(qkv.splits, [&](auto n) {
            hipLaunchKernelGGL((rope_rows<head_dim, n>), dim3(rows), dim3(kRowThreads), 0, stream, qkv, position,
                               p_.rotary_frequencies, rotated_queries, nkv, v.q, cache + w.key, cache + w.value);
        });
    };
    if (dh == 64)
        rope(std::integral_constant<int, 64>{});
    else
        rope(std::integral_constant<int, 128>{});
    if (!last) {
        const float scale = 1.0f / sqrtf(static_cast<float>(dh));
        const dim3 attention_grid((rows + kAttnRows - 1) / kAttnRows, nkv);
        if (dh == 64)
            hipLaunchKernelGGL(attention_tiles<64>, attention_grid, dim3(kAttnThreads), 0, stream, v.q, position, rows, nq, nkv,
                               cache + w.key, cache + w.value, scale, v.attention);
        else
            hipLaunchKernelGGL(attention_tiles<128>, attention_grid, dim3(kAttnThreads), 0, stream, v.q, position, rows, nq, nkv,
                               cache + w.key, cache + w.value, scale, v.attention);
        const GemmRows projected = gemm(stream, v.attention, rows, qw, base + w.Wo, d, v.x, v.r, d, v.partial);
        norm(projected, v.x, v.r, base + w.ffn_norm);
        GemmArgs ffn{v.u, base + w.Wgate, base + w.Wup, nullptr, v.product, nullptr, rows, f, d, f, 1, 0, 0};
        launch_shape<GemmOut::kSilu>(stream, choose_tiling(rows, 2 * f, d, false).shape, ffn);
        // Wdown row-major [hidden][intermediate] on the device (ti_relayout_weights).
        const GemmRows down = gemm(stream, v.product, rows, f, base + w.Wdown, d, v.r, v.x, d, v.partial);
        norm(down, v.r, v.x, weights(layer + 1) + w.attn_norm);
    }
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess)
        return hip_fail(e, "prefill kernel launch");
    return TI_OK;
}

int MatrixPrefill::enqueue(hipStream_t stream, void* kv, const ti_token_id* tokens, int position, int count)
{
    if (!supports(p_))
        return fail(TI_ERR_INVALID_ARGUMENT, "matrix prefill needs a bf16 decoder stack with head_dim 64 or 128");
    if (count <= 0)
        return TI_OK;
    if (position < 0 || position + count > p_.shape.max_context)
        return fail(TI_ERR_INVALID_ARGUMENT, "sequence context capacity reached");
    if (!buffer_) {
        buffer_bytes_ = kPartialFloats * sizeof(float) + row_elements(p_.shape) * kChunkRows * sizeof(uint16_t);
        const hipError_t e = hipMalloc(&buffer_, buffer_bytes_);
        if (e != hipSuccess) {
            buffer_ = nullptr;
            return hip_fail(e, "prefill buffers");
        }
    }
    const Views v = views(buffer_, p_.shape, kChunkRows);
    const uint16_t* embedding = static_cast<const uint16_t*>(p_.weights) + p_.stack.embedding_offset;
    for (int first = 0; first < count; first += kChunkRows) {
        const int rows = std::min(kChunkRows, count - first);
        hipLaunchKernelGGL(gather_rows, dim3(rows), dim3(kRowThreads), 0, stream, embedding, tokens + first, p_.shape.hidden_size,
                           v.x);
        for (int layer = 0; layer < p_.stack.layers; ++layer) {
            const int code = this->layer(stream, kv, layer, position + first, rows);
            if (code != TI_OK)
                return code;
        }
    }
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess)
        return hip_fail(e, "prefill kernel launch");
    return TI_OK;
}

} // namespace tiles
