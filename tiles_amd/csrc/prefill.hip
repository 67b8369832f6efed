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
constexpr int kCus = 256;

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

// Causal attention on the matrix cores: 64-key tiles of one K/V head (blockIdx.y) against 16 HEADS query
// rows a block.  A wave takes 16 rows (positions position + r0 ..) and HEADS of the group's query heads;
// waves of a block share its K and V tiles.
//
// Scores are computed transposed, S^T = K Q^T with v_mfma_f32_16x16x32_bf16 (A: 16 key rows, B: the 16
// query rows of one head), so that lane l holds query l % 16 against keys 4 (l / 16) + i of each 16-key
// subtile.  Each score is bf16(bf16(dot) * scale) (the decode worker's score_of); keys past the query's
// position are masked (in tiles past the wave's first row only; rows past the chunk compute finite
// values nobody stores).  Pass 1 keeps each lane's running maximum M and sum S of 2^((s - M) log2 e) per
// head, rescaled when the maximum grows, and merges the four lanes of a query at the end.  Pass 2
// recomputes the scores, takes P = exp(s - M) / S as 2^((s - M) log2 e - log2 S), rounds it to bf16 once
// and multiplies: O^T = V^T P^T with P as the B operand straight from the score layout: a 32-key step's
// k-elements 8 g .. 8 g + 7 of lane group g are keys 4 g .. 4 g + 3 and 16 + 4 g .. + 3 of the step (the
// sum over keys does not depend on their order), and two transposing LDS reads of the V rows supply the
// same keys.  The output is rounded once.
//
// What bounds it is the arithmetic per score, once per pass: rounding to bf16 (a conversion for two, an
// unpacking each), the maximum, one FMA, v_exp_f32, in pass 2 the rounding of P: 7 instructions a score
// and pass.  The library's exponential and a division per score took 1.7 to 2.1 times as long: 4,096
// rows of 32 heads at position 0 421 us, now 205-217 (0.33 PFLOP/s), 28,672 rows in seven chunks 17.6 ms
// a layer, now 7.6; 210 rows, where one wave then took all four heads, 33 us, now 8.  The exponent's
// rounding moves P by at most a few 2^-23 of it, 2^-13 of the bf16 rounding that follows: layer 1's K
// and V rows of 130 to 4,000-token prompts are 0.00439-0.00450 and 0.00390-0.00394 off 64 bits either way.
//
// K rows (and, in pass 2, V rows) go from memory straight into one of two LDS buffers while the other's
// tile is used: chunk c (16 bytes) of row r at c ^ r mod 8, the rows of an operand read on distinct
// banks.  Keys past the block's last position are clamped to it when loaded and masked.
constexpr int kAttnThreads = 256;

template <int DH, int HEADS>
__global__ void __launch_bounds__(kAttnThreads) __attribute__((amdgpu_waves_per_eu(DH == 64 ? 2 : 1)))
attention_tiles(const uint16_t* q_rot, int position, int rows, int nq, int nkv, const uint16_t* key_cache,
                const uint16_t* value_cache, float scale, uint16_t* out)
{
    static_assert(kMaxGroup == 4, "four waves share a group of up to four heads");
    constexpr int kHeadWaves = kMaxGroup / HEADS;            // waves of a block with the same rows
    constexpr int kRows = 16 * (kAttnThreads / 64) / kHeadWaves;
    constexpr int KS = DH / 32;                              // 32-dim steps of a score
    constexpr int NT = DH / 16;                              // 16-dim output tiles
    constexpr int kVectors = DH / 8;                         // 16-byte chunks of a K or V row
    constexpr int kRowsPerLoad = 64 / kVectors;              // rows one load of a wave covers
    constexpr int kLoads = kTile / kRowsPerLoad / (kAttnThreads / 64);
    constexpr float kLog2e = 1.44269504f;
    __shared__ __attribute__((aligned(16))) uint16_t lds[2][2][kTile * DH];  // buffer, K or V
    // Causal blocks differ in work by their row block (block x reads x + 1 key tiles at position 0).
    // With at most two blocks a CU, all are resident at once and the dispatcher gives blocks L and
    // L + H (H = half the grid) the same CU: block L takes the L-th heaviest (row block, head) and
    // block L + H the L-th lightest, which add up to one average pair.  A larger grid starts with its
    // heaviest.  Any assignment covers every (row block, head) once.
    const int row_blocks = gridDim.x, items = gridDim.x * gridDim.y, half = (items + 1) / 2;
    const int linear = blockIdx.x + gridDim.x * blockIdx.y;
    const int heaviest = linear < half || items > 2 * kCus ? linear : items - 1 - (linear - half);  // index in descending weight
    const int h = heaviest % nkv, group = nq / nkv;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
    const int col = lane & 15, g4 = lane >> 4;
    const int r0 = (row_blocks - 1 - heaviest / nkv) * kRows;
    const int last_key = position + min(r0 + kRows, rows) - 1;  // the block's last key: every load stays at or below it
    const int tiles = last_key / kTile + 1;
    const int wave_row = r0 + 16 * (wave / kHeadWaves), head0 = (wave % kHeadWaves) * HEADS;
    const int full_tiles = (position + wave_row + 1) / kTile;             // tiles every row of the wave sees whole
    const int wave_tiles = min(tiles, (position + wave_row + 15) / kTile + 1);  // tiles any of them sees
    const int qrow = wave_row + col;  // this lane's query row (B operand, output column)
    const int qpos = position + qrow;

    // B operands of the scores: query row qrow of each head, dims 32 k + 8 g4 .. + 7.
    u32x4 qb[HEADS][KS];
#pragma unroll
    for (int g = 0; g < HEADS; ++g)
#pragma unroll
        for (int k = 0; k < KS; ++k) {
            const bool live = head0 + g < group && qrow < rows;
            const size_t at = (static_cast<size_t>(live ? qrow : 0) * nq + h * group + (live ? head0 + g : 0)) * DH + 32 * k + 8 * g4;
            qb[g][k] = live ? *reinterpret_cast<const u32x4*>(q_rot + at) : u32x4{0u, 0u, 0u, 0u};
        }
    // Step t < tiles is pass 1 on tile t, the others pass 2; this wave's part of a step's rows.
    auto issue = [&](int t) {
        const bool second = t >= tiles;
        const int kt = second ? t - tiles : t;
#pragma unroll
        for (int i = 0; i < kLoads; ++i) {
            const int row0 = (wave * kLoads + i) * kRowsPerLoad, row = row0 + lane / kVectors;
            const int chunk = (lane % kVectors) ^ (row & 7);
            const size_t from = (static_cast<size_t>(min(kt * kTile + row, last_key)) * nkv + h) * DH + 8 * chunk;
            load_to_lds(key_cache + from, &lds[t & 1][0][row0 * DH]);
            if (second)
                load_to_lds(value_cache + from, &lds[t & 1][1][row0 * DH]);
        }
    };
    // The step's tile is in LDS for every wave and the other buffer free: its next tile may load.
    auto begin_step = [&](int t) {
        asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
        if (t + 1 < 2 * tiles)
            issue(t + 1);
    };
    // Two values rounded by one v_cvt_pk_bf16_f32: the empty statement keeps the pair whole, which the
    // compiler splits where each half is used by itself, into two conversions and a shift each.
    auto round_pair = [](float lo, float hi) {
        uint32_t pair = pair_bf16(lo, hi);
        asm("" : "+v"(pair));
        return pair;
    };
    // Scores of keys 32 step .. + 31 of the staged tile kt for head g: s[4 j + i] at key
    // 64 kt + 32 step + 16 j + 4 g4 + i.
    auto key_operand = [&](const uint16_t* ks, int subtile, int k) {
        return *reinterpret_cast<const u32x4*>(ks + (16 * subtile + col) * DH + ((4 * k + g4) ^ (col & 7)) * 8);
    };
    auto scores = [&](auto masked, int kt, int step, const u32x4 (&ka)[2][KS], int g, float (&s)[8]) {
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int k = 0; k < KS; ++k)
                acc = mfma_16x16x32_bf16(ka[j][k], qb[g][k], acc);
#pragma unroll
            for (int i = 0; i < 4; i += 2) {
                // Rounded in pairs.  With head_dim 64 the scale is 2^-3: the product of a bf16 value
                // and it is a bf16 value already (short of the subnormal range), so the second
                // rounding is the identity and the product is left to the exponent's factor.
                uint32_t pair = round_pair(acc[i], acc[i + 1]);
                if constexpr (DH != 64)
                    pair = round_pair(__uint_as_float(pair << 16) * scale, __uint_as_float(pair & 0xffff0000u) * scale);
                s[4 * j + i] = __uint_as_float(pair << 16);
                s[4 * j + i + 1] = __uint_as_float(pair & 0xffff0000u);
            }
            if constexpr (decltype(masked)::value)
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    s[4 * j + i] = kt * kTile + 32 * step + 16 * j + 4 * g4 + i <= qpos ? s[4 * j + i] : -INFINITY;
        }
    };
    const float factor = DH == 64 ? 0.125f * kLog2e : kLog2e;  // exact: a power of two times log2 e

    // Pass 1, over this lane's keys: the largest score so far, it times the factor, and the sum of
    // 2^(s factor - reference).  A lane that has seen no key has -inf, -inf and 0.
    float m[HEADS], reference[HEADS], total[HEADS];
#pragma unroll
    for (int g = 0; g < HEADS; ++g) {
        m[g] = reference[g] = -INFINITY;
        total[g] = 0.0f;
    }
    auto pass1_tile = [&](auto masked, int kt, const uint16_t* ks) {
#pragma unroll
        for (int step = 0; step < 2; ++step) {
            u32x4 ka[2][KS];
#pragma unroll
            for (int j = 0; j < 2; ++j)
#pragma unroll
                for (int k = 0; k < KS; ++k)
                    ka[j][k] = key_operand(ks, 2 * step + j, k);
#pragma unroll
            for (int g = 0; g < HEADS; ++g) {
                float s[8];
                scores(masked, kt, step, ka, g, s);
                float grown = m[g];
#pragma unroll
                for (int i = 0; i < 8; i += 2)
                    grown = fmaxf(grown, fmaxf(s[i], s[i + 1]));
                // Rescaled where any lane's maximum grew (by 2^0 = 1 in the others).
                if (__builtin_amdgcn_ballot_w64(grown > m[g]) != 0) {
                    const float to = grown * factor;
                    total[g] = grown > m[g] ? total[g] * __builtin_amdgcn_exp2f(reference[g] - to) : total[g];
                    reference[g] = to;
                    m[g] = grown;
                }
                float sum = 0.0f;
#pragma unroll
                for (int i = 0; i < 8; ++i) {
                    const float e = __builtin_amdgcn_exp2f(fmaf(s[i], factor, -reference[g]));
                    sum += decltype(masked)::value ? (s[i] == -INFINITY ? 0.0f : e) : e;
                }
                total[g] += sum;
            }
        }
    };
    issue(0);
    for (int kt = 0; kt < tiles; ++kt) {
        begin_step(kt);
        if (kt < full_tiles)
            pass1_tile(std::false_type{}, kt, lds[kt & 1][0]);
        else if (kt < wave_tiles)
            pass1_tile(std::true_type{}, kt, lds[kt & 1][0]);
    }
    // The four lanes of a query (lane groups g4 = 0..3) merge, and P = 2^(s factor - shift).
    float shift[HEADS];
#pragma unroll
    for (int g = 0; g < HEADS; ++g) {
#pragma unroll
        for (int offset = 16; offset < 64; offset <<= 1) {
            const float other = __shfl_xor(reference[g], offset), sum = __shfl_xor(total[g], offset);
            const float to = fmaxf(reference[g], other);
            if (to != -INFINITY) {
                total[g] = total[g] * __builtin_amdgcn_exp2f(reference[g] - to) + sum * __builtin_amdgcn_exp2f(other - to);
                reference[g] = to;
            }
        }
        shift[g] = reference[g] + __builtin_amdgcn_logf(total[g]);
    }

    // Pass 2: o[g][n] += V^T P^T for dims 16 n .. + 15.
    f32x4 o[HEADS][NT];
#pragma unroll
    for (int g = 0; g < HEADS; ++g)
#pragma unroll
        for (int n = 0; n < NT; ++n)
            o[g][n] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    // A operand of P V for dims 16 n .. + 15 over keys 4 g4 .. + 3 and 16 + 4 g4 .. + 3 of the 32-key
    // step: two transposing reads (ds_read_b64_tr_b16) of the V rows as stored.  Within a 16-lane
    // group lane j names key row 4 e + .. (e = j / 4) and dims 16 n + 4 (j % 4) .. + 3; lane `col`
    // receives dim 16 n + col of the four rows.
    auto v_operand = [&](const uint16_t* vs, int step, int n) {
        u32x4 r;
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            typedef short v4s __attribute__((ext_vector_type(4)));
            const int row = 32 * step + 16 * j + 4 * g4 + (col >> 2);
            const int chunk = (2 * n + ((col & 3) >> 1)) ^ (row & 7);
            const v4s v = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                (__attribute__((address_space(3))) v4s*)(vs + row * DH + 8 * chunk + 4 * (col & 1)));
            const uint2 pair = __builtin_bit_cast(uint2, v);
            r[2 * j] = pair.x;
            r[2 * j + 1] = pair.y;
        }
        return r;
    };
    auto pass2_tile = [&](auto masked, int kt, const uint16_t* ks, const uint16_t* vs) {
#pragma unroll
        for (int step = 0; step < 2; ++step) {  // keys 32 step .. + 31 of the tile
            u32x4 ka[2][KS], va[NT];
#pragma unroll
            for (int j = 0; j < 2; ++j)
#pragma unroll
                for (int k = 0; k < KS; ++k)
                    ka[j][k] = key_operand(ks, 2 * step + j, k);
#pragma unroll
            for (int n = 0; n < NT; ++n)
                va[n] = v_operand(vs, step, n);
#pragma unroll
            for (int g = 0; g < HEADS; ++g) {
                float s[8];
                scores(masked, kt, step, ka, g, s);
#pragma unroll
                for (int i = 0; i < 8; ++i)
                    s[i] = __builtin_amdgcn_exp2f(fmaf(s[i], factor, -shift[g]));
                const u32x4 p = pack_bf16(s);
#pragma unroll
                for (int n = 0; n < NT; ++n)
                    o[g][n] = mfma_16x16x32_bf16(va[n], p, o[g][n]);
            }
        }
    };
    for (int kt = 0; kt < tiles; ++kt) {
        const int t = tiles + kt;
        begin_step(t);
        if (kt < full_tiles)
            pass2_tile(std::false_type{}, kt, lds[t & 1][0], lds[t & 1][1]);
        else if (kt < wave_tiles)
            pass2_tile(std::true_type{}, kt, lds[t & 1][0], lds[t & 1][1]);
    }
    // o[g][n]: lane l holds query row qrow, dims 16 n + 4 g4 .. + 3.
    if (qrow < rows)
#pragma unroll
        for (int g = 0; g < HEADS; ++g)
            if (head0 + g < group)
#pragma unroll
                for (int n = 0; n < NT; ++n)
                    *reinterpret_cast<uint2*>(out + (static_cast<size_t>(qrow) * nq + h * group + head0 + g) * DH + 16 * n + 4 * g4) =
                        uint2{pair_bf16(o[g][n][0], o[g][n][1]), pair_bf16(o[g][n][2], o[g][n][3])};
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
constexpr size_t kPartialFloats = 16u << 20;  // 64 MiB of partial sums at most

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
    for (const Buffer& b : {short_, long_})
        if (b.data)
            (void)hipFree(b.data);
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
// The partial sums of any product of `rows` rows that choose_tiling splits.
size_t partial_elements(const ti_model_shape& s, size_t rows)
{
    const size_t widest = std::max<size_t>(s.hidden_size, static_cast<size_t>(s.query_heads + 2 * s.kv_heads) * s.head_dim);
    return std::min(kPartialFloats, kMostSplits * rows * widest);
}
Views views(void* buffer, const ti_model_shape& s, size_t rows)
{
    const size_t d = s.hidden_size, q = static_cast<size_t>(s.query_heads) * s.head_dim;
    Views v{};
    v.partial = static_cast<float*>(buffer);
    uint16_t* at = reinterpret_cast<uint16_t*>(v.partial + partial_elements(s, rows));
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

// Attention of `rows` query rows: the most heads a wave (K and V operands read once for all of them)
// that leave two blocks a CU; fewer, and more blocks of fewer rows, for shorter prompts.
template <int DH, int HEADS = kMaxGroup>
void attend_heads(hipStream_t stream, const uint16_t* q, int position, int rows, int nq, int nkv, const uint16_t* k, const uint16_t* v,
                  float scale, uint16_t* out)
{
    const int blocks = (rows + 16 * HEADS - 1) / (16 * HEADS);
    if constexpr (HEADS > 1)
        if (blocks * nkv < 2 * kCus)
            return attend_heads<DH, HEADS / 2>(stream, q, position, rows, nq, nkv, k, v, scale, out);
    hipLaunchKernelGGL((attention_tiles<DH, HEADS>), dim3(blocks, nkv), dim3(kAttnThreads), 0, stream, q, position, rows, nq, nkv, k,
                       v, scale, out);
}
void attend(hipStream_t stream, const uint16_t* q, int position, int rows, int nq, int nkv, int dh, const uint16_t* k,
            const uint16_t* v, float scale, uint16_t* out)
{
    if (dh == 64)
        attend_heads<64>(stream, q, position, rows, nq, nkv, k, v, scale, out);
    else
        attend_heads<128>(stream, q, position, rows, nq, nkv, k, v, scale, out);
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

namespace {
// out = RMSNorm(x), x first completed (into x, from `residual`) when the GEMM left parts.
void norm(hipStream_t stream, const GemmRows& sums, const uint16_t* residual, uint16_t* x, const uint16_t* scale, int rows, int d,
          float eps, uint16_t* out)
{
    with_splits(sums.splits, [&](auto n) {
        hipLaunchKernelGGL(norm_rows<n>, dim3(rows), dim3(kRowThreads), 0, stream, sums, n > 1 ? residual : x, scale, d, eps, x, out);
    });
}
void rope(hipStream_t stream, const GemmRows& qkv, int rows, int position, const float* frequencies, int nq, int nkv, int dh,
          uint16_t* q_rot, uint16_t* key_cache, uint16_t* value_cache)
{
    auto launch = [&](auto head_dim) {
        with_splits(qkv.splits, [&](auto n) {
            hipLaunchKernelGGL((rope_rows<head_dim, n>), dim3(rows), dim3(kRowThreads), 0, stream, qkv, position, frequencies, nq,
                               nkv, q_rot, key_cache, value_cache);
        });
    };
    if (dh == 64)
        launch(std::integral_constant<int, 64>{});
    else
        launch(std::integral_constant<int, 128>{});
}
} // namespace

const uint16_t* MatrixPrefill::weights(int layer) const
{
    return static_cast<const uint16_t*>(p_.weights) + p_.stack.layer_weights_offset +
           static_cast<size_t>(layer) * p_.stack.layer_weight_stride;
}

// From the attention output of `rows` rows (their layer input in x from row `first_row`) to the layer's
// output, in the same rows of x, and its RMSNorm with `next_norm` in u.
void MatrixPrefill::feed_forward(hipStream_t stream, int layer, int rows, int first_row, const uint16_t* next_norm)
{
    const ti_model_shape& s = p_.shape;
    const int d = s.hidden_size, f = s.intermediate_size, qw = s.query_heads * s.head_dim;
    const ti_layer_layout& w = p_.layout;
    const uint16_t* base = weights(layer);
    const Views v = views(buffer_.data, s, buffer_.rows);
    uint16_t* x = v.x + static_cast<size_t>(first_row) * d;
    const float eps = p_.numeric.rms_norm_eps;
    const GemmRows projected = gemm(stream, v.attention, rows, qw, base + w.Wo, d, x, v.r, d, v.partial);
    norm(stream, projected, x, v.r, base + w.ffn_norm, rows, d, eps, v.u);
    GemmArgs ffn{v.u, base + w.Wgate, base + w.Wup, nullptr, v.product, nullptr, rows, f, d, f, 1, 0, 0};
    launch_shape<GemmOut::kSilu>(stream, choose_tiling(rows, 2 * f, d, false).shape, ffn);
    // Wdown row-major [hidden][intermediate] on the device (ti_relayout_weights).
    const GemmRows down = gemm(stream, v.product, rows, f, base + w.Wdown, d, v.r, x, d, v.partial);
    norm(stream, down, v.r, x, next_norm, rows, d, eps, v.u);
}

int MatrixPrefill::layer(hipStream_t stream, void* kv, int layer, int position, int rows)
{
    const ti_model_shape& s = p_.shape;
    const int d = s.hidden_size, dh = s.head_dim, nq = s.query_heads, nkv = s.kv_heads;
    const int qw = nq * dh, kvw = nkv * dh;
    const Views v = views(buffer_.data, s, buffer_.rows);
    const ti_layer_layout& w = p_.layout;
    const uint16_t* base = weights(layer);
    uint16_t* cache = static_cast<uint16_t*>(kv) + static_cast<size_t>(layer) * p_.stack.layer_kv_stride;

    if (layer == 0)
        norm(stream, {v.x, nullptr, 1, 0}, nullptr, v.x, base + w.attn_norm, rows, d, p_.numeric.rms_norm_eps, v.u);
    // Of the last layer's positions only the cache rows are read again (and, where last_row follows,
    // the last one's output): it ends with its K and V.
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
    rope(stream, qkv, rows, position, p_.rotary_frequencies, last ? 0 : nq, nkv, dh, v.q, cache + w.key, cache + w.value);
    if (!last) {
        attend(stream, v.q, position, rows, nq, nkv, dh, cache + w.key, cache + w.value, 1.0f / sqrtf(static_cast<float>(dh)),
               v.attention);
        feed_forward(stream, layer, rows, 0, weights(layer + 1) + w.attn_norm);
    }
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess)
        return hip_fail(e, "prefill kernel launch");
    return TI_OK;
}

int MatrixPrefill::last_row(hipStream_t stream, void* kv, int position, const void** hidden)
{
    if (!buffer_.data || rows_ < 1 || position < rows_ - 1)
        return fail(TI_ERR_INVALID_ARGUMENT, "no prefilled position to finish");
    const ti_model_shape& s = p_.shape;
    const int d = s.hidden_size, dh = s.head_dim, nq = s.query_heads, nkv = s.kv_heads, layer = p_.stack.layers - 1;
    const Views v = views(buffer_.data, s, buffer_.rows);
    const ti_layer_layout& w = p_.layout;
    const uint16_t* cache = static_cast<const uint16_t*>(kv) + static_cast<size_t>(layer) * p_.stack.layer_kv_stride;
    const size_t row = rows_ - 1;
    const GemmRows q = gemm(stream, v.u + row * d, 1, d, weights(layer) + w.Wq, nq * dh, nullptr, v.qkv, nq * dh, v.partial);
    rope(stream, q, 1, position, p_.rotary_frequencies, nq, 0, dh, v.q, nullptr, nullptr);
    attend(stream, v.q, position, 1, nq, nkv, dh, cache + w.key, cache + w.value, 1.0f / sqrtf(static_cast<float>(dh)), v.attention);
    const uint16_t* final_norm = static_cast<const uint16_t*>(p_.weights) + p_.stack.final_norm_offset;
    feed_forward(stream, layer, 1, static_cast<int>(row), final_norm);  // the norm's output is not used
    *hidden = v.x + row * d;
    const hipError_t e = hipGetLastError();
    return e == hipSuccess ? TI_OK : hip_fail(e, "prefill kernel launch");
}

int MatrixPrefill::reserve(int count)
{
    if (long_.data || (short_.data && count <= kShortRows)) {
        buffer_ = long_.data ? long_ : short_;
        return TI_OK;
    }
    Buffer& b = count <= kShortRows ? short_ : long_;
    const int rows = count <= kShortRows ? kShortRows : kChunkRows;
    const size_t bytes = partial_elements(p_.shape, rows) * sizeof(float) + row_elements(p_.shape) * rows * sizeof(uint16_t);
    const hipError_t e = hipMalloc(&b.data, bytes);
    if (e != hipSuccess) {
        b.data = nullptr;
        (void)hipGetLastError();  // the caller may go on without: the next launch's check is not to see it
        return hip_fail(e, "prefill buffers");
    }
    b.rows = rows;
    buffer_ = b;
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
    const int code = reserve(count);
    if (code != TI_OK)
        return code;
    const Views v = views(buffer_.data, p_.shape, buffer_.rows);
    const uint16_t* embedding = static_cast<const uint16_t*>(p_.weights) + p_.stack.embedding_offset;
    for (int first = 0; first < count; first += kChunkRows) {
        const int rows = rows_ = std::min(kChunkRows, count - first);
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
