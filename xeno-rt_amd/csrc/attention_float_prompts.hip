// Causal attention of a step of many tokens in float32 on the matrix cores (v_mfma_f32_16x16x4_f32), heads of 64 and 128 dims,
// to the bits of the general kernel (attention_generic.hip), which takes the steps of few tokens: the instruction adds its four
// products to the sum one after the other, fmaf by fmaf, so two of them from zero make the sum over a piece of 8 dims, and
// 16 of them the sum over a block's 64 values, in the general kernel's order; blocks, chunks of eight blocks and their
// merges are the same, and the probabilities of a block are added up in the order of its sum over a wavefront.
//
// The general kernel is bound by the vector ALUs: one lane a key, 64 fmafs a key and head, every key read for four heads only.
// Here a block of 64 keys of 64 dims takes a workgroup 5 us, of which the matrix cores need 2 (one wavefront a SIMD, whose
// products, softmax and waits come one after the other), and the latest tokens' blocks set the time: 777 tokens, 32 heads of 64 on 8
// 412 -> 94 us, 100 tokens 30 -> 15, 1500 tokens 1299 -> 231; 32 heads of 128 on 8, 777 tokens 763 -> 189; 14 heads of 64 on 2, 150 tokens
// 20 -> 20. Tiles of 32 tokens (v_mfma_f32_32x32x2_f32) took 107, 22 and 279 us.
//
// A wavefront takes 16 tokens of one head, a workgroup four such tiles of one key/value head: where groups are multiples of four heads
// they are heads of the same tokens. The workgroup's tokens may be of several sequences: they are taken run by run. Scores:
// S[key][token] with keys as rows; a lane (token = lane % 16) then holds of every 16 keys four neighbouring ones, and an
// exchange among the quarters of the wavefront (v_permlane32_swap, v_permlane16_swap) makes them the operand of the product with the
// values, O[dim][token]. Keys and values of the next block are on their way into registers while this block is worked on; in LDS, in
// two stages, the elements that a quarter of a wavefront takes of 16 lie together, so that a lane reads four steps at once.
#include <algorithm>

#include "cache_layout.h"
#include "xrt_hip.h"

namespace {

typedef float sums4 __attribute__((ext_vector_type(4)));

constexpr int TILE = 16;                    // tokens of a wavefront
constexpr int WAVES = 4;
constexpr int SPAN = WAVES * TILE;          // tokens of a workgroup at most
constexpr int CHUNK_BLOCKS = 8;             // as in the general kernel
constexpr int THREADS = WAVES * XRT_WAVE;
constexpr float LARGEST = 3.402823466e38f;  // of the finite ones

// The upper 32 lanes of `low` change places with the lower 32 lanes of `high`.
__device__ __forceinline__ void swap_halves(float& low, float& high) {
    const auto both = __builtin_amdgcn_permlane32_swap(__builtin_bit_cast(unsigned, low), __builtin_bit_cast(unsigned, high), false, false);
    const unsigned first = both[0], second = both[1];       // (a vector's element itself is not what a bit cast takes)
    low = __builtin_bit_cast(float, first);
    high = __builtin_bit_cast(float, second);
}
// The odd rows of 16 lanes of `low` change places with the even rows of `high`.
__device__ __forceinline__ void swap_quarters(float& low, float& high) {
    const auto both = __builtin_amdgcn_permlane16_swap(__builtin_bit_cast(unsigned, low), __builtin_bit_cast(unsigned, high), false, false);
    const unsigned first = both[0], second = both[1];
    low = __builtin_bit_cast(float, first);
    high = __builtin_bit_cast(float, second);
}

template <int HD>
__global__ void __launch_bounds__(THREADS, 1) attention_float_prompts_kernel(
    const float* __restrict__ q_rows, int row_width, int tokens, int n_heads, int n_kv_heads,
    const float* __restrict__ k_cache, const float* __restrict__ v_cache, const int* __restrict__ block_table, int table_stride,
    int n_blocks, const int* __restrict__ positions, const int* __restrict__ slots, float* __restrict__ out, float scale) {
#pragma clang fp contract(off)              // (what is one rounding here is written as fmaf, as in the general kernel)
    constexpr int PIECES = HD / 8;          // of a key
    constexpr int DT = HD / 16;             // tiles of 16 dims
    constexpr int BLOCK = XRT_BLOCK_TOKENS * HD;
    constexpr int MINE = BLOCK / 8 / THREADS;                                // pieces of 8 that a thread moves, of keys and of values
    extern __shared__ __attribute__((aligned(16))) float lds[];              // [2 stages][keys | values][BLOCK]
    __shared__ int slot_of[SPAN], position_of[SPAN];
    __shared__ unsigned long long strange[3];                                // tokens of block b (b % 3) that have a value that is infinite or NaN

    const int tid = threadIdx.x, lane = tid % XRT_WAVE, wave = __builtin_amdgcn_readfirstlane(tid / XRT_WAVE);
    const int column = lane % 16, quarter = lane / 16;
    const int group = n_heads / n_kv_heads;
    const int kv_head = blockIdx.y;
    // the latest tiles, which have the most keys, come first; a tile's heads lie side by side
    const long tiles = (tokens + TILE - 1) / TILE, first_pair = ((long)gridDim.x - 1 - blockIdx.x) * WAVES;
    const long pair = first_pair + wave;
    const bool works = pair < tiles * group;
    const int span_begin = (int)(first_pair / group) * TILE;
    const int token = (int)(min(pair, tiles * group - 1) / group) * TILE + column;
    const int head = kv_head * group + (int)(min(pair, tiles * group - 1) % group);
    const int place = token - span_begin;                                    // below SPAN: four pairs name four tiles at most

    for (int i = tid; i < SPAN; i += THREADS) {
        const bool there = span_begin + i < tokens;
        slot_of[i] = there ? slots[span_begin + i] : -2;
        position_of[i] = there ? positions[span_begin + i] : -1;
    }
    __syncthreads();
    const int pos = works ? position_of[place] : -1;
    const int span_end = min((int)((min(first_pair + WAVES, tiles * group) - 1) / group) * TILE + TILE, tokens) - span_begin;

    // the query: of every 8 dims the two that this quarter of the wavefront takes
    float q[PIECES][2];
    {
        const float* row = q_rows + (long)min(token, tokens - 1) * row_width + (long)head * HD + quarter;
#pragma unroll
        for (int p = 0; p < PIECES; ++p) {
            q[p][0] = row[p * 8];
            q[p][1] = row[p * 8 + 4];
        }
    }

    // runs of neighbouring tokens of one sequence
    for (int begin = 0; begin < span_end;) {
        const int slot = __builtin_amdgcn_readfirstlane(slot_of[begin]);
        int end = span_end;
#pragma unroll
        for (int part = SPAN / XRT_WAVE - 1; part >= 0; --part) {
            const int i = part * XRT_WAVE + lane;
            const unsigned long long others = __ballot(i > begin && slot_of[i] != slot);
            if (others != 0) end = min(end, part * XRT_WAVE + (int)__ffsll(others) - 1);
        }
        const bool in_run = works && place >= begin && place < end;
        float* dst = out + ((long)min(token, tokens - 1) * n_heads + head) * HD;
        if (slot < 0) {                                                      // padding
            if (in_run)
                for (int d = quarter * 4; d < HD; d += 16) *reinterpret_cast<float4*>(dst + d) = make_float4(0.f, 0.f, 0.f, 0.f);
            begin = end;
            continue;
        }
        int latest = -1;                                                     // of the workgroup's tokens in the run
#pragma unroll
        for (int part = 0; part < SPAN / XRT_WAVE; ++part) {
            const int i = part * XRT_WAVE + lane;
            if (i >= begin && i < end) latest = max(latest, position_of[i]);
        }
        int wave_latest = in_run ? pos : -1;                                 // of this wavefront's
#pragma unroll
        for (int offset = XRT_WAVE / 2; offset > 0; offset >>= 1) {
            latest = max(latest, __shfl_xor(latest, offset, XRT_WAVE));
            wave_latest = max(wave_latest, __shfl_xor(wave_latest, offset, XRT_WAVE));
        }
        latest = __builtin_amdgcn_readfirstlane(latest);
        wave_latest = __builtin_amdgcn_readfirstlane(wave_latest);
        const int last_block = latest / XRT_BLOCK_TOKENS;                    // (a run has a token, and its position is not negative)
        const int* table = block_table + (long)slot * table_stride;
        auto block_of = [&](int b) { return table[min(b, last_block)]; };

        float4 moving[2][MINE][2];                                           // [keys | values][piece][its halves]
        auto fetch = [&](int b) {
            const int block = min(max(block_of(b), 0), n_blocks - 1);
            const long base = ((long)block * n_kv_heads + kv_head) * BLOCK;
#pragma unroll
            for (int i = 0; i < MINE; ++i)
#pragma unroll
                for (int e = 0; e < 2; ++e) {
                    moving[0][i][e] = *reinterpret_cast<const float4*>(k_cache + base + (long)(i * THREADS + tid) * 8 + e * 4);
                    moving[1][i][e] = *reinterpret_cast<const float4*>(v_cache + base + (long)(i * THREADS + tid) * 8 + e * 4);
                }
        };
        // LDS: keys [two pieces of dims][quarter][key], values [two pieces of tokens][quarter][dim], 16 bytes each: the elements
        // quarter and quarter + 4 of either piece
        auto stash = [&](int stage, int b) {
            float* keys = lds + stage * 2 * BLOCK;
            float* values = keys + BLOCK;
#pragma unroll
            for (int i = 0; i < MINE; ++i) {
                const int piece = i * THREADS + tid, tile = piece / 64, r = piece % 16, c = piece % 64 / 16;
                {
                    const int key = tile / (HD / 32) / 2 * 32 + r / 4 * 8 + tile / (HD / 32) % 2 * 4 + r % 4, of_dims = tile % (HD / 32) * 4 + c;
                    const float4 a = moving[0][i][0], z = moving[0][i][1];
                    float* to = keys + (of_dims / 2 * 4 * XRT_BLOCK_TOKENS + key) * 4 + of_dims % 2 * 2;
                    *reinterpret_cast<float2*>(to) = make_float2(a.x, z.x);
                    *reinterpret_cast<float2*>(to + XRT_BLOCK_TOKENS * 4) = make_float2(a.y, z.y);
                    *reinterpret_cast<float2*>(to + XRT_BLOCK_TOKENS * 8) = make_float2(a.z, z.z);
                    *reinterpret_cast<float2*>(to + XRT_BLOCK_TOKENS * 12) = make_float2(a.w, z.w);
                }
                {
                    const int dim = tile % DT * 16 + r, of_tokens = tile / DT * 4 + c;
                    float v[8] = {moving[1][i][0].x, moving[1][i][0].y, moving[1][i][0].z, moving[1][i][0].w,
                                  moving[1][i][1].x, moving[1][i][1].y, moving[1][i][1].z, moving[1][i][1].w};
                    // what lies beyond the latest token is nobody's; a block with an infinity or a NaN is marked
                    unsigned mask = 0;
#pragma unroll
                    for (int e = 0; e < 8; ++e) {
                        if (b * XRT_BLOCK_TOKENS + of_tokens * 8 + e > latest) v[e] = 0.f;
                        else if (!(fabsf(v[e]) <= LARGEST)) mask |= 1u << e;
                    }
                    if (mask != 0) atomicOr(&strange[b % 3], (unsigned long long)mask << (of_tokens * 8));
                    float* to = values + (of_tokens / 2 * 4 * HD + dim) * 4 + of_tokens % 2 * 2;
#pragma unroll
                    for (int e = 0; e < 4; ++e) *reinterpret_cast<float2*>(to + e * HD * 4) = make_float2(v[e], v[e + 4]);
                }
            }
        };

        float m = -INFINITY, l = 0.f, all_m = -INFINITY, all_l = 0.f;
        sums4 o[DT], all_o[DT];
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) o[dt] = all_o[dt] = sums4{};

        __syncthreads();                                                     // the stages of the run before have been read
        if (tid < 3) strange[tid] = 0;
        fetch(0);
        __syncthreads();
        stash(0, 0);
        for (int b = 0; b <= last_block; ++b) {
            const int stage = b & 1;
            __syncthreads();                                                 // this stage is written, the other one has been read
            if (tid == 0) strange[(b + 2) % 3] = 0;                          // (read before the barrier, written next behind the following one)
            fetch(b + 1);                                                    // (beyond the last block: the last one again, which nobody reads)
            const int block = block_of(b);
            if (b * XRT_BLOCK_TOKENS <= wave_latest && block >= 0 && block < n_blocks) {       // (the host never hands out another block)
                const float* keys = lds + stage * 2 * BLOCK;
                const float* values = keys + BLOCK;
                const bool sees = in_run && b * XRT_BLOCK_TOKENS <= pos;     // of the block's keys this lane's token sees one at least
                const int valid = pos - b * XRT_BLOCK_TOKENS;                // the last of them (or beyond the block)
                // a piece's sums are added up while the matrix cores work on the next piece's (the fences keep the compiler from
                // starting all pieces at once, whose sums find no registers)
                sums4 s[4] = {sums4{}, sums4{}, sums4{}, sums4{}}, of_piece[2][4];
                float4 k_ahead[2][4], v_ahead[2][DT];
                auto read_keys = [&](int pair_of) {
#pragma unroll
                    for (int t = 0; t < 4; ++t)
                        k_ahead[pair_of % 2][t] = *reinterpret_cast<const float4*>(keys + ((pair_of * 4 + quarter) * XRT_BLOCK_TOKENS + t * 16 + column) * 4);
                };
                auto read_values = [&](int t) {
#pragma unroll
                    for (int dt = 0; dt < DT; ++dt)
                        v_ahead[t % 2][dt] = *reinterpret_cast<const float4*>(values + ((t * 4 + quarter) * HD + dt * 16 + column) * 4);
                };
                read_keys(0);
#pragma unroll
                for (int pair_of = 0; pair_of < PIECES / 2; ++pair_of) {
                    if (pair_of + 1 < PIECES / 2) read_keys(pair_of + 1);
                    else read_values(0);
                    const float4 (&k)[4] = k_ahead[pair_of % 2];
#pragma unroll
                    for (int p = 0; p < 2; ++p) {
#pragma unroll
                        for (int t = 0; t < 4; ++t)
                            of_piece[p][t] = __builtin_amdgcn_mfma_f32_16x16x4f32(p ? k[t].z : k[t].x, q[pair_of * 2 + p][0], sums4{}, 0, 0, 0);
#pragma unroll
                        for (int t = 0; t < 4; ++t)
                            of_piece[p][t] = __builtin_amdgcn_mfma_f32_16x16x4f32(p ? k[t].w : k[t].y, q[pair_of * 2 + p][1], of_piece[p][t], 0, 0, 0);
                        if (pair_of + p > 0)
#pragma unroll
                            for (int t = 0; t < 4; ++t)
#pragma unroll
                                for (int e = 0; e < 4; ++e) s[t][e] += of_piece[p ^ 1][t][e];
                    }
                    __builtin_amdgcn_sched_barrier(0);
                }
#pragma unroll
                for (int t = 0; t < 4; ++t)
#pragma unroll
                    for (int e = 0; e < 4; ++e) s[t][e] += of_piece[1][t][e];
                // element e of s[t] is key t * 16 + quarter * 4 + e
                float block_max = -INFINITY;
#pragma unroll
                for (int t = 0; t < 4; ++t)
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        s[t][e] = t * 16 + quarter * 4 + e <= valid ? s[t][e] * scale : -INFINITY;
                        block_max = fmaxf(block_max, s[t][e]);
                    }
                {
                    float other = block_max;
                    swap_halves(block_max, other);                           // either half's, in both
                    block_max = fmaxf(block_max, other);
                    other = block_max;
                    swap_quarters(block_max, other);
                    block_max = fmaxf(block_max, other);
                }
                const float m_new = fmaxf(m, block_max);
#pragma unroll
                for (int t = 0; t < 4; ++t)
#pragma unroll
                    for (int e = 0; e < 4; ++e) s[t][e] = sees && t * 16 + quarter * 4 + e <= valid ? expf(s[t][e] - m_new) : 0.f;
                // a token that sees no key of the block keeps what it has
                const float correction = sees ? expf(m - m_new) : 1.f;
                {
                    // the sum over the 64 keys in the order of a wavefront's, key = lane: bit 5 of the key first, bit 0 last
                    float of_bits[4];
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        of_bits[e] = (s[0][e] + s[2][e]) + (s[1][e] + s[3][e]);
                        float other = of_bits[e];
                        swap_halves(of_bits[e], other);
                        other = of_bits[e] = of_bits[e] + other;
                        swap_quarters(of_bits[e], other);
                        of_bits[e] += other;
                    }
                    const float total = (of_bits[0] + of_bits[2]) + (of_bits[1] + of_bits[3]);
                    l = sees ? fmaf(l, correction, total) : l;
                    m = sees ? m_new : m;
                }
                // Step u of a tile of 16 keys takes key 4 u + quarter: the four quarters of the wavefront and the four elements of s[t]
                // change places.
#pragma unroll
                for (int t = 0; t < 4; ++t) {
                    float a = s[t][0], b2 = s[t][1], c = s[t][2], d = s[t][3];
                    swap_halves(a, c);
                    swap_halves(b2, d);
                    swap_quarters(a, b2);
                    swap_quarters(c, d);
                    s[t] = sums4{a, b2, c, d};
                }
                const unsigned long long odd_ones = strange[b % 3];          // (the same for the whole workgroup)
                sums4 sum[DT];
#pragma unroll
                for (int dt = 0; dt < DT; ++dt) sum[dt] = sums4{};
#pragma unroll
                for (int t = 0; t < 4; ++t) {                                // 16 keys
                    if (t < 3) read_values(t + 1);
                    float4 (&v)[DT] = v_ahead[t % 2];
                    if (odd_ones != 0) {                                     // must not meet the zeros of tokens that do not see it
#pragma unroll
                        for (int dt = 0; dt < DT; ++dt) {
                            v[dt].x = fabsf(v[dt].x) <= LARGEST ? v[dt].x : 0.f; v[dt].y = fabsf(v[dt].y) <= LARGEST ? v[dt].y : 0.f;
                            v[dt].z = fabsf(v[dt].z) <= LARGEST ? v[dt].z : 0.f; v[dt].w = fabsf(v[dt].w) <= LARGEST ? v[dt].w : 0.f;
                        }
                    }
#pragma unroll
                    for (int u = 0; u < 4; ++u)
#pragma unroll
                        for (int dt = 0; dt < DT; ++dt)
                            sum[dt] = __builtin_amdgcn_mfma_f32_16x16x4f32(u == 0 ? v[dt].x : u == 1 ? v[dt].y : u == 2 ? v[dt].z : v[dt].w, s[t][u], sum[dt], 0, 0, 0);
                    __builtin_amdgcn_sched_barrier(0);
                }
                // infinite values and NaN, token by token, for those who see them (seldom any)
                for (unsigned long long left = odd_ones; left != 0; left &= left - 1) {
                    const int key = (int)__ffsll(left) - 1;
                    // its probability lies in step key % 16 / 4 of its tile, in the lanes of quarter key % 4
                    float mine = 0.f;
#pragma unroll
                    for (int t = 0; t < 4; ++t)
#pragma unroll
                        for (int u = 0; u < 4; ++u)
                            if (t == key / 16 && u == key % 16 / 4) mine = s[t][u];
                    const float probability = __shfl(mine, key % 4 * 16 + column, XRT_WAVE);
#pragma unroll
                    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
                        for (int e = 0; e < 4; ++e) {
                            const float v = values[((key / 16 * 4 + key % 4) * HD + dt * 16 + quarter * 4 + e) * 4 + key % 16 / 4];
                            if (key <= valid && !(fabsf(v) <= LARGEST)) sum[dt][e] = fmaf(probability, v, sum[dt][e]);
                        }
                }
#pragma unroll
                for (int dt = 0; dt < DT; ++dt)
#pragma unroll
                    for (int e = 0; e < 4; ++e) o[dt][e] = sees ? fmaf(o[dt][e], correction, sum[dt][e]) : o[dt][e];
            }
            stash(stage ^ 1, b + 1);
            // a chunk's end: what it holds is merged into what the chunks before it left, by the tokens that saw a key of it
            if ((b % CHUNK_BLOCKS == CHUNK_BLOCKS - 1 || b == last_block) && b / CHUNK_BLOCKS * CHUNK_BLOCKS * XRT_BLOCK_TOKENS <= wave_latest) {
                const bool saw = in_run && b / CHUNK_BLOCKS * CHUNK_BLOCKS * XRT_BLOCK_TOKENS <= pos;
                const float m_new = fmaxf(all_m, m);
                const float keep = saw ? expf(all_m - m_new) : 1.f, take = saw ? expf(m - m_new) : 0.f;
                const float taken = l * take;
                all_l = saw ? fmaf(all_l, keep, taken) : all_l;
#pragma unroll
                for (int dt = 0; dt < DT; ++dt)
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        const float part = o[dt][e] * take;
                        all_o[dt][e] = saw ? fmaf(all_o[dt][e], keep, part) : all_o[dt][e];
                        o[dt][e] = 0.f;
                    }
                all_m = saw ? m_new : all_m;
                m = -INFINITY;
                l = 0.f;
            }
        }
        if (in_run) {
            const float inv = all_l > 0.f ? 1.0f / all_l : 0.f;
#pragma unroll
            for (int dt = 0; dt < DT; ++dt)
                *reinterpret_cast<float4*>(dst + dt * 16 + quarter * 4) = make_float4(all_o[dt][0] * inv, all_o[dt][1] * inv, all_o[dt][2] * inv, all_o[dt][3] * inv);
        }
        begin = end;
    }
}

template <int HD>
int launch(const float* q, int row_width, int tokens, int n_heads, int n_kv_heads, const float* k_cache, const float* v_cache, const int* block_table,
           int table_stride, int n_blocks, const int* positions, const int* slots, float* out, float scale, hipStream_t s) {
    constexpr int LDS = 2 * 2 * XRT_BLOCK_TOKENS * HD * (int)sizeof(float);
    static const hipError_t configured = hipFuncSetAttribute(reinterpret_cast<const void*>(attention_float_prompts_kernel<HD>),
                                                             hipFuncAttributeMaxDynamicSharedMemorySize, LDS);
    XRT_REQUIRE(configured == hipSuccess, "attention (float32 prompts): cannot reserve LDS: %s", hipGetErrorString(configured));
    const long pairs = ((long)tokens + TILE - 1) / TILE * (n_heads / n_kv_heads);
    attention_float_prompts_kernel<HD><<<dim3((unsigned)((pairs + WAVES - 1) / WAVES), n_kv_heads), THREADS, LDS, s>>>(
        q, row_width, tokens, n_heads, n_kv_heads, k_cache, v_cache, block_table, table_stride, n_blocks, positions, slots, out, scale);
    XRT_LAUNCH_CHECK("attention (float32 prompts)");
    return 0;
}

}  // namespace

// Whether a step of more (token, head) pairs than the general kernel shares the keys of (8 to a compute unit) takes less here than there, where one wavefront goes
// through all keys of up to four heads of a token. In microseconds: here 4.5 a block of 64 keys of 64 dims and 2 besides, for every pass of a workgroup over
// a sequence's keys, and as often as there are workgroups for a compute unit; there 0.04 a thousand (pair, key) of 64 dims, and no less than 0.15 a key. A workgroup's tokens
// (16, where the heads of a tile are whole workgroups; 64 for groups of one head; else 32, of which some workgroups take parts of two tiles) may be of
// several sequences, which are passes one after the other. Of 586 steps drawn at random (8 to 200 tokens a sequence, 1 to 148 sequences, behind 0 to 2000
// tokens, groups of 1 to 16 heads, 64 and 128 dims) the choice is 5 % off the better of the two on average and never more than 1.5 times; by tokens a
// sequence alone (8, or 32 and 64 where groups are smaller than four heads) it was 30 % off, up to 5 times: 30 sequences of 9 tokens at 60, 14 heads on 2, 17 us there and
// 54 here, 40 of 8 at 300, 10 on 2, 51 and 105. What is served: 40 of 8 at 2000, 32 on 8, 1165 -> 319; 20 of 16 at 2000, 28 on 4, 734 -> 313; 1 of 300 at 3000, 12 on 12, 397 -> 231.
static bool takes_less(int tokens, int n_heads, int n_kv_heads, int head_dim, int fewest, int max_context) {
    const int group = n_heads / n_kv_heads, span = group % WAVES == 0 ? TILE : group == 1 ? SPAN : 2 * TILE;
    const int passes = tokens < 2L * fewest ? 1 : 1 + (span - 2 + fewest) / fewest;
    const double wide = head_dim / 64.0, keys = max_context, pairs = (double)tokens * n_heads;
    const double workgroups = (tokens + TILE - 1) / TILE * (double)n_heads / WAVES;
    const double here = 5 + passes * (4.5 * wide * ((max_context + XRT_BLOCK_TOKENS - 1) / XRT_BLOCK_TOKENS) + 2) * std::max(1.0, workgroups / XRT_COMPUTE_UNITS);
    const double there = 9 + wide * std::max(0.15 * keys, 0.04 * pairs * (keys - 0.5 * fewest) / 1000);
    return here <= there;
}

extern "C" int xrt_attention_float_prompts_accepts(const void* qkv, int tokens, int n_heads, int n_kv_heads, int head_dim, const void* k_cache,
                                                   const void* v_cache, const void* out, int fewest, int max_context) {
    return (head_dim == 64 || head_dim == 128) && n_heads > 0 && n_kv_heads > 0 && n_heads % n_kv_heads == 0 && n_kv_heads <= XRT_GRID_ROWS &&
           fewest >= TILE / 2 && (long)tokens * n_heads > 8L * XRT_COMPUTE_UNITS && max_context > 0 &&
           takes_less(tokens, n_heads, n_kv_heads, head_dim, fewest, max_context) &&
           (uintptr_t)qkv % 16 == 0 && (uintptr_t)out % 16 == 0 && (uintptr_t)k_cache % 32 == 0 && (uintptr_t)v_cache % 32 == 0;
}

extern "C" int xrt_attention_float_prompts(const void* qkv, int tokens, int n_heads, int n_kv_heads, int head_dim, const void* k_cache,
                                           const void* v_cache, const int* block_table, int table_stride, int n_blocks, const int* positions,
                                           const int* slots, void* out, float scale, int fewest, int max_context, void* stream) {
    XRT_REQUIRE(qkv && k_cache && v_cache && block_table && positions && slots && out, "attention (float32 prompts): null operand");
    XRT_REQUIRE(table_stride > 0 && n_blocks > 0, "attention (float32 prompts): empty cache");
    XRT_REQUIRE(xrt_attention_float_prompts_accepts(qkv, tokens, n_heads, n_kv_heads, head_dim, k_cache, v_cache, out, fewest, max_context),
                "attention (float32 prompts): %d tokens, %d at least a sequence, up to %d keys, %d/%d heads of %d dims are not served", tokens, fewest, max_context, n_heads, n_kv_heads, head_dim);
    const int row_width = (n_heads + 2 * n_kv_heads) * head_dim;
    hipStream_t s = (hipStream_t)stream;
    if (head_dim == 64)
        return launch<64>((const float*)qkv, row_width, tokens, n_heads, n_kv_heads, (const float*)k_cache, (const float*)v_cache, block_table, table_stride,
                          n_blocks, positions, slots, (float*)out, scale, s);
    return launch<128>((const float*)qkv, row_width, tokens, n_heads, n_kv_heads, (const float*)k_cache, (const float*)v_cache, block_table, table_stride,
                       n_blocks, positions, slots, (float*)out, scale, s);
}
