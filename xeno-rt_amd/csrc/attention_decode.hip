// Decode attention on the matrix cores: every sequence brings one query token; its keys and
// values are read once from the cache, in chunks spread over many wavefronts, and applied to
// all query heads of a key/value head together.
//
// Formulas: crates/xrt-models/src/llama.rs:504-574 of the reference (score = q.k * scale over
// keys 0..pos, online softmax with running maximum and sum, weighted sum of values, division
// by the sum); query head h uses key/value head h / group.
//
// One wavefront takes one chunk of keys of one (token, key/value head, tile of 16 query
// heads). Scores: S[key][head] = K Q^T with v_mfma_f32_16x16x32_bf16, keys as rows (A operand),
// the query heads as columns. Values: O[dim][head] += V^T P, with the transposed value block
// as A operand and the probabilities, still in the registers the scores came in, as B
// operand: key rows are assigned to accumulator rows such that every lane ends up holding
// eight consecutive keys, exactly the K slots of the next product. A cache block lies in
// memory in the order of these operands (cache_layout.h): every load instruction takes one
// contiguous kilobyte, which nobody else reads, and passes the caches by (non-temporal; with
// keys as rows of head_dim elements an instruction took half a line of each of 16 keys and the
// kernel read 6.1 TB/s where it now reads 6.9). A block's values are asked for before its
// scores are computed, the next block's keys right after. The four (or eight) wavefronts of a workgroup
// merge their results (maximum, sum, O) through LDS into one partial result; a second kernel
// merges the partial results of a token, in order.
//
// The kernel can also finish what follows the q/k/v projection (xrt_qkv_finish: the RMSNorm of every head of q and k,
// the rotation, the write of the new key and value into the cache), so that a decode step of a model with head
// norms needs no kernel between the projection and the attention. The formulas and their order are those of
// qkv_prepare.hip (crates/xrt-models/src/llama.rs:1025-1040, crates/xrt-kernels/src/cpu/rope.rs:59-89). A lane holds
// the dims 32 s + 8 c .. + 7 (s = 0 .. HD/32 - 1) of its query head, so the two dims of a rotation's pair (d and
// d + HD/2) lie in one lane, and the norm's sum over a head is an exchange among four lanes. The new key and
// value are the work of the wavefront whose keys end with the sequence's newest block: its registers hold the block as it came
// from the cache, where the place of the newest token still holds what was there before. The new key's scores are a product of
// their own and take the place of that row's; the new value takes its place in the registers where the block's tail is masked
// anyway; and both are written to the cache for the steps to come.
//
// What bounds short contexts is not memory but one wavefront's chain of instructions and waits: the slot and the position (asked for together), the
// block table, the first keys and values (all on their way before anything is waited for), the heads' finish, scores, values, merge. So what was in that chain and
// need not be there is out of it. The four lanes of a head exchange by row swaps in the vector registers, not through LDS. A lane asks for two gains and one (cosine, sine)
// instead of 32 and 16, and has the others from the 15 lanes beside it as the multiplications run (in full they were 16 loads of a kilobyte a wavefront, and 64 registers, so that
// the first values had to wait until the heads were finished). Up to 12 heads to a key head leave columns of the products empty: the new key is in one of them and
// is finished with the heads, in one pass (with a pass of its own 0.45 us more at 1 to 8 sequences). The tail of a block is masked by whole registers. In us before and now, heads of 128:
// 16 on 8, 1 sequence, 20 keys 6.9, 5.7; 334 keys 8.2, 7.2; 1000 keys 10.9, 9.5; 8 sequences of 334 keys 10.2, 8.7; 32 of 334 14.0, 12.1; 64 on 8, 8 of 1500 15.8, 14.0; 32 on 2, 1 of 334 9.5, 8.6.
// Without a finish 16 on 8, 1 of 334 5.7, 5.0; 8 of 334 7.6, 7.3; 32 of 3000 (the bandwidth of memory) 62.9, 63.3. A step at the Qwen3-0.6B sizes 889 -> 852 us.
#include "cache_layout.h"
#include "xrt_hip.h"

#include <utility>

namespace {

struct Finish {                       // xrt_qkv_finish with its pointers typed
    const void* q_norm; const void* k_norm; int norm_dtype; float norm_eps;
    const float2* rope_table; int table_positions;     // (cosine, sine) of the positions' angles, [position][pair]; null: no rotation
    bf16* k_cache; bf16* v_cache;
};

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float floatx4 __attribute__((ext_vector_type(4)));

constexpr float LOG2E = 1.4426950408889634f;

// Row r of score tile t (0 or 1) of a group of 32 keys stands for key 8 (r / 4) + 4 t + r % 4: accumulator
// register i of lane group c is row 4 c + i, and must be key 8 c + 4 t + i. The cache keeps the keys so:
// lane (r, c) finds its piece of tile ((g * 2 + t) * KS + s) at place r + 16 c, and of the values' tile
// (g * DT + u) likewise.
constexpr int lane_place(int r, int c) { return (r + 16 * c) * 8; }
static_assert(cache_key_offset(32 + 8 * 2 + 4 * 1 + 3, 32 * 3 + 8 * 1, 128) == ((1 * 2 + 1) * 4 + 3) * 512 + lane_place(2 * 4 + 3, 1), "keys of a block");
static_assert(cache_key_offset(8 * 3 + 4 * 0 + 1, 32 * 1 + 8 * 3 + 5, 64) == ((0 * 2 + 0) * 2 + 1) * 512 + lane_place(3 * 4 + 1, 3) + 5, "keys of a block");
static_assert(cache_value_offset(16 * 5 + 9, 32 + 8 * 2 + 6, 128) == (1 * 8 + 5) * 512 + lane_place(9, 2) + 6, "values of a block");

// What finishing a head reads: the norm's gains (none: gain null), and the (cosine, sine) of this position's HD / 2 angles, as
// xrt_rope_table has worked them out (the same sincosf of the same angles as in qkv_prepare.hip: worked out here, for every workgroup again, they would
// cost more than the kernel saves; from null: no rotation). All of it is asked for ahead of the first keys, whose loads then run while the heads are finished.
// The 16 lanes (0 .. 15, c) need the same ones, of the dims 32 s + 8 c + e: of gain s * 8 + e the lane 4 s + e / 2 asks for (two neighbours), of angle s * 8 + e the lane of that number.
template <typename TW> struct alignas(sizeof(TW) * 2) GainPair { TW e[2]; };
template <int HD, typename TW>
__device__ __forceinline__ GainPair<TW> ask_gains(const TW* __restrict__ gain, int r, int c) {
    if (gain == nullptr) return GainPair<TW>{};
    return *reinterpret_cast<const GainPair<TW>*>(gain + r / 4 % (HD / 32) * 32 + c * 8 + r % 4 * 2);
}
template <int HD>
__device__ __forceinline__ float2 ask_turns(const float2* __restrict__ from, int r, int c) {
    return from == nullptr ? make_float2(1.f, 0.f) : from[r / 8 % (HD / 64) * 32 + c * 8 + r % 8];
}
template <int LANE> __device__ __forceinline__ float of_lane(float v) {          // what the lane (LANE, c) holds, in all lanes (r, c)
    return __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, v), 0x150 + LANE, 0xF, 0xF, true));      // row_newbcast
}
template <int LANE> __device__ __forceinline__ float of_lane(float v, float last) {          // the same of `last` in the lanes (12 .. 15, c)
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(__builtin_bit_cast(int, of_lane<LANE>(v)), __builtin_bit_cast(int, last), 0x150 + LANE, 0xF, 0x8, false));
}
template <typename F, int... I> __device__ __forceinline__ void each(F&& f, std::integer_sequence<int, I...>) { (f(std::integral_constant<int, I>{}), ...); }

// One head (the dims of this lane) through its RMSNorm and the rotation by the token's position, in float32, and back to
// bfloat16: what qkv_prepare does to a head. BOTH: the lanes (12 .. 15, c) hold another kind of head, whose gains are last_gains.
template <int HD, bool BOTH, typename TW>
__device__ __forceinline__ void finish_head(bf16x8 (&x)[HD / 32], bool norms, GainPair<TW> gains, GainPair<TW> last_gains, float eps, bool rotates, float2 turns) {
    constexpr int KS = HD / 32;
    float inv_rms = 1.0f;
    if (norms) {
        float squares = 0.f;
#pragma unroll
        for (int ks = 0; ks < KS; ++ks)
#pragma unroll
            for (int e = 0; e < 8; ++e) squares = fmaf((float)x[ks][e], (float)x[ks][e], squares);
        squares = sum_of_four(squares);                        // the four lanes (r, 0 .. 3) hold the head between them
        inv_rms = 1.0f / sqrtf(squares / (float)HD + eps);
    }
    // a pair of the rotation at a time (dims d and d + HD / 2 lie in x[ks] and x[ks + KS / 2])
    each([&](auto number) {
        constexpr int ks = number, upper_ks = ks + KS / 2;
        float lower[8], upper[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) { lower[e] = (float)x[ks][e]; upper[e] = (float)x[upper_ks][e]; }
        if (norms) {
            each([&](auto element) {
                constexpr int e = element;
                const float mine = to_float(gains.e[e % 2]), last = to_float(last_gains.e[e % 2]);
                if constexpr (BOTH) {
                    lower[e] = lower[e] * inv_rms * of_lane<ks * 4 + e / 2>(mine, last);
                    upper[e] = upper[e] * inv_rms * of_lane<upper_ks * 4 + e / 2>(mine, last);
                } else {
                    lower[e] = lower[e] * inv_rms * of_lane<ks * 4 + e / 2>(mine);
                    upper[e] = upper[e] * inv_rms * of_lane<upper_ks * 4 + e / 2>(mine);
                }
            }, std::make_integer_sequence<int, 8>{});
        }
        if (rotates) {
            each([&](auto element) {
                constexpr int e = element;
                const float cosine = of_lane<ks * 8 + e>(turns.x), sine = of_lane<ks * 8 + e>(turns.y);
                const float a = lower[e], b = upper[e];
                lower[e] = a * cosine - b * sine;
                upper[e] = a * sine + b * cosine;
            }, std::make_integer_sequence<int, 8>{});
        }
#pragma unroll
        for (int e = 0; e < 8; ++e) { x[ks][e] = (bf16)lower[e]; x[upper_ks][e] = (bf16)upper[e]; }
    }, std::make_integer_sequence<int, KS / 2>{});
}

enum { FINISH_NONE, FINISH_APART, FINISH_FOLDED };       // nothing to finish; the new key in registers of its own; the new key in the columns 12 .. 15 of the query heads' products

// FINISH: q, k and v come as the projection left them, and `finish` says what is still to do (see the head of this file).
// TW: the element type of the head norms' gains.
template <int HD, int FINISH, int WAVES, typename TW>
__global__ void __launch_bounds__(WAVES * XRT_WAVE, 2) attention_decode_kernel(
    const bf16* __restrict__ qkv, int row_width, int group, int n_kv_heads,
    const bf16* __restrict__ k_cache, const bf16* __restrict__ v_cache, const int* __restrict__ block_table,
    int table_stride, int n_blocks, const int* __restrict__ positions, const int* __restrict__ slots,
    float scale, int chunk_blocks, int n_parts, int q_tiles,
    float* __restrict__ part_o, float* __restrict__ part_ml, bf16* __restrict__ out, const Finish finish) {
    constexpr int KS = HD / 32;                    // K steps of the score product
    constexpr int DT = HD / 16;                    // 16-row tiles of the value product
    extern __shared__ __attribute__((aligned(16))) char lds[];
    floatx4 (*merge_o)[DT][XRT_WAVE] = reinterpret_cast<floatx4 (*)[DT][XRT_WAVE]>(lds);                    // [WAVES]
    float (*merge_ml)[2][16] = reinterpret_cast<float (*)[2][16]>(lds + sizeof(floatx4) * WAVES * DT * XRT_WAVE);      // [WAVES]

    const int lane = threadIdx.x % XRT_WAVE, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / XRT_WAVE);   // in a scalar register, and with it the blocks' numbers
    const int r = lane % 16, c = lane / 16;
    const int part = blockIdx.x;                   // this workgroup's chunks become one partial result
    const int chunk = part * WAVES + wave;
    const int n_heads = group * n_kv_heads;
    int kv_head = blockIdx.y, q_tile = 0;
    if (q_tiles > 1) { kv_head = blockIdx.y / q_tiles; q_tile = blockIdx.y % q_tiles; }
    const int token = blockIdx.z;
    int slot = slots[token], pos = positions[token];
    asm volatile("" : "+s"(slot), "+s"(pos));      // both are there before the branch (left alone, the compiler asks for the position behind it)
    if (slot < 0) {                                // padding: the whole workgroup leaves
        // (with one partial result per head there is no merge kernel after this one to write the zeros)
        if (n_parts == 1 && wave == 0 && q_tile * 16 + r < group) {
            bf16* dst = out + ((long)token * n_heads + kv_head * group + q_tile * 16 + r) * HD;
            for (int d = c; d < HD; d += 4) dst[d] = (bf16)0.f;
        }
        return;
    }
    const int n_keys = pos + 1;
    if (part * WAVES * chunk_blocks * XRT_BLOCK_TOKENS >= n_keys) return;      // nothing here for any wavefront
    const int first_block = chunk * chunk_blocks;
    const bool active = first_block * XRT_BLOCK_TOKENS < n_keys;
    const int last_block = min((n_keys - 1) / XRT_BLOCK_TOKENS, first_block + chunk_blocks - 1);
    const int head_in_group = q_tile * 16 + r;             // this lane's query head (column of the products)
    const bool head_valid = head_in_group < group;
    const int head = kv_head * group + min(head_in_group, group - 1);

    const float scale2 = scale * LOG2E;                    // scores are kept in units of log2
    float m = -INFINITY, l = 0.f;
    floatx4 o[DT];

    if (active) {
        bf16x8 q[KS];
        const bool key_lane = FINISH == FINISH_FOLDED && r >= 12;
        const int row_head = key_lane ? n_heads + kv_head : head;
#pragma unroll
        for (int ks = 0; ks < KS; ++ks)
            q[ks] = *reinterpret_cast<const bf16x8*>(qkv + (long)token * row_width + (long)row_head * HD + ks * 32 + c * 8);
        // Loads are always on their way: a block's values are asked for before its scores are computed, and the
        // next block's keys right after, before the softmax and the value product of this one.
        const int* table = block_table + (long)slot * table_stride;
        auto block_of = [&](int b) { return min(max(table[min(b, last_block)], 0), n_blocks - 1); };   // the host never hands out anything else
        bf16x8 kreg[2][2][KS], vreg[2][DT];
        auto ask_keys = [&](int block) {
            const bf16* kb = k_cache + ((long)block * n_kv_heads + kv_head) * XRT_BLOCK_TOKENS * HD;
#pragma unroll
            for (int g = 0; g < 2; ++g)
#pragma unroll
                for (int t = 0; t < 2; ++t)
#pragma unroll
                    for (int ks = 0; ks < KS; ++ks)
                        kreg[g][t][ks] = __builtin_nontemporal_load(reinterpret_cast<const bf16x8*>(kb + ((g * 2 + t) * KS + ks) * 512 + lane * 8));
        };
        auto ask_values = [&](int block) {
            const bf16* vb = v_cache + ((long)block * n_kv_heads + kv_head) * HD * XRT_BLOCK_TOKENS;
#pragma unroll
            for (int g = 0; g < 2; ++g)
#pragma unroll
                for (int dt = 0; dt < DT; ++dt)
                    vreg[g][dt] = __builtin_nontemporal_load(reinterpret_cast<const bf16x8*>(vb + (g * DT + dt) * 512 + lane * 8));
        };
        // The sequence's newest token: its block and its place there. What is still to do to q and to the new key
        // is done while the first keys and values are on their way, with everything that it reads
        // asked for before them (loads arrive in their order: behind the keys it would wait for those too).
        const int newest_block = (unsigned)pos / XRT_BLOCK_TOKENS;
        const unsigned newest = (unsigned)pos % XRT_BLOCK_TOKENS;
        const bool has_newest = FINISH != FINISH_NONE && last_block == newest_block;
        bf16x8 new_key[KS];                            // (FINISH_APART)
        unsigned short new_value[DT / 4];              // dims 16 (4 i + c) + r
        GainPair<TW> q_gains, k_gains;
        float2 turns;
        const float2* turns_from = nullptr;
        int block = block_of(first_block), next_block = block_of(first_block + 1);
        const int newest_place = FINISH == FINISH_NONE ? 0 : block_of(newest_block);
        if constexpr (FINISH != FINISH_NONE) {
            if (finish.rope_table != nullptr) turns_from = finish.rope_table + (long)min(pos, finish.table_positions - 1) * (HD / 2);   // (the host sends only steps that the table covers)
            q_gains = ask_gains<HD, TW>((const TW*)finish.q_norm, r, c);
            turns = ask_turns<HD>(turns_from, r, c);
            if (has_newest) {                          // (the same for all lanes of the wavefront)
                const bf16* key_row = qkv + (long)token * row_width + (long)(n_heads + kv_head) * HD;
                const unsigned short* value_row = reinterpret_cast<const unsigned short*>(key_row + (long)n_kv_heads * HD);
#pragma unroll
                for (int i = 0; i < DT / 4; ++i) new_value[i] = value_row[(4 * i + c) * 16 + r];
                if constexpr (FINISH == FINISH_APART) {
#pragma unroll
                    for (int ks = 0; ks < KS; ++ks) new_key[ks] = *reinterpret_cast<const bf16x8*>(key_row + ks * 32 + c * 8);
                }
                k_gains = ask_gains<HD, TW>((const TW*)finish.k_norm, r, c);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        ask_keys(block);
        ask_values(block);
        if constexpr (FINISH != FINISH_NONE) {
            __builtin_amdgcn_sched_barrier(0);
            const bool norms = finish.q_norm != nullptr, rotates = turns_from != nullptr;
            if (FINISH == FINISH_FOLDED && has_newest) {
                finish_head<HD, true>(q, norms, q_gains, k_gains, finish.norm_eps, rotates, turns);
            } else {
                finish_head<HD, false>(q, norms, q_gains, q_gains, finish.norm_eps, rotates, turns);
                if constexpr (FINISH == FINISH_APART) {
                    if (has_newest) finish_head<HD, false>(new_key, norms, k_gains, k_gains, finish.norm_eps, rotates, turns);
                }
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        // The newest key against the query heads: in every row of the product (FINISH_APART), or in the rows 12 .. 15 (FINISH_FOLDED)
        float new_score = 0.f;
        if (has_newest) {
            floatx4 product = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int ks = 0; ks < KS; ++ks)
                product = __builtin_amdgcn_mfma_f32_16x16x32_bf16(FINISH == FINISH_FOLDED ? q[ks] : new_key[ks], q[ks], product, 0, 0, 0);
            new_score = FINISH == FINISH_FOLDED ? as_value(of_row<3>(as_word(product[0]))) : product[0];
            if (q_tile == 0) {                             // one of the workgroups that share the key/value head writes to the cache
                const long base = ((long)newest_place * n_kv_heads + kv_head) * XRT_BLOCK_TOKENS * HD;
#pragma unroll
                for (int i = 0; i < DT / 4; ++i)
                    reinterpret_cast<unsigned short*>(finish.v_cache)[base + cache_value_offset((4 * i + c) * 16 + r, newest, HD)] = new_value[i];
                if (r == 15) {
#pragma unroll
                    for (int ks = 0; ks < KS; ++ks)
                        *reinterpret_cast<bf16x8*>(finish.k_cache + base + cache_key_offset(newest, ks * 32 + c * 8, HD)) = FINISH == FINISH_FOLDED ? q[ks] : new_key[ks];
                }
            }
        }
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) o[dt] = floatx4{0.f, 0.f, 0.f, 0.f};
        for (int b = first_block; b <= last_block; ++b) {
            const int valid = min(XRT_BLOCK_TOKENS, n_keys - b * XRT_BLOCK_TOKENS);   // keys of this block that exist
            const bool newest_here = has_newest && b == newest_block;
            // ---- scores of 64 keys: two groups of 32, two tiles of 16 rows each
            floatx4 s[2][2];
#pragma unroll
            for (int g = 0; g < 2; ++g)
#pragma unroll
                for (int t = 0; t < 2; ++t) {
                    s[g][t] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                    for (int ks = 0; ks < KS; ++ks)
                        s[g][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kreg[g][t][ks], q[ks], s[g][t], 0, 0, 0);
                }
            block = next_block;
            next_block = block_of(b + 2);
            if (b < last_block) ask_keys(block);
            if constexpr (FINISH != FINISH_NONE) {
                if (newest_here) {                     // its score takes the place of what the old key there gave
#pragma unroll
                    for (int g = 0; g < 2; ++g)
#pragma unroll
                        for (int t = 0; t < 2; ++t)
#pragma unroll
                            for (int i = 0; i < 4; ++i)
                                s[g][t][i] = g * 32 + c * 8 + t * 4 + i == (int)newest ? new_score : s[g][t][i];
                }
            }
            // register i of s[g][t] is key g*32 + c*8 + t*4 + i, for query head r
            float block_max = -INFINITY;
#pragma unroll
            for (int g = 0; g < 2; ++g)
#pragma unroll
                for (int t = 0; t < 2; ++t)
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        const int key = g * 32 + c * 8 + t * 4 + i;
                        const float v = key < valid ? s[g][t][i] * scale2 : -INFINITY;   // also drops whatever lies past the end
                        s[g][t][i] = v;
                        block_max = fmaxf(block_max, v);
                    }
            block_max = max_of_four(block_max);
            const float m_new = fmaxf(m, block_max);           // finite: key 0 of the block exists
            const float correction = __builtin_amdgcn_exp2f(m - m_new);
            m = m_new;
            l *= correction;
#pragma unroll
            for (int dt = 0; dt < DT; ++dt) o[dt] *= correction;

            // ---- probabilities, and the value product
#pragma unroll
            for (int g = 0; g < 2; ++g) {
                bf16x8 p;
#pragma unroll
                for (int t = 0; t < 2; ++t)
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        const float e = __builtin_amdgcn_exp2f(s[g][t][i] - m_new);
                        l += e;
                        p[t * 4 + i] = (bf16)e;
                    }
                // What lies behind the keys that exist belongs to nobody and must not meet the zeros of p; the newest value takes its place
                const int kept = (newest_here ? valid - 1 : valid) - g * 32;      // of these 32 tokens
                if (kept < 32) {
                    const int mine = kept - c * 8;                 // of the eight of this lane
                    unsigned keep[4], put[4];
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        keep[i] = mine >= 2 * i + 2 ? ~0u : (mine == 2 * i + 1 ? 0xFFFFu : 0u);
                        if constexpr (FINISH != FINISH_NONE) put[i] = !newest_here ? 0u : (mine == 2 * i ? 0xFFFFu : (mine == 2 * i + 1 ? 0xFFFF0000u : 0u));
                    }
                    each([&](auto tile) {
                        constexpr int dt = tile;
                        union { bf16x8 v; unsigned words[4]; } piece{vreg[g][dt]};
                        unsigned value = 0;
                        if constexpr (FINISH != FINISH_NONE) value = of_row<dt % 4>(new_value[dt / 4]) * 0x10001u;
#pragma unroll
                        for (int i = 0; i < 4; ++i) {
                            piece.words[i] &= keep[i];
                            if constexpr (FINISH != FINISH_NONE) piece.words[i] |= value & put[i];
                        }
                        vreg[g][dt] = piece.v;
                    }, std::make_integer_sequence<int, DT>{});
                }
#pragma unroll
                for (int dt = 0; dt < DT; ++dt) o[dt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vreg[g][dt], p, o[dt], 0, 0, 0);
            }
            if (b < last_block) ask_values(block);
        }
        l = sum_of_four(l);
    } else {
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) o[dt] = floatx4{0.f, 0.f, 0.f, 0.f};
    }

    // ---- the wavefronts' results become one, in wavefront order
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) merge_o[wave][dt][lane] = o[dt];
    if (c == 0) {
        merge_ml[wave][0][r] = m;                  // -inf for a wavefront without keys
        merge_ml[wave][1][r] = l;
    }
    __syncthreads();
    if (!head_valid) return;
    float m_all = merge_ml[0][0][r];
#pragma unroll
    for (int w = 1; w < WAVES; ++w) m_all = fmaxf(m_all, merge_ml[w][0][r]);
    float l_all = 0.f, weight[WAVES];
#pragma unroll
    for (int w = 0; w < WAVES; ++w) {
        weight[w] = __builtin_amdgcn_exp2f(merge_ml[w][0][r] - m_all);      // 0 for a wavefront without keys
        l_all += weight[w] * merge_ml[w][1][r];
    }
    const float inv = l_all > 0.f ? 1.0f / l_all : 0.f;
    const long row = (long)token * n_heads + head, index = row * n_parts + part;
    // every wavefront adds up some of the tiles of dims; accumulator register i of tile dt is dimension dt*16 + c*4 + i, for query head r
    for (int dt = wave; dt < DT; dt += WAVES) {
        floatx4 total = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int w = 0; w < WAVES; ++w) total += merge_o[w][dt][lane] * weight[w];
        if (n_parts == 1) {
            // the workgroup has seen all keys of the sequence: this is the result, and no merge kernel follows
            struct alignas(8) Four { bf16 e[4]; } four;
#pragma unroll
            for (int i = 0; i < 4; ++i) four.e[i] = (bf16)(total[i] * inv);
            *reinterpret_cast<Four*>(out + row * HD + dt * 16 + c * 4) = four;
        } else {
            *reinterpret_cast<floatx4*>(part_o + index * HD + dt * 16 + c * 4) = total;
        }
    }
    if (n_parts > 1 && wave == 0 && c == 0) {
        part_ml[index * 2] = m_all;
        part_ml[index * 2 + 1] = l_all;
    }
}

// Merges the partial results of one (token, head): out = sum_k w_k O_k / sum_k w_k l_k with
// w_k = 2^(m_k - max m), in order. One thread per dimension. The weights are worked out once,
// by one thread per partial result, and shared through LDS; maximum and sum are wavefront
// reductions in a fixed order.
template <int HD>
__global__ void __launch_bounds__(HD) attention_decode_merge_kernel(
    const float* __restrict__ part_o, const float* __restrict__ part_ml, const int* __restrict__ positions,
    const int* __restrict__ slots, int n_heads, int part_keys, int n_parts, bf16* __restrict__ out) {
    extern __shared__ float weights[];                    // n_parts
    __shared__ float reduce[HD / XRT_WAVE][2];
    const int token = blockIdx.y, head = blockIdx.x, d = threadIdx.x;
    const int lane = d % XRT_WAVE, wave = d / XRT_WAVE;
    bf16* dst = out + ((long)token * n_heads + head) * HD;
    const long base = ((long)token * n_heads + head) * n_parts;
    const float* column = part_o + base * HD + d;
    // Everything this thread may need is asked for at once, before it is known how many partial
    // results count: the loads then cost one trip to memory instead of one after the other.
    // What lies beyond the partial results that count is read (it is inside the workspace) and
    // never used.
    constexpr int EARLY = 16;
    float early_o[EARLY];
#pragma unroll
    for (int k = 0; k < EARLY; ++k) early_o[k] = k < n_parts ? column[(long)k * HD] : 0.f;
    const float2 early_ml = d < n_parts ? *reinterpret_cast<const float2*>(part_ml + (base + d) * 2) : make_float2(0.f, 0.f);
    const int slot = slots[token];
    const int n_keys = positions[token] + 1;
    if (slot < 0) {
        dst[d] = (bf16)0.f;
        return;
    }
    const int parts = min(n_parts, (n_keys + part_keys - 1) / part_keys);
    float m = d < parts ? early_ml.x : -INFINITY;
    for (int k = d + HD; k < parts; k += HD) m = fmaxf(m, part_ml[(base + k) * 2]);
    m = whole_wave_max(m);
    if (lane == 0) reduce[wave][0] = m;
    __syncthreads();
    m = reduce[0][0];
#pragma unroll
    for (int w = 1; w < HD / XRT_WAVE; ++w) m = fmaxf(m, reduce[w][0]);
    float l = 0.f;
    if (d < parts) {
        const float weight = __builtin_amdgcn_exp2f(early_ml.x - m);
        weights[d] = weight;
        l = weight * early_ml.y;
    }
    for (int k = d + HD; k < parts; k += HD) {
        const float weight = __builtin_amdgcn_exp2f(part_ml[(base + k) * 2] - m);
        weights[k] = weight;
        l = fmaf(weight, part_ml[(base + k) * 2 + 1], l);
    }
    l = whole_wave_sum(l);
    if (lane == 0) reduce[wave][1] = l;
    __syncthreads();
    l = reduce[0][1];
#pragma unroll
    for (int w = 1; w < HD / XRT_WAVE; ++w) l += reduce[w][1];
    float acc = 0.f;
#pragma unroll
    for (int k = 0; k < EARLY; ++k)
        if (k < parts) acc = fmaf(weights[k], early_o[k], acc);
#pragma unroll 8
    for (int k = EARLY; k < parts; ++k) acc = fmaf(weights[k], column[(long)k * HD], acc);
    dst[d] = (bf16)(l > 0.f ? acc / l : 0.f);
}

// How the keys of the longest sequence are cut: blocks per wavefront, and partial results
// (each from the wavefronts of a workgroup) per (token, head).
struct Cut { int chunk_blocks, n_parts, waves; };

Cut cut_for(int tokens, int n_kv_heads, int q_tiles, int max_context, int head_dim) {
    constexpr int WAVES = 4;                       // of a workgroup, but for the short contexts below
    const int max_blocks = (max_context + XRT_BLOCK_TOKENS - 1) / XRT_BLOCK_TOKENS;
    const long pairs = (long)tokens * n_kv_heads * q_tiles;
    // Up to eight blocks: one workgroup sees all keys, and nothing is left to merge. From five blocks on it has eight wavefronts, a block
    // each, where every pair finds a compute unit of its own, and four of two blocks beyond (16 heads of 128 on 8, 334 keys: 1 sequence 7.4 us in two
    // parts and their merge, 6.0 with four wavefronts, 5.8 with eight; 16 sequences 9.1, 8.4, 7.9; 48 sequences 18.0, 14.4, 15.9; heads of 64 gain
    // 0.2 to 1 us by the eight; all before the chain was as short as it is: 5.0 and 7.3 for 1 and 8 sequences now). Nine blocks and more: two blocks one after the other in
    // eight wavefronts cost less than parts and their merge where the sequences are much shorter than max_context and more where they are not (1 sequence, with the finish, 334 keys of up to 1024
    // 6.6 against 8.4, 600 keys 8.5 and 8.5, 1000 keys 11.5 against 9.0: a compute unit takes its half megabyte at 50 bytes a cycle). (max_context is what the caller says of the step:
    // a recorded decode step says the engine's limit or the next 1024 tokens, whichever is less, so that it comes here in engines for up to 512 tokens.)
    if (max_blocks <= 8) {
        const int waves = max_blocks > 4 && pairs <= XRT_COMPUTE_UNITS ? 8 : 4;
        return Cut{(max_blocks + waves - 1) / waves, 1, waves};
    }
    // How long the kernel takes is set by the compute unit with the most to do: workgroups are dealt out to
    // the 256 compute units in turn, and a compute unit works off its share at its own pace (two workgroups
    // at a time are no faster than one after the other). Measured at head size 128: 6.3 us for a block of 64
    // keys per wavefront, 0.7 us per workgroup, about 5 us for the merge kernel. So the cut is chosen for
    // the fewest blocks per compute unit: 384 workgroups of 16 blocks (two on every second compute unit) are
    // slower than 768 of 8. The longer chunk wins among equals (less to merge); with one workgroup per (token,
    // key/value head) pair nothing is left to merge and the merge kernel is not launched.
    const long block_ns = 6300L * head_dim / 128, group_ns = 700, merge_ns = 5000;
    const int longest = (max_blocks + WAVES - 1) / WAVES;
    long best_ns = -1;
    Cut best{longest, 1, WAVES};
    for (int chunk_blocks = longest; chunk_blocks >= 1; --chunk_blocks) {
        const int n_chunks = (max_blocks + chunk_blocks - 1) / chunk_blocks;
        const int n_parts = (n_chunks + WAVES - 1) / WAVES;
        if ((long)(n_parts - 1) * WAVES * chunk_blocks >= max_blocks) continue;         // a part without keys: a shorter chunk does the same
        const long per_unit = (pairs * n_parts + XRT_COMPUTE_UNITS - 1) / XRT_COMPUTE_UNITS;
        const long ns = per_unit * (chunk_blocks * block_ns + group_ns) + (n_parts > 1 ? merge_ns : 0);
        if (best_ns < 0 || ns < best_ns) { best_ns = ns; best = Cut{chunk_blocks, n_parts, WAVES}; }
    }
    // (Eight wavefronts where one workgroup sees all keys of a longer context: the same on average over 451 steps drawn at random, up to 1.18 times as long where a
    // few blocks do not divide among them, 193 sequences of 1104, 16 heads of 64 on 4: 42 -> 49 us.)
    return best;
}

template <int HD>
int launch(const bf16* qkv, int tokens, int n_heads, int n_kv_heads, const bf16* k_cache, const bf16* v_cache,
           const int* block_table, int table_stride, int n_blocks, const int* positions, const int* slots, bf16* out,
           float scale, int max_context, float* workspace, long workspace_floats, const Finish* finish, hipStream_t s) {
    const int group = n_heads / n_kv_heads;
    const int q_tiles = (group + 15) / 16;
    const Cut cut = cut_for(tokens, n_kv_heads, q_tiles, max_context, HD);
    const long need = cut.n_parts == 1 ? 0 : (long)tokens * n_heads * cut.n_parts * (HD + 2);
    XRT_REQUIRE(need == 0 || (workspace != nullptr && workspace_floats >= need),
                "attention (decode): workspace of %ld floats given, %ld needed", workspace_floats, need);
    float* part_o = workspace;
    float* part_ml = workspace + (long)tokens * n_heads * cut.n_parts * HD;
    const int row_width = (n_heads + 2 * n_kv_heads) * HD;
    XRT_REQUIRE(tokens <= XRT_GRID_ROWS && n_kv_heads * q_tiles <= XRT_GRID_ROWS, "attention (decode): grid too large");
    const dim3 grid(cut.n_parts, n_kv_heads * q_tiles, tokens);
    const size_t lds = cut.waves * (sizeof(floatx4) * HD / 16 * XRT_WAVE + 2 * 16 * sizeof(float));
#define XRT_DECODE(FINISH_, WAVES_, TW_, HOW)                                                                                           \
    do {                                                                                                                            \
        static const hipError_t room = hipFuncSetAttribute(reinterpret_cast<const void*>(attention_decode_kernel<HD, FINISH_, WAVES_, TW_>),   \
                                                           hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);                 \
        XRT_REQUIRE(room == hipSuccess, "attention (decode): cannot reserve LDS: %s", hipGetErrorString(room));                    \
        attention_decode_kernel<HD, FINISH_, WAVES_, TW_><<<grid, WAVES_ * XRT_WAVE, lds, s>>>(                                            \
            qkv, row_width, group, n_kv_heads, k_cache, v_cache, block_table, table_stride, n_blocks, positions, slots,              \
            scale, cut.chunk_blocks, cut.n_parts, q_tiles, part_o, part_ml, out, HOW);                                              \
    } while (0)
    const bool float_gains = finish != nullptr && finish->norm_dtype == XRT_F32;
#define XRT_DECODE_FINISHING(FINISH_)                                                          \
    do {                                                                                       \
        if (cut.waves == 8 && float_gains) XRT_DECODE(FINISH_, 8, float, *finish);             \
        else if (cut.waves == 8) XRT_DECODE(FINISH_, 8, bf16, *finish);                        \
        else if (float_gains) XRT_DECODE(FINISH_, 4, float, *finish);                          \
        else XRT_DECODE(FINISH_, 4, bf16, *finish);                                            \
    } while (0)
    // (up to 12 heads the columns 12 .. 15 are empty: see the head of this file)
    if (finish != nullptr && group <= 12) XRT_DECODE_FINISHING(FINISH_FOLDED);
    else if (finish != nullptr) XRT_DECODE_FINISHING(FINISH_APART);
    else if (cut.waves == 8) XRT_DECODE(FINISH_NONE, 8, bf16, Finish{});
    else XRT_DECODE(FINISH_NONE, 4, bf16, Finish{});
#undef XRT_DECODE_FINISHING
#undef XRT_DECODE
    XRT_LAUNCH_CHECK("attention (decode)");
    if (cut.n_parts == 1) return 0;
    const int part_keys = cut.chunk_blocks * cut.waves * XRT_BLOCK_TOKENS;
    attention_decode_merge_kernel<HD><<<dim3(n_heads, tokens), HD, cut.n_parts * sizeof(float), s>>>(
        part_o, part_ml, positions, slots, n_heads, part_keys, cut.n_parts, out);
    XRT_LAUNCH_CHECK("attention (decode merge)");
    return 0;
}

}  // namespace

bool xrt_attention_decode_accepts(int head_dim) { return head_dim == 64 || head_dim == 128; }

// floats of workspace that a decode step of `tokens` sequences needs: the partial results of the cut that
// the launcher will choose (none where one workgroup sees all keys of a sequence)
long xrt_attention_decode_workspace(int tokens, int n_heads, int n_kv_heads, int head_dim, int max_context) {
    const int q_tiles = (n_heads / n_kv_heads + 15) / 16;
    const Cut cut = cut_for(tokens, n_kv_heads, q_tiles, max_context, head_dim);
    return cut.n_parts == 1 ? 0 : (long)tokens * n_heads * cut.n_parts * (head_dim + 2);
}

int xrt_attention_decode(const void* qkv, int tokens, int n_heads, int n_kv_heads, int head_dim, const void* k_cache,
                         const void* v_cache, const int* block_table, int table_stride, int n_blocks,
                         const int* positions, const int* slots, void* out, float scale, int max_context,
                         float* workspace, long workspace_floats, const xrt_qkv_finish* finish, hipStream_t s) {
    Finish typed{};
    if (finish != nullptr) {
        XRT_REQUIRE((finish->q_norm == nullptr) == (finish->k_norm == nullptr), "attention (decode): q_norm and k_norm come together");
        XRT_REQUIRE(finish->q_norm == nullptr || finish->norm_dtype == XRT_F32 || finish->norm_dtype == XRT_BF16,
                    "attention (decode): unknown norm dtype %d", finish->norm_dtype);
        XRT_REQUIRE(finish->rope_table == nullptr || (finish->rope_dim == head_dim && finish->table_positions >= max_context),
                    "attention (decode): the rotation that is finished here spans the whole head (%d of %d dims) and its table covers the step's positions (%d of %d)",
                    finish->rope_dim, head_dim, finish->table_positions, max_context);
        XRT_REQUIRE((uintptr_t)k_cache % 16 == 0 && (uintptr_t)qkv % 16 == 0 && (uintptr_t)finish->q_norm % 32 == 0 &&
                    (uintptr_t)finish->k_norm % 32 == 0 && (uintptr_t)finish->rope_table % 16 == 0,
                    "attention (decode): operands must be aligned to 16 bytes (norm weights to 32)");
        // the new keys and values go where the old ones are read from
        typed = Finish{finish->q_norm, finish->k_norm, finish->norm_dtype, finish->norm_eps,
                       (const float2*)finish->rope_table, finish->rope_table ? finish->table_positions : 0,
                       (bf16*)const_cast<void*>(k_cache), (bf16*)const_cast<void*>(v_cache)};
    }
    const Finish* typed_or_none = finish != nullptr ? &typed : nullptr;
    if (head_dim == 64)
        return launch<64>((const bf16*)qkv, tokens, n_heads, n_kv_heads, (const bf16*)k_cache, (const bf16*)v_cache,
                          block_table, table_stride, n_blocks, positions, slots, (bf16*)out, scale, max_context,
                          workspace, workspace_floats, typed_or_none, s);
    return launch<128>((const bf16*)qkv, tokens, n_heads, n_kv_heads, (const bf16*)k_cache, (const bf16*)v_cache,
                       block_table, table_stride, n_blocks, positions, slots, (bf16*)out, scale, max_context,
                       workspace, workspace_floats, typed_or_none, s);
}
