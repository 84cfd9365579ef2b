// After the q/k/v projection, in one pass over a token's heads: RMSNorm of every head of
// q and k (one weight [head_dim] each), rotation of q and k by the token's position, and
// the write of k (rotated) and v (raw) into the sequence's cache block.
//
// Reference formulas: head norm crates/xrt-models/src/llama.rs:1025-1040 (val * inv_rms * w);
// rotation crates/xrt-kernels/src/cpu/rope.rs:59-89: angle = pos * scale / theta_i, pairs
// (i, i + rope_dim/2), d[i] = a cos - b sin, d[i + half] = a sin + b cos; elements beyond
// rope_dim stay. Norm, angle, sine, cosine and rotation are float32.
//
// Two kernels. The vector kernel takes the usual case (the rotation spans the whole head, and
// the head size is 16 bytes times a power of two, twice): the lanes of a head each hold 16 bytes
// of its lower and of its upper half, which are each other's partners in the rotation, so a
// head is read and written in 16-byte pieces and the norm's sum is a few lane exchanges. When a
// step brings many tokens, the values go to their transposed cache blocks through workgroups of
// their own, which turn tiles of 64 tokens in LDS so that writes to the cache are whole lines.
// Where a key or a value lies inside its block: cache_layout.h.
// A projection that was split along k comes as the float32 sums of its parts (AT_ONCE > 0): the vector kernel then adds
// them, in order, and rounds them to bfloat16 as the kernel that adds them alone does, before it goes on as ever.
// The general kernel (one wavefront per (token, head), any even head size and rotation width)
// takes the rest. A token with a negative slot is padding and is not cached. Per head, all
// kernels use the same formulas in the same order; only the order of the norm's sum differs,
// and which kernel a model takes depends on its sizes alone, never on the step.
#include "cache_layout.h"
#include "xrt_hip.h"

namespace {

constexpr int MAX_HEAD_DIM = 512;
constexpr int WAVES = 4;

template <typename T, typename TW>
__global__ void __launch_bounds__(WAVES * XRT_WAVE) qkv_prepare_kernel(
    T* __restrict__ qkv, int items, int n_heads, int n_kv_heads, int head_dim,
    const int* __restrict__ positions, const int* __restrict__ slots,
    const TW* __restrict__ q_norm, const TW* __restrict__ k_norm, float norm_eps,
    const float* __restrict__ rope_theta, int rope_dim, float rope_scale,
    T* __restrict__ k_cache, T* __restrict__ v_cache, const int* __restrict__ block_table,
    int table_stride, int n_blocks) {
    __shared__ float buffer[WAVES][MAX_HEAD_DIM];
    const int wave = threadIdx.x / XRT_WAVE, lane = threadIdx.x % XRT_WAVE;
    const long item = (long)blockIdx.x * WAVES + wave;
    if (item >= items) return;                      // whole wave leaves together; no block barrier below
    const int heads_total = n_heads + 2 * n_kv_heads;
    const int token = (int)(item / heads_total), head = (int)(item % heads_total);
    const bool is_q = head < n_heads, is_k = !is_q && head < n_heads + n_kv_heads, is_v = !is_q && !is_k;
    T* row = qkv + (long)token * heads_total * head_dim + (long)head * head_dim;
    float* x = buffer[wave];
    const int pos = positions[token];

    long cache_base = -1;                           // element offset of this head's block in the cache
    if ((is_k || is_v) && k_cache != nullptr) {
        const int slot = slots[token];
        if (slot >= 0) {
            const int block = block_table[(long)slot * table_stride + pos / XRT_BLOCK_TOKENS];
            if (block >= 0 && block < n_blocks) {
                const int kv_head = head - n_heads - (is_v ? n_kv_heads : 0);
                cache_base = ((long)block * n_kv_heads + kv_head) * XRT_BLOCK_TOKENS * head_dim;
            }
        }
    }
    const int within = pos % XRT_BLOCK_TOKENS;

    if (is_v) {
        if (cache_base >= 0)
            for (int e = lane; e < head_dim; e += XRT_WAVE)
                v_cache[cache_base + cache_value_offset(e, within, head_dim)] = row[e];
        return;
    }

    float sum_sq = 0.f;
    for (int e = lane; e < head_dim; e += XRT_WAVE) {
        const float v = to_float(row[e]);
        x[e] = v;
        sum_sq = fmaf(v, v, sum_sq);
    }
    const TW* norm = is_q ? q_norm : k_norm;
    if (norm != nullptr) {
        sum_sq = wave_sum(sum_sq);
        const float inv_rms = 1.0f / sqrtf(sum_sq / (float)head_dim + norm_eps);
        for (int e = lane; e < head_dim; e += XRT_WAVE) x[e] = x[e] * inv_rms * to_float(norm[e]);
    }
    wave_sync();
    if (rope_theta != nullptr) {
        const int half = rope_dim / 2;
        for (int i = lane; i < half; i += XRT_WAVE) {
            const float angle = (float)pos * rope_scale / rope_theta[i];
            float sine, cosine;
            sincosf(angle, &sine, &cosine);
            const float a = x[i], b = x[i + half];
            x[i] = a * cosine - b * sine;
            x[i + half] = a * sine + b * cosine;
        }
    }
    wave_sync();
    for (int e = lane; e < head_dim; e += XRT_WAVE) {
        const T value = from_float<T>(x[e]);
        row[e] = value;
        if (is_k && cache_base >= 0) k_cache[cache_base + cache_key_offset(within, e, head_dim)] = value;
    }
}


template <typename T, int N> struct alignas(sizeof(T) * N) Pack { T e[N]; };

// The parts of a projection split along k: part p of element i at values[p * stride + i]. splits 0: there are none.
struct QkvParts { const float* values; long stride; int splits; };

// PIECES pieces of 16 bytes of a row of q/k/v, `apart` elements from one another; `at` counts elements from the first row's first. AT_ONCE 0: as they lie in
// qkv. Else the parts' sums: AT_ONCE parts of all pieces are asked for at once (those beyond the last: that one again, not added), then added in order.
// What is asked for stays within a turn: kept across turns (and across the angles, asked for ahead of them) it took a wavefront 154 registers
// instead of 58, 74 or 90 (2, 3 or 4 at once), three wavefronts a SIMD instead of eight, six or five. Parts just written, microseconds, so / kept across / piece by
// piece with a branch around every part: 333 tokens of 32 heads of 128 on 8 in three parts 8.2 / 9.1 / 8.2, in two 8.3 / 9.8 / 8.8; 100 tokens of 32 heads of 64 on 8 in
// four 4.8 / 4.9 / 5.4. 17 to 160 tokens of four such shapes in 2 to 16 parts 0.87 / 0.93 / 1, 200 to 789 tokens 0.98 / 1.09 / 1.
template <int AT_ONCE, int PIECES, typename T>
__device__ __forceinline__ void read_qkv(const T* qkv, const QkvParts& parts, long at, long apart, Pack<T, 16 / (int)sizeof(T)> (&out)[PIECES]) {
    constexpr int VEC = 16 / (int)sizeof(T);
    if constexpr (AT_ONCE == 0) {
#pragma unroll
        for (int i = 0; i < PIECES; ++i) out[i] = *reinterpret_cast<const Pack<T, VEC>*>(qkv + at + i * apart);
    } else {
        static_assert(sizeof(T) == 2, "parts are rounded to bfloat16");
        typedef float4 Asked[AT_ONCE][PIECES][2];
        auto ask = [&](int p0, Asked& asked) {
#pragma unroll
            for (int u = 0; u < AT_ONCE; ++u) {
                const float* from = parts.values + min(p0 + u, parts.splits - 1) * parts.stride + at;
#pragma unroll
                for (int i = 0; i < PIECES; ++i)
#pragma unroll
                    for (int q = 0; q < 2; ++q) asked[u][i][q] = *reinterpret_cast<const float4*>(from + i * apart + 4 * q);
            }
        };
        float sum[PIECES][VEC] = {};
        auto add = [&](int p0, const Asked& asked) {
#pragma unroll
            for (int u = 0; u < AT_ONCE; ++u) {
                const bool there = p0 + u < parts.splits;
#pragma unroll
                for (int i = 0; i < PIECES; ++i)
#pragma unroll
                    for (int q = 0; q < 2; ++q) {
                        const float4 part = asked[u][i][q];
                        float* of = sum[i] + 4 * q;
                        of[0] = there ? of[0] + part.x : of[0];
                        of[1] = there ? of[1] + part.y : of[1];
                        of[2] = there ? of[2] + part.z : of[2];
                        of[3] = there ? of[3] + part.w : of[3];
                    }
            }
        };
        Asked first;                                           // (a turn of its own: nothing has been added up yet, 16 registers less)
        ask(0, first);
        add(0, first);
        for (int p0 = AT_ONCE; p0 < parts.splits; p0 += AT_ONCE) {
            __builtin_amdgcn_sched_barrier(0);
            Asked more;
            ask(p0, more);
            __builtin_amdgcn_sched_barrier(0);
            add(p0, more);
        }
#pragma unroll
        for (int i = 0; i < PIECES; ++i)
#pragma unroll
            for (int e = 0; e < VEC; ++e) out[i].e[e] = from_float<T>(sum[i][e]);
    }
}

// 32 dims of the values of 64 consecutive tokens of a step and one key/value head: read row by row (a piece a thread), turned in
// LDS, and written so that a store instruction of a wavefront takes 8 tokens of 8 dims: where the
// tokens follow each other in a sequence these are the eight pieces of one line of the cache block
// (cache_layout.h). Tokens of different sequences or blocks may share a tile: every token has its
// own block.
constexpr int TILE_DIMS = 32;
// A store step reads 8 tokens (rows) x 8 dims: with rows of 40 elements the 8 rows start at banks 0, 20, 40, .. (bfloat16) or
// 0, 40, 80, .. (float32) of the 64, and the step's 32 or 64 words lie in as many banks.
template <typename T> struct ValueTile {
    T tile[XRT_WAVE][TILE_DIMS + 8];
    long bases[XRT_WAVE];                                             // of the tile's tokens: their block (-1: none) ...
    int withins[XRT_WAVE];                                            // ... and their place in it
};
template <typename T, int AT_ONCE>
__device__ __forceinline__ void write_values(
    ValueTile<T>& shared, int first, int kv_head, int d0, T* __restrict__ qkv, const QkvParts& parts, int tokens, int n_heads, int n_kv_heads, int head_dim,
    const int* __restrict__ positions, const int* __restrict__ slots, T* __restrict__ v_cache,
    const int* __restrict__ block_table, int table_stride, int n_blocks) {
    const int wave = threadIdx.x / XRT_WAVE, lane = threadIdx.x % XRT_WAVE;
    const int heads_total = n_heads + 2 * n_kv_heads;
    if (wave == 0) {
        const int token = first + lane;
        long cache_base = -1;
        int within = 0;
        if (token < tokens) {
            const int pos = positions[token];
            cache_base = cache_block_base(block_table, table_stride, n_blocks, slots[token], pos, n_kv_heads, kv_head, head_dim);
            within = pos % XRT_BLOCK_TOKENS;
        }
        shared.bases[lane] = cache_base;
        shared.withins[lane] = within;
    }
    const long source = (long)(n_heads + n_kv_heads + kv_head) * head_dim;
    constexpr int VEC = 16 / (int)sizeof(T);                  // the launcher sends only head sizes that are multiples of this
    const int dims = min(TILE_DIMS, head_dim - d0);
    const int pieces = dims / VEC;                            // 16-byte pieces per row
    for (int i = threadIdx.x; i < XRT_WAVE * pieces; i += WAVES * XRT_WAVE) {
        const int r = i / pieces, d = (i % pieces) * VEC;
        const long from = min(first + r, tokens - 1);         // rows past the end repeat the last one; nobody writes them to the cache
        const long at = source + from * heads_total * head_dim + d0 + d;
        Pack<T, VEC> piece[1];
        read_qkv<AT_ONCE>(qkv, parts, at, 0, piece);
        if constexpr (AT_ONCE > 0) if (first + r < tokens) *reinterpret_cast<Pack<T, VEC>*>(qkv + at) = piece[0];
        *reinterpret_cast<Pack<T, VEC>*>(&shared.tile[r][d]) = piece[0];
    }
    __syncthreads();
    // a store of a wavefront: tokens 8 g .. 8 g + 7 of the tile (lane % 8), dims 8 h .. 8 h + 7 (lane / 8);
    // a wavefront keeps its tokens while it walks the dims
    for (int g = wave; g < XRT_WAVE / 8; g += WAVES) {
        const int token = g * 8 + lane % 8;
        const long cache_base = shared.bases[token];
        const int within = shared.withins[token];
        if (cache_base < 0) continue;
#pragma unroll 4
        for (int d = lane / 8; d < dims; d += 8)
            v_cache[cache_base + cache_value_offset(d0 + d, within, head_dim)] = shared.tile[token][d];
    }
}

// The first value_tiles * n_kv_heads * (pieces of 32 dims) workgroups turn values (none of them: the others write the values themselves); then
// come `chunks` workgroups per token. LANES lanes per head; head_dim = 2 * LANES * VEC with VEC elements in
// 16 bytes. Sine and cosine of the token's angles are worked out once, into LDS, and serve all
// the workgroup's heads.
// One launch for both: as kernels of their own, values after heads, they took 11.5 + 6.1 us (2048 tokens, 32 heads of 128 on 8) and 3.3 + 4.1
// (100 tokens, 32 heads of 64 on 8).
template <typename T, typename TW, int LANES, int AT_ONCE>
__global__ void __launch_bounds__(WAVES * XRT_WAVE) qkv_prepare_vector_kernel(
    T* __restrict__ qkv, const QkvParts parts, int tokens, int n_heads, int n_kv_heads,
    const int* __restrict__ positions, const int* __restrict__ slots,
    const TW* __restrict__ q_norm, const TW* __restrict__ k_norm, float norm_eps,
    const float* __restrict__ rope_theta, float rope_scale,
    T* __restrict__ k_cache, T* __restrict__ v_cache, const int* __restrict__ block_table,
    int table_stride, int n_blocks, int value_tiles, int chunks) {
    constexpr int VEC = 16 / (int)sizeof(T);
    constexpr int HALF = LANES * VEC, HEAD = 2 * HALF;
    constexpr int HEADS_PER_WAVE = XRT_WAVE / LANES;
    __shared__ __attribute__((aligned(16))) union { struct { float cosines[HALF], sines[HALF]; } angles; ValueTile<T> values; } shared;
    constexpr int PIECES = (HEAD + TILE_DIMS - 1) / TILE_DIMS;
    const int value_blocks = value_tiles * n_kv_heads * PIECES;
    if ((int)blockIdx.x < value_blocks) {
        write_values<T, AT_ONCE>(shared.values, (int)blockIdx.x / PIECES % value_tiles * XRT_WAVE, (int)blockIdx.x / PIECES / value_tiles,
                               (int)blockIdx.x % PIECES * TILE_DIMS, qkv, parts, tokens, n_heads, n_kv_heads, HEAD, positions, slots, v_cache, block_table, table_stride, n_blocks);
        return;
    }
    float* cosines = shared.angles.cosines;
    float* sines = shared.angles.sines;
    const int wave = threadIdx.x / XRT_WAVE, lane = threadIdx.x % XRT_WAVE;
    const int item = (int)blockIdx.x - value_blocks, chunks_here = AT_ONCE > 0 ? chunks : 1;      // (a division less where it is known)
    const int token = item / chunks_here, chunk = item % chunks_here;
    const int at = (lane % LANES) * VEC;           // this lane's elements: at.. in the lower half, HALF + at.. in the upper
    const int heads_total = n_heads + 2 * n_kv_heads;
    const int heads_here = value_blocks == 0 ? heads_total : n_heads + n_kv_heads;     // value heads come last
    const int pos = positions[token];
    const int slot = slots[token];
    float theta = 1.f;
    if constexpr (AT_ONCE > 0) {                   // (asked for beside the position, not behind it: 333 tokens of 32 heads of 128 on 8, three parts, 8.4 -> 8.1 us in a model)
        if (rope_theta != nullptr) theta = rope_theta[min((int)threadIdx.x, HALF - 1)];
        __builtin_amdgcn_sched_barrier(0);
    }
    if (rope_theta != nullptr) {
        for (int i = threadIdx.x; i < HALF; i += WAVES * XRT_WAVE) {
            const float angle = (float)pos * rope_scale / (AT_ONCE > 0 && i < WAVES * XRT_WAVE ? theta : rope_theta[i]);
            sincosf(angle, &sines[i], &cosines[i]);
        }
    }
    __syncthreads();
    const int within = pos % XRT_BLOCK_TOKENS;
    // (with parts the chunks are as many as leave no workgroup a second turn)
    for (int head = (chunk * WAVES + wave) * HEADS_PER_WAVE + lane / LANES; head < heads_here; head = AT_ONCE > 0 ? heads_here : head + WAVES * HEADS_PER_WAVE) {
        // lanes of one head stay together: the exchanges below are within a head
        const bool is_q = head < n_heads, is_v = head >= n_heads + n_kv_heads, is_k = !is_q && !is_v;
        const long row_at = ((long)token * heads_total + head) * HEAD;
        T* row = qkv + row_at;
        Pack<T, VEC> both[2];
        read_qkv<AT_ONCE>(qkv, parts, row_at + at, HALF, both);
        const Pack<T, VEC> lower = both[0], upper = both[1];
        long cache_base = -1;
        if (!is_q && k_cache != nullptr)
            cache_base = cache_block_base(block_table, table_stride, n_blocks, slot, pos, n_kv_heads,
                                          head - n_heads - (is_v ? n_kv_heads : 0), HEAD);
        if (is_v) {
            if constexpr (AT_ONCE > 0) {
                *reinterpret_cast<Pack<T, VEC>*>(row + at) = lower;
                *reinterpret_cast<Pack<T, VEC>*>(row + HALF + at) = upper;
            }
            if (cache_base >= 0) {
#pragma unroll
                for (int e = 0; e < VEC; ++e) {
                    v_cache[cache_base + cache_value_offset(at + e, within, HEAD)] = lower.e[e];
                    v_cache[cache_base + cache_value_offset(HALF + at + e, within, HEAD)] = upper.e[e];
                }
            }
            continue;
        }
        float a[VEC], b[VEC];
        float sum_sq = 0.f;
#pragma unroll
        for (int e = 0; e < VEC; ++e) { a[e] = to_float(lower.e[e]); sum_sq = fmaf(a[e], a[e], sum_sq); }
#pragma unroll
        for (int e = 0; e < VEC; ++e) { b[e] = to_float(upper.e[e]); sum_sq = fmaf(b[e], b[e], sum_sq); }
        const TW* norm = is_q ? q_norm : k_norm;
        if (norm != nullptr) {
#pragma unroll
            for (int offset = LANES / 2; offset > 0; offset >>= 1) sum_sq += __shfl_xor(sum_sq, offset, XRT_WAVE);
            const float inv_rms = 1.0f / sqrtf(sum_sq / (float)HEAD + norm_eps);
#pragma unroll
            for (int e = 0; e < VEC; ++e) {
                a[e] = a[e] * inv_rms * to_float(norm[at + e]);
                b[e] = b[e] * inv_rms * to_float(norm[HALF + at + e]);
            }
        }
        if (rope_theta != nullptr) {
#pragma unroll
            for (int e = 0; e < VEC; ++e) {
                const float sine = sines[at + e], cosine = cosines[at + e];
                const float lo = a[e], hi = b[e];
                a[e] = lo * cosine - hi * sine;
                b[e] = lo * sine + hi * cosine;
            }
        }
        Pack<T, VEC> out_lower, out_upper;
#pragma unroll
        for (int e = 0; e < VEC; ++e) { out_lower.e[e] = from_float<T>(a[e]); out_upper.e[e] = from_float<T>(b[e]); }
        *reinterpret_cast<Pack<T, VEC>*>(row + at) = out_lower;
        *reinterpret_cast<Pack<T, VEC>*>(row + HALF + at) = out_upper;
        if (is_k && cache_base >= 0) {
            T* dst = k_cache + cache_base;                  // (16 bytes from a multiple of 16 bytes stay together in the cache's order)
            *reinterpret_cast<Pack<T, VEC>*>(dst + cache_key_offset(within, at, HEAD)) = out_lower;
            *reinterpret_cast<Pack<T, VEC>*>(dst + cache_key_offset(within, HALF + at, HEAD)) = out_upper;
        }
    }
}

__global__ void __launch_bounds__(256) rope_table_kernel(const float* __restrict__ rope_theta, int half, float rope_scale,
                                                         long entries, float2* __restrict__ table) {
    const long index = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (index >= entries) return;
    const int pos = (int)(index / half), i = (int)(index % half);
    const float angle = (float)pos * rope_scale / rope_theta[i];       // as in the kernels above
    float sine, cosine;
    sincosf(angle, &sine, &cosine);
    table[index] = make_float2(cosine, sine);
}

}  // namespace

extern "C" int xrt_rope_table(const float* rope_theta, int rope_dim, float rope_scale, int positions, float* table, void* stream) {
    XRT_REQUIRE(rope_theta && table && rope_dim > 0 && rope_dim % 2 == 0 && positions > 0 && (uintptr_t)table % 8 == 0,
                "rope_table: a rotation over an even number of dims, at least one position, a table aligned to 8 bytes");
    const long entries = (long)positions * (rope_dim / 2);
    rope_table_kernel<<<(unsigned)((entries + 255) / 256), 256, 0, (hipStream_t)stream>>>(rope_theta, rope_dim / 2, rope_scale, entries, (float2*)table);
    XRT_LAUNCH_CHECK("rope_table");
    return 0;
}

// What the vector kernel takes: rotation over the whole head (or none), 16-byte pieces, a power of two of lanes per head.
static int vector_lanes(const void* qkv, int dtype, int head_dim, const float* rope_theta, int rope_dim, const void* k_cache) {
    const int vec = dtype == XRT_F32 ? 4 : 8;
    const int lanes = head_dim % (2 * vec) == 0 ? head_dim / (2 * vec) : 0;
    return lanes >= 1 && lanes <= XRT_WAVE && (lanes & (lanes - 1)) == 0 && (rope_theta == nullptr || rope_dim == head_dim) &&
           (uintptr_t)qkv % 16 == 0 && (k_cache == nullptr || (uintptr_t)k_cache % 16 == 0) ? lanes : 0;
}

// Whether xrt_qkv_prepare_parts takes the sums of a projection's parts (bfloat16 results).
bool xrt_qkv_prepare_takes_parts(const void* qkv, const float* parts, int head_dim, const float* rope_theta, int rope_dim, const void* k_cache) {
    return (uintptr_t)parts % 16 == 0 && vector_lanes(qkv, XRT_BF16, head_dim, rope_theta, rope_dim, k_cache) > 0;
}

static int prepare(void* qkv, const QkvParts& parts, int dtype, int tokens, int n_heads, int n_kv_heads, int head_dim,
                   const int* positions, const int* slots, const void* q_norm, const void* k_norm,
                   int norm_dtype, float norm_eps, const float* rope_theta, int rope_dim,
                   float rope_scale, void* k_cache, void* v_cache, const int* block_table,
                   int table_stride, int n_blocks, int longest_run, void* stream) {
    XRT_REQUIRE(tokens >= 0 && n_heads > 0 && n_kv_heads > 0, "qkv_prepare: bad head counts %d/%d", n_heads, n_kv_heads);
    XRT_REQUIRE(head_dim > 0 && head_dim % 2 == 0 && head_dim <= MAX_HEAD_DIM,
                "qkv_prepare: head_dim %d must be even and at most %d", head_dim, MAX_HEAD_DIM);
    XRT_REQUIRE(dtype == XRT_F32 || dtype == XRT_BF16, "qkv_prepare: unknown dtype %d", dtype);
    XRT_REQUIRE(norm_dtype == XRT_F32 || norm_dtype == XRT_BF16, "qkv_prepare: unknown norm dtype %d", norm_dtype);
    XRT_REQUIRE(rope_theta == nullptr || (rope_dim > 0 && rope_dim % 2 == 0 && rope_dim <= head_dim),
                "qkv_prepare: rope_dim %d must be even and at most head_dim %d", rope_dim, head_dim);
    XRT_REQUIRE((k_cache == nullptr) == (v_cache == nullptr), "qkv_prepare: key and value cache come together");
    XRT_REQUIRE(k_cache == nullptr || (block_table != nullptr && table_stride > 0 && n_blocks > 0 && slots != nullptr),
                "qkv_prepare: a cache write needs slots and a block table");
    XRT_REQUIRE(positions != nullptr, "qkv_prepare: positions missing");
    if (tokens == 0) return 0;
    const long items = (long)tokens * (n_heads + 2 * n_kv_heads);
    hipStream_t s = (hipStream_t)stream;
    const int lanes = vector_lanes(qkv, dtype, head_dim, rope_theta, rope_dim, k_cache);
    if (lanes > 0) {
        // sequences that bring many tokens: their values go through the workgroups that turn them;
        // otherwise element by element from those that do the heads
        const bool values_apart = v_cache != nullptr && longest_run >= XRT_QKV_VALUES_APART;
        const int value_tiles = values_apart ? (tokens + XRT_WAVE - 1) / XRT_WAVE : 0;
        // a workgroup per token, which walks the heads; with parts, whose sums have a long way, as many as the heads fill
        const int heads = n_heads + (values_apart ? 1 : 2) * n_kv_heads, heads_at_once = WAVES * (XRT_WAVE / lanes);
        const int chunks = parts.splits > 0 ? (heads + heads_at_once - 1) / heads_at_once : 1;
        const long blocks = (long)value_tiles * n_kv_heads * ((head_dim + TILE_DIMS - 1) / TILE_DIMS) + (long)tokens * chunks;
        XRT_REQUIRE(blocks < (1L << 31), "qkv_prepare: too many workgroups");
        const unsigned grid = (unsigned)blocks;
#define XRT_VEC(T, TW, L, AT_ONCE)                                                                           \
    qkv_prepare_vector_kernel<T, TW, L, AT_ONCE><<<grid, WAVES * XRT_WAVE, 0, s>>>(                          \
        (T*)qkv, parts, tokens, n_heads, n_kv_heads, positions, slots, (const TW*)q_norm, (const TW*)k_norm, \
        norm_eps, rope_theta, rope_scale, (T*)k_cache, (T*)v_cache, block_table, table_stride, n_blocks,   \
        value_tiles, chunks)
#define XRT_VEC_LANES(T, TW, AT_ONCE)                                                                      \
    switch (lanes) {                                                                                       \
        case 1: XRT_VEC(T, TW, 1, AT_ONCE); break;                                                           \
        case 2: XRT_VEC(T, TW, 2, AT_ONCE); break;                                                           \
        case 4: XRT_VEC(T, TW, 4, AT_ONCE); break;                                                           \
        case 8: XRT_VEC(T, TW, 8, AT_ONCE); break;                                                           \
        case 16: XRT_VEC(T, TW, 16, AT_ONCE); break;                                                         \
        case 32: XRT_VEC(T, TW, 32, AT_ONCE); break;                                                         \
        default: XRT_VEC(T, TW, 64, AT_ONCE); break;                                                         \
    }
// (a step's parts all in as few turns as four at once make, evenly)
#define XRT_VEC_PARTS(TW)                                                                                  \
    if (at_once <= 2) { XRT_VEC_LANES(bf16, TW, 2) }                                                       \
    else if (at_once == 3) { XRT_VEC_LANES(bf16, TW, 3) }                                                  \
    else { XRT_VEC_LANES(bf16, TW, 4) }
        if (parts.splits > 0) {
            const int turns = (parts.splits + 3) / 4, at_once = (parts.splits + turns - 1) / turns;
            XRT_REQUIRE(dtype == XRT_BF16, "qkv_prepare: the parts of a projection become bfloat16");
            if (norm_dtype == XRT_F32) { XRT_VEC_PARTS(float) }
            else { XRT_VEC_PARTS(bf16) }
        } else if (dtype == XRT_F32 && norm_dtype == XRT_F32) { XRT_VEC_LANES(float, float, 0) }
        else if (dtype == XRT_F32) { XRT_VEC_LANES(float, bf16, 0) }
        else if (norm_dtype == XRT_F32) { XRT_VEC_LANES(bf16, float, 0) }
        else { XRT_VEC_LANES(bf16, bf16, 0) }
#undef XRT_VEC_PARTS
#undef XRT_VEC_LANES
#undef XRT_VEC
        XRT_LAUNCH_CHECK("qkv_prepare");
        return 0;
    }
    XRT_REQUIRE(parts.splits == 0, "qkv_prepare: heads of %d dims take no parts of a projection", head_dim);
    const unsigned grid = (unsigned)((items + WAVES - 1) / WAVES);
#define XRT_PREP(T, TW)                                                                                   \
    qkv_prepare_kernel<T, TW><<<grid, WAVES * XRT_WAVE, 0, s>>>(                                          \
        (T*)qkv, (int)items, n_heads, n_kv_heads, head_dim, positions, slots, (const TW*)q_norm,          \
        (const TW*)k_norm, norm_eps, rope_theta, rope_dim, rope_scale, (T*)k_cache, (T*)v_cache,          \
        block_table, table_stride, n_blocks)
    if (dtype == XRT_F32 && norm_dtype == XRT_F32) XRT_PREP(float, float);
    else if (dtype == XRT_F32) XRT_PREP(float, bf16);
    else if (norm_dtype == XRT_F32) XRT_PREP(bf16, float);
    else XRT_PREP(bf16, bf16);
#undef XRT_PREP
    XRT_LAUNCH_CHECK("qkv_prepare");
    return 0;
}

extern "C" int xrt_qkv_prepare(void* qkv, int dtype, int tokens, int n_heads, int n_kv_heads, int head_dim,
                               const int* positions, const int* slots, const void* q_norm, const void* k_norm,
                               int norm_dtype, float norm_eps, const float* rope_theta, int rope_dim,
                               float rope_scale, void* k_cache, void* v_cache, const int* block_table,
                               int table_stride, int n_blocks, int longest_run, void* stream) {
    return prepare(qkv, QkvParts{nullptr, 0, 0}, dtype, tokens, n_heads, n_kv_heads, head_dim, positions, slots, q_norm, k_norm, norm_dtype, norm_eps,
                   rope_theta, rope_dim, rope_scale, k_cache, v_cache, block_table, table_stride, n_blocks, longest_run, stream);
}

// The same for a bfloat16 projection that comes as `splits` parts of tokens x (all heads' dims) float32 sums, one after another.
int xrt_qkv_prepare_parts(const float* parts, int splits, void* qkv, int tokens, int n_heads, int n_kv_heads, int head_dim,
                          const int* positions, const int* slots, const void* q_norm, const void* k_norm,
                          int norm_dtype, float norm_eps, const float* rope_theta, int rope_dim,
                          float rope_scale, void* k_cache, void* v_cache, const int* block_table,
                          int table_stride, int n_blocks, int longest_run, void* stream) {
    XRT_REQUIRE(parts != nullptr && splits > 0, "qkv_prepare: no parts");
    return prepare(qkv, QkvParts{parts, (long)tokens * (n_heads + 2 * n_kv_heads) * head_dim, splits}, XRT_BF16, tokens, n_heads, n_kv_heads, head_dim,
                   positions, slots, q_norm, k_norm, norm_dtype, norm_eps, rope_theta, rope_dim, rope_scale, k_cache, v_cache, block_table, table_stride,
                   n_blocks, longest_run, stream);
}
