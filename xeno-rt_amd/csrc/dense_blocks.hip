// The layers of a plain dense decoder (pre-norm blocks of grouped-query attention and a gated feed-forward) launched from one call.
//
// A layer is 5 to 14 kernels. Launched one by one through the Python classes, with their checks, a kernel costs the host 8 to 10 us, and a prompt of up to
// some hundred tokens through a small model waited for the host most of the time. Here the same launches, in the same order and with the same operands,
// cost 3 us each. Prompts of 5 / 17 / 64 / 100 / 200 / 400 tokens: 28 layers of width 1024 2426 / 3017 / 3116 / 3058 / 3039 / 3265 -> 983 / 1529 / 1973 / 2418 / 2617 /
// 3196 us, 16 layers of width 2048 1340 / 1672 / 1679 / 1842 / 1864 / 2354 -> 828 / 1087 / 1257 / 1586 / 1843 / 2280, a tiny model's 306 -> 202.
// What each product, norm and attention takes is asked of the functions that the single calls ask (xrt_hip.h). Nothing is kept
// between calls: the caller describes the layers' matrices, vectors and caches each time.
//
// Memory: one piece, given by the caller, whose size the call itself says beforehand (arena null). A layer's buffers lie where the layer's before lay (the
// stream's order keeps them apart); what a layer hands to the next lies in two places that take turns.
#include <algorithm>

#include "common.h"
#include "xrt_hip.h"

bool xrt_attention_decode_accepts(int head_dim);

namespace {

struct Arena {
    char* base;
    long at = 0, most = 0;
    const bool plan;
    explicit Arena(void* memory) : base((char*)memory), plan(memory == nullptr) {}
    void* take(long bytes) {                                    // (a plan's pointers are never followed; they are aligned like the real ones)
        char* p = (plan ? (char*)256 : base) + at;
        at += (bytes + 255) / 256 * 256;
        most = max(most, at);
        return p;
    }
};

struct Norm { const void* gain; int dtype; float eps; };

// rows on their way through a norm: normed, or (squares) still to be divided by their rms by the product that reads them
struct Rows {
    const void* values = nullptr;
    const float* squares = nullptr;
    int tiles = 0;
    float eps = 0.f;
};
// where a product may put such rows
struct Room { void* values; float* squares; };

// Whether the attention of a step's `rows` wanted rows alone, as a step in which every row is a sequence with one token, takes less than that of all its tokens.
// The decode kernel reads a row's keys for that row only, the kernel for prompts shares them among the rows of a tile. In nanoseconds, for keys of the step's
// average position: a row of the one costs 200 a thousand keys of 8 heads of 128 and somewhat more where they lie beyond the caches, a row of the other 16 a thousand keys of 32 query heads
// of 128, and 6000 + 2 a key once; every sequence's keys are read once either way. Fitted to 1280 steps (32 heads on 8, 16 on 8 and 64 on 8 of 128 dims, 32 on 8
// of 64; 17 to 8192 tokens of one sequence or four behind 0 to 16000; a row of 4 to the last alone): 0.6 % off the better of the two on
// average, where the wanted rows alone at all times are 22 % off. 32 heads of 128 on 8: 2048 of 8192 tokens 2121 us alone, 671 all (behind 16000
// 14091 and 2581), 256 of them 260 (1609); 41 of 333 behind 4000 46 and 55, 83 of them 91.
// Whole steps, two layers, before any of this, with the wanted rows alone at all times, and by this rule: 8B sizes, 2048 of 8192 tokens 8151, 8116, 6601 us; 250 of 1000 behind
// 8000 1555, 2002, 1341; Qwen3-0.6B sizes, 512 of 2048 behind 8000 940, 1903, 879; float32, Llama-3.2-1B sizes, 250 of 1000 behind 4000 13646, 5135, 4232.
// float32, to the same bits: where the matrix cores take the step, a thousand keys are 240 us to a wavefront of the general kernel that goes through them by itself,
// which it does with more (token, head) pairs than the kernel of the many takes from; below that it shares them out (2048 tokens, 32 heads of 64 on 8: 428 us all, 64 rows alone 242, 128 482).
bool wanted_alone(const xrt_dense_step& s, const xrt_dense_layer& l, const void* qkv, int rows) {
    if (s.dtype == XRT_F32)
        return (long)rows * l.n_heads <= 8L * XRT_COMPUTE_UNITS ||
               !xrt_attention_float_prompts_accepts(qkv, s.tokens, l.n_heads, l.n_kv_heads, l.head_dim, l.k_cache, l.v_cache, qkv, s.fewest, s.max_context);
    if (!xrt_attention_decode_accepts(l.head_dim)) return true;                // (the general kernel, a token at a time either way)
    if (rows > XRT_GRID_ROWS) return false;
    const double keys = std::max(1.0, s.max_context - 0.5 * s.max_count), row = (200 + 0.008 * keys) * (l.n_kv_heads * l.head_dim / 1024.0) * keys / 1000;
    return row * (rows - s.n_seqs) <= 6000 + 2 * keys + 16 * (l.n_heads * l.head_dim / 4096.0) * keys / 1000 * s.tokens;
}

struct Step {
    const xrt_dense_step& s;
    Arena& arena;
    long element;
    Step(const xrt_dense_step& step, Arena& memory) : s(step), arena(memory), element(step.dtype == XRT_F32 ? 4 : 2) {}
    long squares_bytes() const { return ((long)s.hidden / 8 + 1) * XRT_SQUARES_STRIDE * 4; }       // tiles of eight columns at least
    Room room() { return Room{arena.take((long)s.tokens * s.hidden * element), (float*)arena.take(squares_bytes())}; }

    int norm(const float* x, const Norm& n, int rows, void* out) {
        if (arena.plan) return 0;
        return xrt_rmsnorm(x, n.gain, n.dtype, n.eps, out, s.dtype, nullptr, rows, s.hidden, s.stream);
    }

    // out (+)= a w^T; with `then` (an accumulating product) the norm behind it, as far as the product can do it: `after` says what there is of it
    int product(const Rows& a, const xrt_dense_matrix& w, void* out, int out_dtype, int M, int N, int K, int mode, const Norm* then = nullptr,
                const Room* room = nullptr, Rows* after = nullptr) {
        const xrt_packing* packing = w.packing.kind ? &w.packing : nullptr;
        const int takes = then != nullptr && mode == 1 && N % 8 == 0 ? xrt_linear_takes_norm(a.values, w.data, packing, s.dtype, M, N, K, mode) : 0;
        xrt_linear_norm around = {};
        long need = 0;
        if (takes == 2 && a.squares == nullptr && out_dtype == XRT_F32 && (uintptr_t)out % 16 == 0 && (uintptr_t)then->gain % 16 == 0) {
            around.eps = then->eps;
            around.scaled_out = room->values; around.gain = then->gain; around.gain_dtype = then->dtype;
            *after = Rows{room->values, nullptr, 0, 0.f};
            need = xrt_linear_whole_norm_workspace(a.values, w.data, s.dtype, M, N, K, mode);
        } else {
            if (a.squares != nullptr) { around.squares_in = a.squares; around.tiles_in = a.tiles; around.width_in = K; around.eps = a.eps; }
            if (takes == 1) {
                around.scaled_out = room->values; around.squares_out = room->squares; around.gain = then->gain; around.gain_dtype = then->dtype;
                *after = Rows{room->values, room->squares, xrt_linear_norm_tiles(a.values, w.data, packing, s.dtype, M, N, K), then->eps};
                XRT_REQUIRE((long)after->tiles * XRT_SQUARES_STRIDE * 4 <= squares_bytes(), "dense blocks: %d tiles of sums of squares", after->tiles);
            }
            need = xrt_linear_workspace(a.values, w.data, s.dtype, M, N, K, mode);
        }
        const long before = arena.at;
        float* workspace = need > 0 ? (float*)arena.take(need * 4) : nullptr;
        arena.at = before;                                      // (the next kernel may have it: it starts when this one is done)
        if (arena.plan) return 0;
        if (around.squares_in != nullptr || around.scaled_out != nullptr)
            return xrt_linear_normed(a.values, w.data, packing, s.dtype, out, out_dtype, M, N, K, mode, &around, workspace, need, s.stream);
        return xrt_linear_with(a.values, w.data, packing, s.dtype, out, out_dtype, M, N, K, mode, workspace, need, s.stream);
    }

    // attention over the cache for `rows` queries in rows of `qkv`
    int attention(const xrt_dense_layer& l, const void* qkv, int rows, const int* positions, const int* slots, const int* offsets, const int* seq_slots,
                  const int* starts, int n_seqs, int max_count, int fewest, const xrt_qkv_finish* finish, void* out) {
        if (s.dtype == XRT_F32 && xrt_attention_float_prompts_accepts(qkv, rows, l.n_heads, l.n_kv_heads, l.head_dim, l.k_cache, l.v_cache, out, fewest, s.max_context)) {
            if (arena.plan) return 0;
            return xrt_attention_float_prompts(qkv, rows, l.n_heads, l.n_kv_heads, l.head_dim, l.k_cache, l.v_cache, l.block_table, l.table_stride, l.n_blocks,
                                               positions, slots, out, l.scale, fewest, s.max_context, s.stream);
        }
        const long need = xrt_attention_workspace(s.dtype, rows, l.n_heads, l.n_kv_heads, l.head_dim, 0, max_count, s.max_context);
        const long before = arena.at;
        float* workspace = need > 0 ? (float*)arena.take(need * 4) : nullptr;
        arena.at = before;
        if (arena.plan) return 0;
        if (finish != nullptr)
            return xrt_attention_finishing(qkv, s.dtype, rows, l.n_heads, l.n_kv_heads, l.head_dim, l.k_cache, l.v_cache, l.block_table, l.table_stride,
                                           l.n_blocks, positions, slots, out, l.scale, finish, s.max_context, workspace, need, s.stream);
        return xrt_attention(qkv, s.dtype, rows, l.n_heads, l.n_kv_heads, l.head_dim, l.k_cache, l.v_cache, l.block_table, l.table_stride, l.n_blocks,
                             positions, slots, out, l.scale, 0, nullptr, offsets, seq_slots, starts, n_seqs, max_count, s.max_context, workspace, need, s.stream);
    }

    // One layer. h: its first norm of x if the layer before made it (in), the next layer's (out); wanted: the last layer's, or null.
    int layer(const xrt_dense_layer& l, const xrt_dense_wanted* wanted, Rows& h, const Norm* next, const Room& handed_on) {
        const int width = (l.n_heads + 2 * l.n_kv_heads) * l.head_dim, q_width = l.n_heads * l.head_dim;
        const Norm first{l.mixer_gain, l.mixer_gain_dtype, l.mixer_eps}, second{l.ff_gain, l.ff_gain_dtype, l.ff_eps};
        float* x = s.x;
        int rows = s.tokens;
        if (h.values == nullptr) {
            void* normed = arena.take((long)rows * s.hidden * element);
            if (norm(x, first, rows, normed)) return 1;
            h = Rows{normed, nullptr, 0, 0.f};
        }
        void* qkv = arena.take((long)rows * width * element);
        // a decode step with head norms: the attention finishes q, k and v itself, where it can
        const bool finishes = wanted == nullptr && l.q_norm != nullptr && l.writable && s.dtype == XRT_BF16 && (l.rope_theta == nullptr || l.rope_table != nullptr) &&
            xrt_attention_finishes_qkv(s.dtype, l.n_heads, l.n_kv_heads, l.head_dim, 0, s.max_count, l.rope_theta ? l.rope_dim : 0, l.table_positions, s.max_context);
        xrt_qkv_finish finish = {l.q_norm, l.k_norm, l.head_norm_dtype, l.head_norm_eps, l.rope_theta ? l.head_dim : 0, l.rope_table, l.table_positions};
        if (finishes) {
            if (product(h, l.qkv, qkv, s.dtype, rows, width, s.hidden, 0)) return 1;
        } else {
            xrt_linear_norm around = {};
            if (h.squares != nullptr) { around.squares_in = h.squares; around.tiles_in = h.tiles; around.width_in = s.hidden; around.eps = h.eps; }
            const long need = xrt_linear_workspace(h.values, l.qkv.data, s.dtype, rows, width, s.hidden, 0), before = arena.at;
            float* workspace = need > 0 ? (float*)arena.take(need * 4) : nullptr;
            arena.at = before;
            if (!arena.plan &&
                xrt_linear_qkv(h.values, l.qkv.data, l.qkv.packing.kind ? &l.qkv.packing : nullptr, s.dtype, qkv, rows, s.hidden,
                               h.squares != nullptr ? &around : nullptr, l.n_heads, l.n_kv_heads, l.head_dim, s.positions, s.slots, l.q_norm, l.k_norm,
                               l.head_norm_dtype, l.head_norm_eps, l.rope_theta, l.rope_theta ? l.rope_dim : 0, l.rope_scale, l.writable ? l.k_cache : nullptr,
                               l.writable ? l.v_cache : nullptr, l.writable ? l.block_table : nullptr, l.writable ? l.table_stride : 0,
                               l.writable ? l.n_blocks : 0, s.max_count, workspace, need, s.stream))
                return 1;
        }
        if (wanted != nullptr && wanted->count == 0) return 0;
        const bool alone = wanted != nullptr && wanted_alone(s, l, qkv, wanted->count);
        void* out = nullptr;
        if (!alone) {
            out = arena.take((long)rows * q_width * element);
            if (attention(l, qkv, rows, s.positions, s.slots, s.seq_offsets, s.seq_slots, s.seq_starts, s.n_seqs, s.max_count, s.fewest, finishes ? &finish : nullptr, out))
                return 1;
        }
        if (wanted != nullptr) {
            // The rows that somebody wants go on alone: with their queries, as a step in which every row is a sequence with one token, or with what
            // the attention of all rows has made.
            rows = wanted->count;
            const void* of = alone ? qkv : out;
            const long of_stride = alone ? width * element : q_width * element;
            void* taken = arena.take(rows * of_stride);
            int* described = (int*)arena.take((3L * rows + 1) * 4);
            x = wanted->x;
            if (!arena.plan && xrt_take_rows(of, of_stride, (int)(q_width * element), taken, of_stride, s.x, s.hidden * 4, x, s.positions, s.slots,
                                             wanted->rows, rows, s.tokens, described, s.stream))
                return 1;
            out = taken;
            if (alone) {
                out = arena.take((long)rows * q_width * element);
                if (attention(l, taken, rows, described, described + rows, described + 2 * rows, described + rows, described, rows, 1, 1, nullptr, out)) return 1;
            }
        }
        const Room between = room();
        Rows middle;
        if (product(Rows{out, nullptr, 0, 0.f}, l.o, x, XRT_F32, rows, s.hidden, q_width, 1, &second, &between, &middle)) return 1;
        if (middle.values == nullptr) {
            if (norm(x, second, rows, between.values)) return 1;
            middle = Rows{between.values, nullptr, 0, 0.f};
        }
        void* act = arena.take((long)rows * l.intermediate * element);
        if (product(middle, l.gate_up, act, s.dtype, rows, l.intermediate, s.hidden, XRT_GATED(XRT_ACT_SILU))) return 1;
        h = Rows{};
        return product(Rows{act, nullptr, 0, 0.f}, l.down, x, XRT_F32, rows, s.hidden, l.intermediate, 1, next, &handed_on, &h);
    }
};

}  // namespace

extern "C" int xrt_dense_wanted_alone(const xrt_dense_layer* layer, const xrt_dense_step* step, int rows) {
    return layer == nullptr || step == nullptr || rows <= 0 ? -1 : wanted_alone(*step, *layer, nullptr, rows);
}

extern "C" long xrt_dense_blocks(const xrt_dense_layer* layers, int count, const xrt_dense_step* step, const xrt_dense_wanted* wanted, void* arena, long arena_bytes) {
    const auto refuse = [](const char* what) -> long { xrt_set_error("dense blocks: %s", what); return -1; };
    if (layers == nullptr || step == nullptr || count <= 0) return refuse("nothing to run");
    const xrt_dense_step& s = *step;
    if ((s.dtype != XRT_F32 && s.dtype != XRT_BF16) || s.tokens <= 0 || s.hidden <= 0 || s.n_seqs <= 0 || s.n_seqs > s.tokens || s.max_count <= 0 || s.max_context <= 0)
        return refuse("a step needs tokens, sequences and their lengths");
    if (!s.x || !s.positions || !s.slots || !s.seq_offsets || !s.seq_slots || !s.seq_starts) return refuse("null operand of the step");
    if (wanted != nullptr && (wanted->count < 0 || (wanted->count > 0 && (!wanted->rows || !wanted->x)))) return refuse("wanted rows without their operands");
    for (int i = 0; i < count; ++i) {
        const xrt_dense_layer& l = layers[i];
        if (!l.mixer_gain || !l.ff_gain || !l.qkv.data || !l.o.data || !l.gate_up.data || !l.down.data || !l.k_cache || !l.v_cache || !l.block_table ||
            (l.q_norm == nullptr) != (l.k_norm == nullptr))
            return refuse("null operand of a layer");
        if (l.n_heads <= 0 || l.n_kv_heads <= 0 || l.n_heads % l.n_kv_heads != 0 || l.head_dim <= 0 || l.intermediate <= 0 || l.table_stride <= 0 || l.n_blocks <= 0 ||
            (l.rope_theta != nullptr && l.rope_dim <= 0))
            return refuse("bad sizes of a layer");
        if (s.max_context > (long)l.table_stride * XRT_BLOCK_TOKENS) return refuse("a sequence exceeds the block table");
    }
    if (arena != nullptr && (uintptr_t)arena % 256 != 0) return refuse("the memory must be aligned to 256 bytes");
    Arena memory(arena);
    Step run(s, memory);
    const Room handed[2] = {run.room(), run.room()};
    const long kept = memory.at;
    if (arena != nullptr) {
        const long need = xrt_dense_blocks(layers, count, step, wanted, nullptr, 0);
        if (need < 0) return -1;
        if (arena_bytes < need) return refuse("the memory is too small");
    }
    Rows h;
    for (int i = 0; i < count; ++i) {
        memory.at = kept;
        const bool last = i + 1 == count;
        const Norm next{last ? nullptr : layers[i + 1].mixer_gain, last ? 0 : layers[i + 1].mixer_gain_dtype, last ? 0.f : layers[i + 1].mixer_eps};
        if (run.layer(layers[i], last ? wanted : nullptr, h, last ? nullptr : &next, handed[i % 2])) return -1;
    }
    return memory.most;
}
