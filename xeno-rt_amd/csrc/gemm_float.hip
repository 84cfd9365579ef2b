// Float32 products of more than 16 rows of a on the matrix cores: out[m, n] = sum_k a[m, k] * w[n, k], to the bits of the kernels of
// gemm_simple.hip. v_mfma_f32_16x16x4_f32 adds its four products to the sum one after the other, fmaf by fmaf, denormals and infinities
// included, so four of them from zero make the sum of 16 consecutive k (a chunk) as those kernels make it, and the chunks' sums are added
// up on the vector ALU in the order of k: an output has the same bits whichever kernel made it.
//
// Bound by the matrix cores, and by every vector instruction beside them: while a float32 product runs, its SIMD issues no vector
// instruction, of whichever wavefront (eight products of 512 cycles beside 128 additions of another wavefront: 1096 cycles; bfloat16
// products let most of them through). So the loop has next to none but the additions themselves, 4 for each 4 products of 32 cycles: operands
// go global -> LDS past the registers, with addresses that only scalar instructions advance, and an LDS read is a lane's own four bytes (k = 4 s +
// lane / 16 of a row), not 16 bytes that would have to be changed about. The reads of the next chunk's operands stand between the products of this
// one, a step's loads between slices of them: a wavefront alone on its SIMD (a tile to a compute unit is the rule) then waits for neither. Rows of
// LDS change their pieces of 16 bytes about by the row's number, so that the 16 rows of a block lie in all banks.
//
// Two ways to share a tile of 16 R rows of a among four wavefronts:
//   apart     each has 16 columns of its own (gated: 16 gate rows of w and the up rows of the same outputs) and walks all of k; 64 columns a tile;
//   together  all have the same 16 columns and take the chunks of k in turn; the chunks' sums meet in LDS, where every thread adds up some outputs
//             in the order of k, two steps behind the products. Four times as many tiles, for products that have few.
// Rows of a come in blocks of 16, so that a tile of 5 or 7 blocks divides what is left over: 777 rows, 2048 columns are 224 tiles of 7 blocks by
// 64, one round; in blocks of 64 by 64, as it was before, 416 tiles for 256 compute units. Before (32x32x2, operands through registers) and now,
// us, k = 2048 unless said, four matrices in turn:
//   rows of a                         17 .. 20      64           100          200          400          777
//   2048 columns                      50 -> 10      50 -> 12     50 -> 18     51 -> 26     53 -> 41     88 -> 67
//   3072 columns                      49 -> 12      50 -> 18     51 -> 25     53 -> 33     86 -> 49     121 -> 86
//   8192 gated                        50 -> 30      51 -> 40     86 -> 70     161 -> 123   271 -> 242   499 -> 427
//   2048 columns, k = 8192            184 -> 37     186 -> 44    187 -> 80    187 -> 91    189 -> 141   320 -> 232
// The last column is 63, 75, 80 and 72 % of what the matrix cores do (157 TFLOP/s), counted with the rows and columns that fill tiles up; of the compute units that have a
// tile in the last round 72, 80, 80 and 82 %. The additions alone take 11 %.
#include <type_traits>
#include <utility>
#include <cmath>
#include "common.h"
#include "xrt_hip.h"
#include "gemm_float.h"
#include "activation.h"

namespace {

enum { MODE_STORE = 0, MODE_ACCUMULATE = 1, MODE_GATED = 2 };
typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef float floatx2 __attribute__((ext_vector_type(2)));

constexpr int THREADS = 256, WAVES = 4;
constexpr int STAGES = 4;          // steps along k in LDS: the one being multiplied, the next (whose first operands are read ahead), two on their way

template <int... I, typename F>
__device__ __forceinline__ void each(std::integer_sequence<int, I...>, F f) { (f(std::integral_constant<int, I>{}), ...); }

// R: blocks of 16 rows of a in a tile.
template <int MODE, int R, bool TOGETHER>
struct Shape {
    static constexpr int C = MODE == MODE_GATED ? 2 : 1;        // blocks of 16 rows of w of a wavefront
    static constexpr int APART = TOGETHER ? 1 : WAVES;          // wavefronts side by side along the columns
    static constexpr int CHUNKS = TOGETHER ? WAVES : 2;         // chunks of 16 columns of k in a step
    static constexpr int BK = 16 * CHUNKS, PIECES = BK / 4;     // columns of k in a step, and pieces of 16 bytes of a row
    static constexpr int ROWS_A = 16 * R, ROWS_W = 16 * C * APART, OUTPUTS = 16 * APART;
    static constexpr int AT_ONCE = XRT_WAVE / PIECES;           // rows that one load instruction brings
    static constexpr int LOADS = (ROWS_A + ROWS_W) / AT_ONCE, PER_WAVE = (LOADS + WAVES - 1) / WAVES;
    static constexpr int STAGE = (ROWS_A + ROWS_W) * BK;        // floats
    static constexpr int PARTS = TOGETHER ? 2 * WAVES * R * C * 256 : 0;
    static constexpr size_t LDS = (size_t)(STAGES * STAGE + PARTS) * 4;
};

template <int MODE, int R, bool TOGETHER>
__global__ void __launch_bounds__(THREADS, 2) gemm_float_kernel(
    const float* __restrict__ a, const float* __restrict__ w, float* __restrict__ out, int M, int N, int K, int tiles_m, int activation) {
    typedef Shape<MODE, R, TOGETHER> S;
    constexpr int C = S::C;
    extern __shared__ __attribute__((aligned(16))) float lds[];
    const int tid = threadIdx.x, lane = tid % XRT_WAVE, wave = __builtin_amdgcn_readfirstlane(tid / XRT_WAVE);
    // neighbouring workgroups go to different XCDs: every XCD takes a run of tiles of its own, down the rows first, so that
    // the tiles that run there together share their w
    const int total = gridDim.x, per = total / 8;
    const int id = blockIdx.x < per * 8 ? blockIdx.x % 8 * per + blockIdx.x / 8 : blockIdx.x;
    const long m0 = (long)(id % tiles_m) * S::ROWS_A, n0 = (long)(id / tiles_m) * S::OUTPUTS;

    // ---- the loads of this wavefront: AT_ONCE rows each, the pieces of a row changed about by the row's number
    auto swap_of = [](int row) { return S::PIECES == 8 ? row / 2 % 8 : row % 16; };
    const float* from[S::PER_WAVE];
    unsigned offset[S::PER_WAVE], into[S::PER_WAVE];
#pragma unroll
    for (int i = 0; i < S::PER_WAVE; ++i) {
        const int load = min(wave + i * WAVES, S::LOADS - 1);    // (beyond the last: the last again, the same bytes to the same place)
        const int first = load * S::AT_ONCE, row = first + lane / S::PIECES;
        const int piece = (lane % S::PIECES) ^ swap_of(row);
        long within;                                             // row of the operand, from its base
        if (first < S::ROWS_A) {
            from[i] = a + m0 * K;
            within = min((long)row, (long)M - 1 - m0);
        } else {
            const int block = (first - S::ROWS_A) / 16;         // blocks of 16 rows of w: of the first wavefront, of the second ...
            const int r = (row - S::ROWS_A) % 16;
            from[i] = w + (n0 + (MODE == MODE_GATED && block % 2 == 1 ? (long)N : 0L)) * K;
            within = min((long)(MODE == MODE_GATED ? block / 2 : block) * 16 + r, (long)N - 1 - n0);
        }
        offset[i] = (unsigned)((within * K + piece * 4) * 4);
        into[i] = lds_address(lds) + first * S::BK * 4;
    }
    const int steps = (K + S::BK - 1) / S::BK;
    const int last_piece = K / 4 - (steps - 1) * S::PIECES;      // pieces of the last step that lie inside of K
    auto ask_one = [&](int i, int stage, int step) { load_to_lds(from[i] + (long)step * S::BK, offset[i], into[i] + stage * S::STAGE * 4); };
    auto ask = [&](int stage, int step) {
        if (step < steps - 1 || last_piece == S::PIECES) {
#pragma unroll
            for (int i = 0; i < S::PER_WAVE; ++i) ask_one(i, stage, step);
        } else {                                                 // beyond K: some piece inside; zeroed when it has come
#pragma unroll
            for (int i = 0; i < S::PER_WAVE; ++i) {
                const int load = min(wave + i * WAVES, S::LOADS - 1);
                const int piece = (lane % S::PIECES) ^ swap_of(load * S::AT_ONCE + lane / S::PIECES);
                load_to_lds(from[i] + (long)step * S::BK, offset[i] - (unsigned)(max(0, piece - (last_piece - 1)) * 16), into[i] + stage * S::STAGE * 4);
            }
        }
    };
    auto clear_beyond = [&](int stage) {                         // of the last step's pieces that this wavefront has asked for (and that have come)
#pragma unroll
        for (int i = 0; i < S::PER_WAVE; ++i) {
            const int load = min(wave + i * WAVES, S::LOADS - 1), first = load * S::AT_ONCE;
            const int piece = (lane % S::PIECES) ^ swap_of(first + lane / S::PIECES);
            if (piece >= last_piece) *reinterpret_cast<floatx4*>(lds + stage * S::STAGE + first * S::BK + lane * 4) = floatx4{0.f, 0.f, 0.f, 0.f};
        }
    };

    // ---- operands: of 16 columns of k, step s of the products takes 4 s + lane / 16
    const int r = lane % 16, c = lane / 16;
    struct Operands { float of_a[R][4], of_w[C][4]; };
    constexpr int PLACES = TOGETHER ? 4 : S::PIECES;
    // of piece p of row r, the same for all blocks of 16 rows; worked out once for the first half of the stages and once for the others, so
    // that what is added to it fits an instruction's 16 bits
    typedef const __attribute__((address_space(3))) float* LdsFloat;
    LdsFloat place[2][PLACES], place_w[2][PLACES];
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int p = 0; p < PLACES; ++p) {
            place[h][p] = (LdsFloat)lds + h * (STAGES / 2) * S::STAGE + r * S::BK + ((TOGETHER ? wave * 4 + p : p) ^ swap_of(r)) * 4 + c;
            place_w[h][p] = place[h][p] + S::ROWS_A * S::BK + (TOGETHER ? 0 : wave * C * 16 * S::BK);
            asm volatile("" : "+v"(place[h][p]), "+v"(place_w[h][p]));      // (kept, not worked out again in every step)
        }
    auto read_slice = [&](Operands& o, int stage, int chunk, int s) {
        const int p = TOGETHER ? s : chunk * 4 + s, h = stage / (STAGES / 2), within = stage % (STAGES / 2) * S::STAGE;
#pragma unroll
        for (int b = 0; b < C; ++b) o.of_w[b][s] = place_w[h][p][within + b * 16 * S::BK];
#pragma unroll
        for (int b = 0; b < R; ++b) o.of_a[b][s] = place[h][p][within + b * 16 * S::BK];
    };
    auto read = [&](Operands& o, int stage, int chunk) {
#pragma unroll
        for (int s = 0; s < 4; ++s) read_slice(o, stage, chunk, s);
    };
    // The products of a chunk, in four slices; among each slice's the reads of a slice of the next chunk's operands, behind it what `between` does.
    auto products = [&](const Operands& o, floatx4 (&part)[C][R], Operands& next, int next_stage, int next_chunk, auto within, auto between) {
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            __builtin_amdgcn_sched_barrier(0);
            within(s);
            read_slice(next, next_stage, next_chunk, s);
#pragma unroll
            for (int b = 0; b < R; ++b)
#pragma unroll
                for (int n = 0; n < C; ++n)
                    part[n][b] = __builtin_amdgcn_mfma_f32_16x16x4f32(o.of_w[n][s], o.of_a[b][s], s == 0 ? floatx4{0.f, 0.f, 0.f, 0.f} : part[n][b], 0, 0, 0);
#pragma unroll
            for (int i = 0; i < R * C; ++i) {
                __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                __builtin_amdgcn_sched_group_barrier(0x080, TOGETHER ? 2 : 1, 0);
            }
            __builtin_amdgcn_sched_barrier(0);
            between(s);
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    const bool wide = N % 4 == 0 && (uintptr_t)out % 16 == 0;
    // what an accumulating product adds to is asked for ahead of everything else, where it comes in whole pieces
    constexpr int V = !TOGETHER || R % 4 == 0 ? 4 : (R % 2 == 0 ? 2 : 1), GROUPS = TOGETHER ? R / V : R;     // together: a thread adds up GROUPS times V neighbouring outputs
    typedef float Some __attribute__((ext_vector_type(V)));
    auto place_of = [&](int g, long& m, long& n) {               // row and first column of the outputs of this thread
        const int element = TOGETHER ? (g * THREADS + tid) * V : 0, of_lane = TOGETHER ? element % 256 / 4 : lane;
        m = m0 + (TOGETHER ? element / 256 : g) * 16 + of_lane % 16;
        n = n0 + (TOGETHER ? 0 : wave * 16) + of_lane / 16 * 4 + (TOGETHER ? element % 4 : 0);
    };
    Some before[MODE == MODE_ACCUMULATE ? GROUPS : 1];
    if constexpr (MODE == MODE_ACCUMULATE) {
#pragma unroll
        for (int g = 0; g < GROUPS; ++g) {
            long m, n;
            place_of(g, m, n);
            if (wide && m < M && n < N) before[g] = *reinterpret_cast<const Some*>(out + m * (long)N + n);
        }
    }
    auto write = [&](auto value) {                               // value(g, e): output e of group g
#pragma unroll
        for (int g = 0; g < GROUPS; ++g) {
            long m, n;
            place_of(g, m, n);
            if (m >= M || n >= N) continue;
            float* dst = out + m * (long)N + n;
            Some made;
#pragma unroll
            for (int e = 0; e < V; ++e) made[e] = value(g, e);
            if (wide) {                                          // (N is a multiple of 4, and n of V: all of them or none)
                if constexpr (MODE == MODE_ACCUMULATE) {
#pragma unroll
                    for (int e = 0; e < V; ++e) made[e] = before[g][e] + made[e];
                }
                *reinterpret_cast<Some*>(dst) = made;
            } else {
#pragma unroll
                for (int e = 0; e < V; ++e)
                    if (n + e < N) dst[e] = MODE == MODE_ACCUMULATE ? dst[e] + made[e] : made[e];
            }
        }
    };

#pragma unroll
    for (int s = 0; s < STAGES - 1; ++s)
        if (s < steps) ask(s, s);
    // Before step t: its operands' stage and the next one have come, for every wavefront; the stage of step t - 1 has been read.
    auto arrive = [&](int t, int stage) {
        const int there = min(t + 1, steps - 1);                 // the newest step that must have come
        if (there == steps - 1 && last_piece < S::PIECES && (t + 1 == steps - 1 || (t == 0 && steps == 1))) {
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            clear_beyond(steps == 1 ? 0 : (stage + 1) % STAGES);
        }
        if (t + STAGES - 1 <= steps) wait_loads_and_barrier<(STAGES - 3) * S::PER_WAVE>();       // (all of the loads asked for: t + STAGES - 1 steps')
        else wait_loads_and_barrier<0>();
    };
    if constexpr (!TOGETHER) {
        floatx4 acc[C][R];
#pragma unroll
        for (int n = 0; n < C; ++n)
#pragma unroll
            for (int b = 0; b < R; ++b) acc[n][b] = floatx4{0.f, 0.f, 0.f, 0.f};
        auto add = [&](const floatx4 (&part)[C][R]) {
#pragma unroll
            for (int b = 0; b < R; ++b)
#pragma unroll
                for (int n = 0; n < C; ++n) acc[n][b] += part[n][b];
        };
        Operands even, odd;
        floatx4 part[C][R];
        // a step's loads go out between the slices of its products
        auto step = [&](auto stage, int t, auto ask_slice) {
            products(even, part, odd, stage, 1, [](int) {}, ask_slice);
            add(part);
            products(odd, part, even, (stage + 1) % STAGES, 0, [](int) {}, [&](int s) { ask_slice(s + 4); });
            add(part);
        };
        auto one = [&](auto stage, int t) {
            arrive(t, stage);
            if (t == 0) read(even, stage, 0);
            if (t + STAGES - 1 < steps) ask((stage + STAGES - 1) % STAGES, t + STAGES - 1);
            step(stage, t, [](int) {});
        };
        auto steady = [&](auto stage, int t) {
            wait_loads_and_barrier<(STAGES - 3) * S::PER_WAVE>();
            step(stage, t, [&](int s) {
                constexpr int EACH = (S::PER_WAVE + 6) / 7;
#pragma unroll
                for (int i = s * EACH; i < (s + 1) * EACH; ++i)
                    if (i < S::PER_WAVE) ask_one(i, (stage + STAGES - 1) % STAGES, t + STAGES - 1);
            });
        };
        const std::make_integer_sequence<int, STAGES> stages;
        // (the first steps, one for each stage; then as many at a time, while what they ask for lies inside of K)
        each(stages, [&](auto stage) { if (stage < steps) one(stage, stage); });
        int t = STAGES;
        for (; t + 2 * STAGES - 1 < steps; t += STAGES) each(stages, [&](auto stage) { steady(stage, t + stage); });
        for (; t < steps; t += STAGES) each(stages, [&](auto stage) { if (t + stage < steps) one(stage, t + stage); });
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        // element i of a block is row c * 4 + i of w's 16, row r of a's
        write([&](int g, int e) -> float {
            if constexpr (MODE == MODE_GATED) return gate_activation(acc[0][g][e], activation) * acc[1][g][e];
            else return acc[0][g][e];
        });
    } else {
        // ---- the wavefronts take a chunk each of a step's four; the chunks' sums meet in LDS and are added in the order of k
        float* parts = lds + STAGES * S::STAGE;
        float sum[C][GROUPS][V];
#pragma unroll
        for (int n = 0; n < C; ++n)
#pragma unroll
            for (int g = 0; g < GROUPS; ++g)
#pragma unroll
                for (int v = 0; v < V; ++v) sum[n][g][v] = 0.f;
        struct Ones { float v[WAVES][C][GROUPS][V]; };
        auto fetch = [&](Ones& ones, int set, int u) {            // what wavefront u left
#pragma unroll
            for (int n = 0; n < C; ++n)
#pragma unroll
                for (int g = 0; g < GROUPS; ++g) {
                    const Some some = *reinterpret_cast<const Some*>(parts + (((set * WAVES + u) * C + n) * R * 256) + (g * THREADS + tid) * V);
#pragma unroll
                    for (int v = 0; v < V; ++v) ones.v[u][n][g][v] = some[v];
                }
        };
        auto fetch_all = [&](Ones& ones, int set) {
#pragma unroll
            for (int u = 0; u < WAVES; ++u) fetch(ones, set, u);
        };
        auto add = [&](const Ones& ones) {
#pragma unroll
            for (int u = 0; u < WAVES; ++u)
#pragma unroll
                for (int n = 0; n < C; ++n)
#pragma unroll
                    for (int g = 0; g < GROUPS; ++g)
#pragma unroll
                        for (int v = 0; v < V; ++v) sum[n][g][v] += ones.v[u][n][g][v];
        };
        Operands operands[2];
        floatx4 part[2][C][R];
        Ones ones;
        auto put = [&](int set, int first, int every) {
#pragma unroll
            for (int i = first; i < C * R; i += every) *reinterpret_cast<floatx4*>(parts + ((set * WAVES + wave) * C * R + i) * 256 + lane * 4) = part[set][i / R][i % R];
        };
        // In step t the products of its chunks; the sums of the chunks of step t - 1 go into LDS, those of step t - 2 are added up.
        auto step = [&](auto stage, bool puts, bool adds, auto ask_slice) {
            products(operands[stage % 2], part[stage % 2], operands[(stage + 1) % 2], (stage + 1) % STAGES, 0, [&](int s) {
                if (adds) fetch(ones, stage % 2, s);
                if (puts) put((stage + 1) % 2, s, 4);
            }, ask_slice);
            if (adds) add(ones);
        };
        static_assert(STAGES % 2 == 0, "two sets of operands and of parts in turn, and the stages");
        auto one = [&](auto stage, int t) {
            arrive(t, stage);
            if (t == 0) read(operands[0], stage, 0);
            if (t + STAGES - 1 < steps) ask((stage + STAGES - 1) % STAGES, t + STAGES - 1);
            step(stage, t > 0, t > 1, [](int) {});
        };
        auto steady = [&](auto stage, int t) {
            wait_loads_and_barrier<(STAGES - 3) * S::PER_WAVE>();
            step(stage, true, true, [&](int s) {
                constexpr int EACH = (S::PER_WAVE + 2) / 3;
#pragma unroll
                for (int i = s * EACH; i < (s + 1) * EACH; ++i)
                    if (i < S::PER_WAVE) ask_one(i, (stage + STAGES - 1) % STAGES, t + STAGES - 1);
            });
        };
        const std::make_integer_sequence<int, STAGES> stages;
        each(stages, [&](auto stage) { if (stage < steps) one(stage, stage); });
        int t = STAGES;
        for (; t + 2 * STAGES - 1 < steps; t += STAGES) each(stages, [&](auto stage) { steady(stage, t + stage); });
        for (; t < steps; t += STAGES) each(stages, [&](auto stage) { if (t + stage < steps) one(stage, t + stage); });
        wait_loads_and_barrier<0>();
        if (steps > 1) {
            fetch_all(ones, steps % 2);
            add(ones);
        }
        if (steps % 2 == 1) put(0, 0, 1);
        else put(1, 0, 1);
        wait_loads_and_barrier<0>();
        fetch_all(ones, (steps - 1) % 2);
        add(ones);
        write([&](int g, int e) -> float {
            if constexpr (MODE == MODE_GATED) return gate_activation(sum[0][g][e], activation) * sum[C - 1][g][e];
            else return sum[0][g][e];
        });
    }
}

template <int MODE, int R, bool TOGETHER>
int launch(const float* a, const float* w, float* out, int M, int N, int K, int activation, hipStream_t s) {
    typedef Shape<MODE, R, TOGETHER> S;
    const int tiles_m = (M + S::ROWS_A - 1) / S::ROWS_A;
    const long tiles = (long)tiles_m * ((N + S::OUTPUTS - 1) / S::OUTPUTS);
    XRT_REQUIRE(tiles < (1L << 31), "linear (float32): %ld tiles", tiles);
    static const hipError_t room = hipFuncSetAttribute(reinterpret_cast<const void*>(gemm_float_kernel<MODE, R, TOGETHER>), hipFuncAttributeMaxDynamicSharedMemorySize, (int)S::LDS);
    XRT_REQUIRE(room == hipSuccess, "linear (float32): cannot reserve LDS: %s", hipGetErrorString(room));
    gemm_float_kernel<MODE, R, TOGETHER><<<(unsigned)tiles, THREADS, S::LDS, s>>>(a, w, out, M, N, K, tiles_m, activation);
    XRT_LAUNCH_CHECK("linear (float32, matrix cores)");
    return 0;
}

// The tiles that there are, and what a product takes in them, in us: fixed + ends * n + chunks of k * max(alone, share * n), n being the tiles of the fullest compute unit. Alone: a chunk of
// a tile that has a compute unit to itself; share: what each tile adds where several run there; ends: a tile's first loads and its epilogue, of each of the kinds below. Fitted to 2994 products
// drawn at random (17 to 2500 rows of a, 8 to 9000 columns, k of 4 to 8192), of which every tile was timed: what it chooses is 1.5 % off the best of nine (blocks of 1 to 7, of 1 and 2 shared), takes
// 0.544 of what the kernel before these took, and 55 of them more than 1.03 of that, 14 more than 1.1 (gated, k up to 350 and few rounds of tiles, or k of 4 to 16 and nothing but
// ends: 49 x 5136, k = 44 5.3 -> 6.2 us, 2414 x 8504, k = 12 61 -> 75, the most; of 1494 more 32 and 7, 1040 x 452, k = 140 8.6 -> 12.5: 255 tiles of 64 x 32 then, 264 of 32 x 64 now). Without the ends, which a short k consists of, 90 were above 1.03 and 49 above 1.1, up to 1.45 (358 x 3536 gated, k = 8
// 7.4 -> 10.6, now 7.9). Six blocks gated close the gap between five and seven, where as many tiles make two rounds and one (551 x 2484, k = 192 19.5 -> 17.2, 18.3 before).
enum { STORES_WIDE, STORES_NARROW, ADDS_WIDE, ADDS_NARROW };       // results in pieces of 16 bytes, or one by one; gated ones are stores
struct Takes { double fixed, alone, share, ends[4]; };
struct Tile { int rows; bool together; Takes plain, gated; };
constexpr Takes NEVER = {1e9, 0, 0, {}};
constexpr Tile TILES[] = {
    {1, false, {3.2, 0.115, 0.089, {0.5, 0.7, 0.5, 1.1}}, {2.9, 0.195, 0.168, {1.2, 1.3}}}, {2, false, {2.9, 0.178, 0.143, {0.8, 1.3, 1.0, 2.1}}, {2.8, 0.304, 0.270, {1.7, 1.9}}},
    {5, false, {2.5, 0.278, 0.338, {1.8, 3.2, 2.4, 5.6}}, {2.1, 0.277, 0.665, {4.5, 5.3}}}, {7, false, {1.1, 0.470, 0.456, {3.9, 6.0, 5.2, 10.1}}, {1.9, 0.126, 0.931, {5.5, 6.6}}},
    {1, true, {3.4, 0.047, 0.037, {0.3, 0.3, 0.4, 0.5}}, {3.2, 0.029, 0.063, {0.6, 0.6}}}, {2, true, {3.3, 0.016, 0.060, {0.5, 0.6, 0.7, 1.0}}, {2.2, 0.014, 0.109, {2.0, 2.0}}},
    {6, false, NEVER, {1.9, 0.127, 0.777, {4.9, 6.0}}}};

int tile_for(int M, int N, int K, int mode) {
    const int kind = (N % 4 == 0 ? STORES_WIDE : STORES_NARROW) + (mode == MODE_ACCUMULATE ? ADDS_WIDE : 0);
    int best = 0;
    double least = 0;
    for (int i = 0; i < (int)(sizeof(TILES) / sizeof(TILES[0])); ++i) {
        const Tile& t = TILES[i];
        const Takes& takes = mode == MODE_GATED ? t.gated : t.plain;
        const long tiles = (((long)M + 16 * t.rows - 1) / (16 * t.rows)) * ((N + (t.together ? 15 : 63L)) / (t.together ? 16 : 64));
        const long fullest = (tiles + XRT_COMPUTE_UNITS - 1) / XRT_COMPUTE_UNITS;
        const double us = takes.fixed + takes.ends[kind] * fullest + (K + 15L) / 16 * std::fmax(takes.alone, takes.share * fullest);
        if (i == 0 || us < least) { best = i; least = us; }
    }
    return best;
}

template <int MODE>
int launch_mode(const float* a, const float* w, float* out, int M, int N, int K, int activation, hipStream_t s) {
    switch (tile_for(M, N, K, MODE)) {
        case 0: return launch<MODE, 1, false>(a, w, out, M, N, K, activation, s);
        case 1: return launch<MODE, 2, false>(a, w, out, M, N, K, activation, s);
        case 2: return launch<MODE, 5, false>(a, w, out, M, N, K, activation, s);
        case 3: return launch<MODE, 7, false>(a, w, out, M, N, K, activation, s);
        case 4: return launch<MODE, 1, true>(a, w, out, M, N, K, activation, s);
        case 5: return launch<MODE, 2, true>(a, w, out, M, N, K, activation, s);
        default: break;
    }
    if constexpr (MODE == MODE_GATED) return launch<MODE, 6, false>(a, w, out, M, N, K, activation, s);
    XRT_REQUIRE(false, "linear (float32): no tile for such a product");
}

}  // namespace

bool xrt_linear_float_accepts(const void* a, const void* w, int M, int K) {
    return M > 16 && K % 4 == 0 && K <= (1 << 22) && (uintptr_t)a % 16 == 0 && (uintptr_t)w % 16 == 0;
}

int xrt_linear_float(const float* a, const float* w, float* out, int M, int N, int K, int mode, int activation, hipStream_t s) {
    if (mode == MODE_STORE) return launch_mode<MODE_STORE>(a, w, out, M, N, K, activation, s);
    if (mode == MODE_ACCUMULATE) return launch_mode<MODE_ACCUMULATE>(a, w, out, M, N, K, activation, s);
    return launch_mode<MODE_GATED>(a, w, out, M, N, K, activation, s);
}

extern "C" int xrt_linear_float_tile(int M, int N, int K, int mode, int* rows, int* together) {
    if (M <= 16 || N <= 0 || K <= 0 || mode < 0 || mode > 2 || rows == nullptr || together == nullptr) return 1;
    const Tile& t = TILES[tile_for(M, N, K, mode)];
    *rows = 16 * t.rows;
    *together = t.together;
    return 0;
}
