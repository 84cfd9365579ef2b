// Matrix product for many rows (prefill), bfloat16 operands, float32 accumulation on the
// matrix cores: out[m, n] = sum_k a[m, k] * w[n, k]; both operands are contiguous along k.
//
// The large tiles (256, 192 or 128 rows by 256, eight wavefronts; K a multiple of 64) are gemm_large_tile. In the others
// a workgroup computes a BM x BN tile of the output with v_mfma_f32_32x32x16_bf16. Tiles of
// a and w travel through LDS, several steps ahead of the matrix cores, with one barrier per
// step. When K is a multiple of 64 they are loaded from global memory straight into LDS, in a
// swizzled layout; otherwise they pass through registers into rows padded by 16 bytes (64 wide
// in k, the last tile filled with zeros). Either layout keeps the 16-byte operand reads of
// consecutive rows in different banks. Each wavefront owns a (BM/WM) x (BN/WN) part of the
// tile and keeps its accumulators in registers for the whole K loop.
//
// Workgroup ids are remapped so that the workgroups that run on one XCD (ids are dealt
// round-robin to the 8 XCDs) work on neighbouring tiles and share their operands in that
// XCD's L2.
//
// Epilogues: store (bfloat16 or float32), accumulate into float32, or the gated pair
// silu(gate) * up: then the w tile holds BN/2 gate rows and the BN/2 up rows that belong to
// them (rows n and n + N of w), arranged so that each wavefront holds both of a pair.
#include <climits>
#include <cstdlib>
#include <type_traits>
#include "packing.h"
#include "gemm_skinny.h"
#include "activation.h"

namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float floatx16 __attribute__((ext_vector_type(16)));
typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef unsigned uint4v __attribute__((ext_vector_type(4)));

template <typename T> struct alignas(sizeof(T) * 4) Four { T e[4]; };

constexpr int BK = 64;
constexpr int PITCH = BK + 8;          // bf16 elements per LDS row
enum { MODE_STORE = 0, MODE_ACCUMULATE = 1, MODE_GATED = 2 };

// Which tile of tiles_m x tiles_n a workgroup takes. Ids are dealt to the XCDs round-robin: each XCD gets a contiguous run of
// tiles, and a run is walked n-fastest inside panels of 8 n-tiles, so that the tiles that run at one time on an XCD share a
// and w in its L2; m-fastest where there are up to four rows of tiles (a panel's tiles of one n would often lie on two XCDs, which then both read their w), but not where k
// is no multiple of 64 (panels): operands then go through the registers, and tiles of one n that run side by side took up to 1.12 times as long as those of one m (331 rows of
// x, 12696 of w, k = 8480 160 -> 180 us; 150 such products otherwise the same). An id beyond the tiles (grids are whole rounds over the XCDs) has none: m is negative.
struct TilePlace { int m, n; };
__host__ __device__ __forceinline__ TilePlace tile_place(int id, int tiles_m, int tiles_n, bool panels = false) {
    const int total = tiles_m * tiles_n;
    const int xcds = 8;
    id = (id % xcds) * ((total + xcds - 1) / xcds) + id / xcds;
    if (id >= total) return TilePlace{-1, 0};
    if (tiles_m <= 4 && !panels) return TilePlace{id % tiles_m, id / tiles_m};
    constexpr int PANEL = 8;
    const int panel = id / (PANEL * tiles_m), in_panel = id % (PANEL * tiles_m);
    const int panel_width = min(PANEL, tiles_n - panel * PANEL);
    return TilePlace{in_panel / panel_width, panel * PANEL + in_panel % panel_width};
}

// The same of a product whose k is split into parts, in one of two orders. By columns: an XCD gets a run of tiles and all parts of them, a grid row each. By
// parts (by_parts: their number; else 0, and `row` is the workgroup's grid row): it gets a run of tiles and parts, part after part, so that it reads some
// slices of k of a, which its L2 holds, instead of all of a, and no XCD has more to do for a number of tiles that does not divide.
struct PartPlace { TilePlace tile; int part; };
__host__ __device__ __forceinline__ PartPlace part_place(int id, int row, int tiles_m, int tiles_n, int by_parts) {
    if (by_parts == 0) return PartPlace{tile_place(id, tiles_m, tiles_n), row};
    constexpr int XCDS = 8;
    const int tiles = tiles_m * tiles_n, total = tiles * by_parts;
    id = (id % XCDS) * ((total + XCDS - 1) / XCDS) + id / XCDS;
    if (id >= total) return PartPlace{TilePlace{-1, 0}, 0};
    const int tile = id % tiles;
    return PartPlace{TilePlace{tile % tiles_m, tile / tiles_m}, id / tiles};
}
// Workgroups that such a product's launch has, places that no tile is dealt to among them.
inline long part_ids(long tiles, int parts, bool by_parts) { return by_parts ? (tiles * parts + 7) / 8 * 8 : (tiles + 7) / 8 * 8 * parts; }

// The rows of a that come without their RMSNorm's division (see xrt_linear_norm in xrt_hip.h): the sums of
// squares per tile of 16 columns, from which a tile of up to 64 rows works out 1 / rms of its rows and
// multiplies its sums by it before the epilogue. squares null: nothing of the kind.
struct RowScale { const float* squares; int tiles; int width; float eps; int activation; };     // (activation: of a gated epilogue)

// One tile of the product, or of one part of its k, by one workgroup: `id` is the workgroup's number among them.
// PAST_CACHES: w is asked for past the caches.
template <int BM, int BN, int WM, int WN, int MODE, int DK, int STAGES, typename TO, bool PAST_CACHES = false>
__device__ __forceinline__ void gemm_tile(
    const bf16* __restrict__ a, const bf16* __restrict__ w, TO* __restrict__ out, int M, int N, int K,
    int id, int tiles_m, int tiles_n, int by_parts, int k_per_split, const Packing packing, const RowScale scale) {
    constexpr int THREADS = WM * WN * XRT_WAVE;
    constexpr int WAVE_M = BM / WM, WAVE_N = BN / WN;        // part of the tile owned by one wavefront
    constexpr int TM = WAVE_M / 32, TN = WAVE_N / 32;        // 32x32 accumulator tiles of a wavefront
    constexpr int CHUNKS_A = BM * BK / 8 / THREADS;          // 16-byte chunks each thread moves per step
    constexpr int CHUNKS_B = BN * BK / 8 / THREADS;

    extern __shared__ __attribute__((aligned(16))) unsigned char lds_raw[];
    bf16* lds_a = reinterpret_cast<bf16*>(lds_raw);                    // [2][BM][PITCH]; laid out differently on the direct path
    bf16* lds_b = lds_a + 2 * BM * PITCH;                              // [2][BN][PITCH]

    // (a float32 store may be of a part; of the others none is, and their way to the first loads is shorter)
    const PartPlace of_part = MODE == MODE_STORE && sizeof(TO) == 4 && DK != 0 ? part_place(id, blockIdx.y, tiles_m, tiles_n, by_parts)
                                                                               : PartPlace{tile_place(id, tiles_m, tiles_n, DK == 0), 0};
    const TilePlace place = of_part.tile;
    if (place.m < 0) return;
    // (rows, columns and byte offsets fit 32 bits: the launcher checks)
    const int m0 = place.m * BM;
    constexpr int BN_OUT = MODE == MODE_GATED ? BN / 2 : BN;          // output columns of a tile
    const int n0 = place.n * BN_OUT;

    const int tid = threadIdx.x, lane = tid % XRT_WAVE, wave = tid / XRT_WAVE;
    const int wave_m = wave / WN, wave_n = wave % WN;

    // Row of w behind row r of the tile. In the gated mode the rows that one wavefront owns are
    // half gate rows and half the up rows of the same outputs (rows n and n + N of w), so that the
    // pair meets in that wavefront's registers. Rows beyond the operands are clamped to the last
    // row: loads then need no guard, and what such a row contributes lands in outputs that are
    // not written.
    auto w_row = [&](int r) -> int {
        if constexpr (MODE == MODE_GATED) {
            constexpr int HALF = WAVE_N / 2;
            const int within = r % WAVE_N;
            return min(n0 + (r / WAVE_N) * HALF + within % HALF, N - 1) + (within / HALF) * N;
        } else {
            return min(n0 + r, N - 1);
        }
    };
    // 1 / rms of the tile's rows, if the rows of a come without it. The sums of squares are asked for now,
    // all at once (a thread takes four neighbouring rows of every sixteenth tile, or eighth where there are 128 threads, 16 bytes a load), and added
    // up after the main loop, when they have long arrived.
    constexpr int SUMMERS = THREADS < 256 ? THREADS / 16 : 16; // threads that add up the sums of a row
    constexpr int SQUARE_LOADS = 256 / SUMMERS;                // tiles of 16 columns per thread: rows of up to 256 * 16 columns
    __shared__ float row_scale[BM <= 64 ? 64 : 1];
    __shared__ float row_parts[BM <= 64 ? SUMMERS : 1][64];
    float4 early_squares[BM <= 64 ? SQUARE_LOADS : 1];
    const bool scaled = BM <= 64 && scale.squares != nullptr;
    if constexpr (BM <= 64) {
        if (scaled && tid < 256) {
#pragma unroll
            for (int u = 0; u < SQUARE_LOADS; ++u) {
                const int t = tid / 16 + SUMMERS * u;
                early_squares[u] = t < scale.tiles
                    ? *reinterpret_cast<const float4*>(scale.squares + (long)t * XRT_SQUARES_STRIDE + (tid % 16) * 4)
                    : make_float4(0.f, 0.f, 0.f, 0.f);
            }
        }
    }
    floatx16 acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.f;

    if constexpr (DK != 0) {
        // Tiles go from global memory straight into LDS (global_load_lds_dwordx4): no registers and
        // no LDS write instructions in between. Tiles are DK wide in k and LDS holds STAGES of
        // them: while one is multiplied, the next is complete and STAGES - 2 more are on their
        // way. One load instruction of a wavefront fills 64 consecutive 16-byte places of LDS,
        // lane by lane, which is 64 / CHUNKS whole rows; rows can therefore not be padded. Instead
        // the chunks of a row are stored in permuted places, place = chunk ^ swizzle(row), and
        // each lane fetches the chunk that belongs in its place. The swizzles are chosen so that
        // the operand reads of 8 and of 16 consecutive rows at one chunk fall into different
        // 16-byte bank groups.
        constexpr int CHUNKS = DK / 8;                             // 16-byte chunks per row: 4 or 8
        constexpr int ROWS = 64 / CHUNKS;                          // rows that one load instruction fills
        constexpr int WAVES = WM * WN;
        // load instructions per wavefront and tile; where the row blocks do not divide among the
        // wavefronts, the spare instructions fetch the last block once more (same bytes, same place)
        constexpr int BLOCKS_A = BM / ROWS, BLOCKS_B = BN / ROWS;
        constexpr int LOADS_A = (BLOCKS_A + WAVES - 1) / WAVES, LOADS_B = (BLOCKS_B + WAVES - 1) / WAVES;
        constexpr int SLICES = DK / 16;
        static_assert(DK == 32 || DK == 64, "swizzles exist for rows of 4 and of 8 chunks");
        static_assert(BM % ROWS == 0 && BN % ROWS == 0, "tile rows do not divide into load instructions");
        bf16* stage_a = lds_a;                                     // [STAGES][BM][DK]
        bf16* stage_b = lds_a + STAGES * BM * DK;                  // [STAGES][BN][DK]
        auto swizzle_of = [](int r) { return CHUNKS == 4 ? (r / 2 % 4) ^ (r / 8 % 2) : (r % 8) ^ (r / 8 % 2); };
        const int sub = lane / CHUNKS;                             // row within the rows of one instruction
        auto chunk_of = [&](int row) { return ((lane % CHUNKS) ^ swizzle_of(row)) * 8; };   // what belongs in this lane's place
        unsigned off_a[LOADS_A], off_b[LOADS_B];                   // bytes
#pragma unroll
        for (int i = 0; i < LOADS_A; ++i) {
            const int r = min(i * WAVES + wave, BLOCKS_A - 1) * ROWS + sub;
            off_a[i] = ((unsigned)min(m0 + r, M - 1) * (unsigned)K + (unsigned)chunk_of(r)) * 2u;
        }
        // A packed w is copied as it lies: an instruction takes one whole tile of the packing (16 packed rows x 32
        // columns, a contiguous kilobyte, lane by lane), and the stage holds the tile's groups of 16 packed rows
        // one after another, two tiles of 32 columns each. The 16 lanes that read an operand's 16 rows at one
        // piece of 8 columns then read 256 contiguous bytes of LDS. (Fetched piece by piece into the layout of
        // rows contiguous along k, every four lanes would touch four cache lines: a fifth slower, measured.)
        // The tile's rows are then packed rows first_packed .. + BN, and the epilogue finds the outputs they make.
        const bool packed_b = is_packed(packing);
        const int first_packed = MODE == MODE_GATED ? 2 * n0 : n0;
        const int last_group = ((MODE == MODE_GATED ? 2 * N : N) + 15) / 16 - 1;
        if (packed_b) {
#pragma unroll
            for (int i = 0; i < LOADS_B; ++i) {
                const int block = min(i * WAVES + wave, BLOCKS_B - 1);
                const int group = min(first_packed / 16 + block / 2, last_group);        // groups beyond the matrix: the last one again
                off_b[i] = ((unsigned)group * (unsigned)(K / 32) + (unsigned)(block % 2)) * 1024u + (unsigned)lane * 16u;
            }
        } else {
#pragma unroll
            for (int i = 0; i < LOADS_B; ++i) {
                const int r = min(i * WAVES + wave, BLOCKS_B - 1) * ROWS + sub;
                off_b[i] = ((unsigned)w_row(r) * (unsigned)K + (unsigned)chunk_of(r)) * 2u;
            }
        }
        // a step of k0 columns along k moves a row contiguous along k by k0 elements, a packed one by k0 / 32 tiles
        const unsigned w_step = packed_b ? 32u : 2u;                // bytes per column of k
        const int wave_uniform = __builtin_amdgcn_readfirstlane(wave);
        const unsigned lds_a0 = lds_address(stage_a), lds_b0 = lds_address(stage_b);
        auto issue = [&](int stage, int k0) {
#pragma unroll
            for (int i = 0; i < LOADS_A; ++i) {
                const int block = min(i * WAVES + wave_uniform, BLOCKS_A - 1);
                load_to_lds(a, off_a[i] + (unsigned)k0 * 2u, lds_a0 + (unsigned)((stage * BM + block * ROWS) * DK * 2));
            }
#pragma unroll
            for (int i = 0; i < LOADS_B; ++i) {
                const int block = min(i * WAVES + wave_uniform, BLOCKS_B - 1);
                const unsigned to = lds_b0 + (unsigned)((stage * BN + block * ROWS) * DK * 2);
                if constexpr (PAST_CACHES) stream_to_lds(w, off_b[i] + (unsigned)k0 * w_step, to);
                else load_to_lds(w, off_b[i] + (unsigned)k0 * w_step, to);
            }
        };
        const int swizzle = swizzle_of(lane % 16);                 // of every row this lane reads: they differ by multiples of 32
        // where this lane finds its piece of the w operand for each slice, from the start of its wavefront's rows
        int b_place[SLICES];
#pragma unroll
        for (int slice = 0; slice < SLICES; ++slice)
            b_place[slice] = packed_b ? (lane % 32 / 16 * 2 + slice / 2) * 512 + ((slice % 2 * 2 + lane / 32) * 16 + lane % 16) * 8
                                      : (lane % 32) * DK + ((slice * 2 + lane / 32) ^ swizzle) * 8;
        // operands of one 16-wide slice of k: TM row blocks of a, TN row blocks of w
        struct Operands { bf16x8 a[TM], b[TN]; };
        auto read = [&](Operands& r, int stage, int slice) {
            const int place = ((slice * 2 + lane / 32) ^ swizzle) * 8;
            const bf16* tile_a = stage_a + ((long)stage * BM + wave_m * WAVE_M + lane % 32) * DK + place;
            const bf16* tile_b = stage_b + ((long)stage * BN + wave_n * WAVE_N) * DK + b_place[slice];
#pragma unroll
            for (int i = 0; i < TM; ++i) r.a[i] = *reinterpret_cast<const bf16x8*>(tile_a + i * 32 * DK);
#pragma unroll
            for (int j = 0; j < TN; ++j) r.b[j] = *reinterpret_cast<const bf16x8*>(tile_b + j * 32 * DK);
        };
        auto multiply = [&](const Operands& r) {
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int j = 0; j < TN; ++j)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(r.a[i], r.b[j], acc[i][j], 0, 0, 0);
        };
        // The launcher sends only K that is a multiple of DK here. Every step issues the loads of
        // the tile STAGES - 1 steps ahead; beyond the end of k it repeats the last tile (into a
        // stage nobody uses any more), so that the number of loads in flight is the same at every
        // wait. The operands of each slice are read from LDS while the matrix cores work on the
        // slice before it, across the barrier too: the first slice of the next tile is read right
        // after the barrier, under the products of the last slice of this one.
        constexpr int AHEAD = STAGES - 1;
        constexpr int IN_FLIGHT = (AHEAD - 1) * (LOADS_A + LOADS_B);   // loads that may be outstanding when the next tile is needed
        // part p of a product split along k takes k_per_split from p * k_per_split on (less at the
        // end) and writes its sums to the p-th copy of out
        const int k_begin = of_part.part * k_per_split;
        const int steps = min(k_per_split, K - k_begin) / DK;
        const int last_k = k_begin + (steps - 1) * DK;
        out += (long)of_part.part * M * N;
#pragma unroll
        for (int i = 0; i < AHEAD; ++i) issue(i, min(k_begin + i * DK, last_k));
        wait_loads_and_barrier<IN_FLIGHT>();                      // tile 0 is in LDS
        Operands operands[2];
        read(operands[0], 0, 0);
        for (int t = 0; t < steps; ++t) {
            issue((t + AHEAD) % STAGES, min(k_begin + (t + AHEAD) * DK, last_k));   // that stage was read in step t-1, before the last barrier
#pragma unroll
            for (int slice = 0; slice + 1 < SLICES; ++slice) {
                read(operands[(slice + 1) % 2], t % STAGES, slice + 1);
                __builtin_amdgcn_sched_barrier(0);                // keeps the reads ahead of the products that hide them
                multiply(operands[slice % 2]);
                __builtin_amdgcn_sched_barrier(0);
            }
            wait_loads_and_barrier<IN_FLIGHT>();                  // tile t+1 has arrived from every wavefront, tile t has been read by all
            read(operands[0], (t + 1) % STAGES, 0);               // after the last step: a repeated tile, not used
            __builtin_amdgcn_sched_barrier(0);
            multiply(operands[(SLICES - 1) % 2]);
        }
        wait_loads_and_barrier<0>();                              // nothing lands in LDS after this
    } else {
        // element offsets of this thread's chunks from the operands' bases (32 bits: the launcher checks)
        unsigned off_a[CHUNKS_A], off_b[CHUNKS_B];
    #pragma unroll
        for (int i = 0; i < CHUNKS_A; ++i) {
            const int chunk = tid + i * THREADS;
            off_a[i] = (unsigned)min(m0 + chunk / 8, M - 1) * (unsigned)K + (unsigned)(chunk % 8) * 8u;
        }
    #pragma unroll
        for (int i = 0; i < CHUNKS_B; ++i) {
            const int chunk = tid + i * THREADS;
            off_b[i] = (unsigned)weight_offset(packing, w_row(chunk / 8), (chunk % 8) * 8, K);
        }
        const unsigned w_step = is_packed(packing) ? 16u : 1u;      // elements per column of k (tiles are 64 wide here: whole tiles of the packing)

        struct Stage { bf16x8 a[CHUNKS_A], b[CHUNKS_B]; };
        auto fetch = [&](Stage& stage, int k0) {                  // a whole tile of 64 along k, no guards
    #pragma unroll
            for (int i = 0; i < CHUNKS_A; ++i) stage.a[i] = *reinterpret_cast<const bf16x8*>(a + (off_a[i] + (unsigned)k0));
    #pragma unroll
            for (int i = 0; i < CHUNKS_B; ++i) stage.b[i] = *reinterpret_cast<const bf16x8*>(w + (off_b[i] + (unsigned)k0 * w_step));
        };
        auto fetch_tail = [&](Stage& stage, int k0) {             // the last tile when K is no multiple of 64: zeros beyond K
    #pragma unroll
            for (int i = 0; i < CHUNKS_A; ++i) {
                const int k = k0 + ((tid + i * THREADS) % 8) * 8;
                stage.a[i] = k + 8 <= K ? *reinterpret_cast<const bf16x8*>(a + (off_a[i] + (unsigned)k0)) : bf16x8{};
            }
    #pragma unroll
            for (int i = 0; i < CHUNKS_B; ++i) {
                const int k = k0 + ((tid + i * THREADS) % 8) * 8;
                stage.b[i] = k + 8 <= K ? *reinterpret_cast<const bf16x8*>(w + (off_b[i] + (unsigned)k0 * w_step)) : bf16x8{};
            }
        };
        auto stash = [&](const Stage& stage, int buffer) {
    #pragma unroll
            for (int i = 0; i < CHUNKS_A; ++i) {
                const int chunk = tid + i * THREADS, r = chunk / 8, kc = chunk % 8;
                *reinterpret_cast<bf16x8*>(lds_a + ((long)buffer * BM + r) * PITCH + kc * 8) = stage.a[i];
            }
    #pragma unroll
            for (int i = 0; i < CHUNKS_B; ++i) {
                const int chunk = tid + i * THREADS, r = chunk / 8, kc = chunk % 8;
                *reinterpret_cast<bf16x8*>(lds_b + ((long)buffer * BN + r) * PITCH + kc * 8) = stage.b[i];
            }
        };

        // The products of one LDS buffer. `between` runs ahead of them: it writes the next tile to the
        // other LDS buffer and requests the tile after it. (Placing it halfway through the products
        // was measured slower: the fetched registers then stay live across all of them.)
        auto compute = [&](int buffer, auto between) {
            const bf16* tile_a = lds_a + ((long)buffer * BM + wave_m * WAVE_M + lane % 32) * PITCH + (lane / 32) * 8;
            const bf16* tile_b = lds_b + ((long)buffer * BN + wave_n * WAVE_N + lane % 32) * PITCH + (lane / 32) * 8;
    #pragma unroll
            for (int ks = 0; ks < BK / 16; ++ks) {
                if (ks == 0) between();
                bf16x8 ra[TM], rb[TN];
    #pragma unroll
                for (int i = 0; i < TM; ++i) ra[i] = *reinterpret_cast<const bf16x8*>(tile_a + i * 32 * PITCH + ks * 16);
    #pragma unroll
                for (int j = 0; j < TN; ++j) rb[j] = *reinterpret_cast<const bf16x8*>(tile_b + j * 32 * PITCH + ks * 16);
    #pragma unroll
                for (int i = 0; i < TM; ++i)
    #pragma unroll
                    for (int j = 0; j < TN; ++j)
                        acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ra[i], rb[j], acc[i][j], 0, 0, 0);
            }
        };
        auto nothing = [] {};

        // Tiles travel global -> registers -> LDS ahead of the matrix cores. During step t the
        // registers hold tile t+1 (fetched a step ago): it is written into the LDS buffer that step t-1
        // has finished with, the registers are refilled with tile t+2, and tile t is multiplied. The steady-state loop has no branch.
        const int whole = K / BK;                                 // tiles of 64 that lie inside K
        Stage s0;
        if (whole > 0) {
            fetch(s0, 0);
            stash(s0, 0);
            if (whole > 1) fetch(s0, BK);
            __syncthreads();
            int t = 0;                                            // LDS buffer 0 holds tile t, the registers tile t+1
            for (; t + 3 < whole; t += 2) {
                compute(0, [&] { stash(s0, 1); fetch(s0, (t + 2) * BK); });
                __syncthreads();
                compute(1, [&] { stash(s0, 0); fetch(s0, (t + 3) * BK); });
                __syncthreads();
            }
            const int left = whole - t;                           // 1, 2 or 3
            compute(0, [&] { if (left >= 2) stash(s0, 1); if (left == 3) fetch(s0, (t + 2) * BK); });
            if (left >= 2) {
                __syncthreads();
                compute(1, [&] { if (left == 3) stash(s0, 0); });
            }
            if (left == 3) {
                __syncthreads();
                compute(0, nothing);
            }
        }
        if (whole * BK < K) {
            fetch_tail(s0, whole * BK);
            __syncthreads();                                      // everyone is done with buffer 0
            stash(s0, 0);
            __syncthreads();
            compute(0, nothing);
        }
    }

    // ---- epilogue: accumulator element e of tile (i, j) is row (e/4)*8 + (lane/32)*4 + e%4, column lane%32
    if constexpr (BM <= 64) {
        if (scaled) {                                          // the same for all threads of the workgroup
            if (tid < 256) {
                float4 sum = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
                for (int u = 0; u < SQUARE_LOADS; ++u) {
                    sum.x += early_squares[u].x; sum.y += early_squares[u].y; sum.z += early_squares[u].z; sum.w += early_squares[u].w;
                }
                // rows of more than 4096 columns: the tiles beyond, one after the other
                for (int t = tid / 16 + SUMMERS * SQUARE_LOADS; t < scale.tiles; t += SUMMERS) {
                    const float4 more = *reinterpret_cast<const float4*>(scale.squares + (long)t * XRT_SQUARES_STRIDE + (tid % 16) * 4);
                    sum.x += more.x; sum.y += more.y; sum.z += more.z; sum.w += more.w;
                }
                *reinterpret_cast<float4*>(&row_parts[tid / 16][(tid % 16) * 4]) = sum;
            }
            __syncthreads();
            if (tid < 64) {
                float total = 0.f;
#pragma unroll
                for (int part = 0; part < SUMMERS; ++part) total += row_parts[part][tid];
                row_scale[tid] = 1.0f / sqrtf(total / (float)scale.width + scale.eps);
            }
            __syncthreads();
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int e = 0; e < 16; ++e) {
                    const float by = row_scale[wave_m * WAVE_M + i * 32 + (e / 4) * 8 + (lane / 32) * 4 + e % 4];
#pragma unroll
                    for (int j = 0; j < TN; ++j) acc[i][j][e] *= by;
                }
        }
    }
    // With a packed w that was copied as it lies (whole tiles along k), column q of the tile is packed row
    // first_packed + q of w: the outputs are found through the packing.
    const bool packed_columns = DK != 0 && is_packed(packing);
    if (MODE == MODE_GATED && packed_columns) {
        // A group of 16 packed rows: the gate rows of 8 outputs, then their up rows: a lane's partner is 8 lanes away.
        // The two share the work: of two neighbouring rows of the tile the lane with the gates finishes the first
        // (with its partner's up sum), the lane with the ups the second (with its partner's gate sum).
        const int q = lane % 32;
        const bool has_gates = q % 16 < 8;
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j) {
                const long n = n0 + (wave_n * WAVE_N + j * 32) / 2 + q / 16 * 8 + q % 8;
#pragma unroll
                for (int e = 0; e < 16; e += 2) {
                    const float first = acc[i][j][e], second = acc[i][j][e + 1];
                    const float partner_first = from_eight_lanes_away(first), partner_second = from_eight_lanes_away(second);
                    const float gate = has_gates ? first : partner_second, up = has_gates ? partner_first : second;
                    const long m = m0 + wave_m * WAVE_M + i * 32 + (e / 4) * 8 + (lane / 32) * 4 + e % 4 + (has_gates ? 0 : 1);
                    if (m < M && n < N) out[m * (long)N + n] = from_float<TO>(gate_activation<sizeof(TO) == 2>(gate, scale.activation) * up);
                }
            }
    } else if constexpr (MODE == MODE_GATED) {
        static_assert(TN % 2 == 0, "a wavefront holds as many gate blocks as up blocks");
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN / 2; ++j)
#pragma unroll
                for (int e = 0; e < 16; ++e) {
                    const long m = m0 + wave_m * WAVE_M + i * 32 + (e / 4) * 8 + (lane / 32) * 4 + e % 4;
                    const long n = n0 + wave_n * (WAVE_N / 2) + j * 32 + lane % 32;
                    if (m < M && n < N) out[m * (long)N + n] = from_float<TO>(gate_activation<sizeof(TO) == 2>(acc[i][j][e], scale.activation) * acc[i][j + TN / 2][e]);
                }
    } else {
        long column[TN];                                        // the output column of this lane in each block of 32
#pragma unroll
        for (int j = 0; j < TN; ++j) {
            column[j] = n0 + wave_n * WAVE_N + j * 32 + lane % 32;
            if (packed_columns) column[j] = column[j] < N ? logical_row(packing, column[j]) : (long)N;     // (packed rows beyond w make nothing)
        }
#pragma unroll
        for (int i = 0; i < TM; ++i) {
            // When accumulating, what the outputs of one row block hold is read in one go, from
            // addresses clamped into the matrix, before any of them is written: guarded, each
            // read would wait for the one before it.
            float before[TN][16];
            if constexpr (MODE == MODE_ACCUMULATE) {
#pragma unroll
                for (int j = 0; j < TN; ++j)
#pragma unroll
                    for (int e = 0; e < 16; ++e) {
                        const long m = min(m0 + wave_m * WAVE_M + i * 32 + (e / 4) * 8 + (lane / 32) * 4 + e % 4, M - 1);      // (of an int and a long: the double's min)
                        const long n = min(column[j], (long)N - 1);
                        before[j][e] = to_float(out[m * (long)N + n]);
                    }
            }
#pragma unroll
            for (int j = 0; j < TN; ++j)
#pragma unroll
                for (int e = 0; e < 16; ++e) {
                    const long m = m0 + wave_m * WAVE_M + i * 32 + (e / 4) * 8 + (lane / 32) * 4 + e % 4;
                    const long n = column[j];
                    if (m < M && n < N) {
                        if constexpr (MODE == MODE_STORE) out[m * (long)N + n] = from_float<TO>(acc[i][j][e]);
                        else out[m * (long)N + n] = from_float<TO>(before[j][e] + acc[i][j][e]);
                    }
                }
        }
    }
}

// ---- the large tiles' small pieces
// The upper 32 lanes of `low` change places with the lower 32 lanes of `high`.
__device__ __forceinline__ void exchange_halves(float& low, float& high) {
    const auto both = __builtin_amdgcn_permlane32_swap(__builtin_bit_cast(unsigned, low), __builtin_bit_cast(unsigned, high), false, false);
    const unsigned first = both[0], second = both[1];          // (a vector's element itself is not what a bit cast takes)
    low = __builtin_bit_cast(float, first);
    high = __builtin_bit_cast(float, second);
}
// In every row of 16 lanes the upper eight lanes of `low` change places with the lower eight lanes of `high`.
__device__ __forceinline__ void exchange_eights(unsigned& low, unsigned& high) {
    const unsigned l = low, h = high;
    low = __builtin_amdgcn_update_dpp(l, h, 0x128 /* row_ror:8 */, 0xf, 0xc /* lanes 8 to 15 */, false);
    high = __builtin_amdgcn_update_dpp(h, l, 0x128, 0xf, 0x3 /* lanes 0 to 7 */, false);
}
__device__ __forceinline__ void exchange_eights(float& low, float& high) {
    unsigned l = __builtin_bit_cast(unsigned, low), h = __builtin_bit_cast(unsigned, high);
    exchange_eights(l, h);
    low = __builtin_bit_cast(float, l);
    high = __builtin_bit_cast(float, h);
}
template <typename TO>
__device__ __forceinline__ unsigned two_bf16(float a, float b) {
    return (unsigned)__builtin_bit_cast(unsigned short, from_float<bf16>(a)) | (unsigned)__builtin_bit_cast(unsigned short, from_float<bf16>(b)) << 16;
}
// Four values of each of two blocks, rounded to bfloat16, exchanged between the two rows of 16 lanes of each half of the
// wavefront: the first row gets the first block's values of both rows (eight neighbours), the second row the second block's.
template <typename TO>
__device__ __forceinline__ uint4v join_rows(const float (&first)[4], const float (&second)[4]) {
    const auto low = __builtin_amdgcn_permlane16_swap(two_bf16<TO>(first[0], first[1]), two_bf16<TO>(second[0], second[1]), false, false);
    const auto high = __builtin_amdgcn_permlane16_swap(two_bf16<TO>(first[2], first[3]), two_bf16<TO>(second[2], second[3]), false, false);
    return uint4v{low[0], high[0], low[1], high[1]};
}
// Four neighbouring columns of a row of out [M][N], in one piece where `wide` says that rows and columns allow it.
template <typename TO>
__device__ __forceinline__ void load_four(const TO* out, long m, long n, int M, int N, float (&v)[4], bool wide) {
    const TO* row = out + min(m, (long)M - 1) * (long)N;       // (rows and columns beyond the matrix: something inside, not used)
    if (wide) {
        const Four<TO> four = *reinterpret_cast<const Four<TO>*>(row + min(n, (long)N - 4));
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = to_float(four.e[e]);
    } else {
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = to_float(row[min(n + e, (long)N - 1)]);
    }
}
template <typename TO>
__device__ __forceinline__ void store_four(TO* out, long m, long n, int M, int N, const float (&v)[4], bool wide) {
    if (m >= M || n >= N) return;
    TO* row = out + m * (long)N;
    if (wide) {
        Four<TO> four;
#pragma unroll
        for (int e = 0; e < 4; ++e) four.e[e] = from_float<TO>(v[e]);
        *reinterpret_cast<Four<TO>*>(row + n) = four;
    } else {
#pragma unroll
        for (int e = 0; e < 4; ++e)
            if (n + e < N) row[n + e] = from_float<TO>(v[e]);
    }
}

constexpr int LARGE_BN = 256;

// The large tiles: eight wavefronts, two to a SIMD, BM (256, 192 or 128) x 256, for K that is a multiple of 64; any split of k and all three epilogues.
//
// What bounds them is the chip's power: run without a pause on random operands the clock falls to 1.5 GHz, and what counts is
// the energy of a product, not its cycles. v_mfma_f32_16x16x32_bf16 moves half as many partial sums per product through the
// registers as the 32x32x16 instruction does: on operands that stay in registers 2060 against 1820 TFLOP/s (zeros, which cost
// no power: 2430 and 2460). The instruction's A operand is w and its B operand x, so that a lane ends up with four
// neighbouring columns of one row of the output, and the epilogue moves 16 bytes a lane.
//
// The wavefronts take turns: of the two on a SIMD (one of each group of four) one reads the operands of its next products
// from LDS and asks for tiles to come while the other multiplies; a barrier ends a turn, and the second group runs one barrier
// behind the first. A wavefront's part (BM/2 x 64) is four quarters of 64 x 64 along k: (half h of its rows of x, half g of its
// rows of w) in the order (0,0) (0,1) (1,1) (1,0), so that every turn reads one new half: w0, w1, x1, and x0 of the next tile.
// A half is loaded into the place of the same half two tiles ago as soon as both groups have read that, seven quarters before
// it is needed, and the waits leave the newer six quarters' loads in flight. So the matrix cores are busy in 98 % of the
// loop's cycles (2084 a step of 64 for 2048 of products; with one barrier a step and every wavefront doing both at once: 61 %).
//
// height: the rows of a that a tile stands for, a multiple of 16 up to BM. The rows of a product are dealt to its tiles evenly (even_height), so that none has
// more than it must: the first four wavefronts take half of the blocks of 16, or one more than the others, and a wavefront runs the loop that is made for its
// number of blocks (all, one or two fewer). The chip's power bounds the loop, so that products left out are time: 333 rows in two tiles of 176 instead of 192
// and 141, 28672 rows of w in pairs, k = 4096 77.6 -> 73.9 us, 51200, k = 5120 194 -> 179; 400 rows (208 each) 221 -> 196.
template <int BM, int MODE, typename TO>
__device__ __forceinline__ void gemm_large_tile(
    const bf16* __restrict__ a, const bf16* __restrict__ w, TO* __restrict__ out, int M, int N, int K,
    const TilePlace place, int n_first, int part, int k_per_split, const Packing packing, const int activation, const int height = BM, const int lda = 0,
    const int ldw = 0) {
    constexpr int BN = LARGE_BN, DK = 64, WAVES_N = 4;
    constexpr int WAVE_M = BM / 2, WAVE_N = BN / WAVES_N;      // the wavefront's part of the tile
    constexpr int TM = WAVE_M / 16, TN = WAVE_N / 16, HM = TM / 2, HN = TN / 2;      // blocks of 16 rows of x and of w: all, and a half
    constexpr int BLOCKS_A = BM / 16;                          // kilobytes of one half of x: where they do not divide among the wavefronts, the spare loads fetch the last one again
    constexpr int LOADS_A = (BLOCKS_A + 7) / 8, LOADS_B = BN / 128;      // load instructions of a wavefront for one half
    extern __shared__ __attribute__((aligned(16))) unsigned char lds_raw[];
    bf16* stage_a = reinterpret_cast<bf16*>(lds_raw);          // [2][BM][64]: rows of eight 16-byte pieces, swizzled
    bf16* stage_b = stage_a + 2 * BM * DK;                     // [2][256][64]: likewise, or packed tiles as they lie

    // (rows, columns and byte offsets fit 32 bits: the launchers check; a short way to the first loads counts in every launch)
    const int m0 = place.m * height;
    constexpr int BN_OUT = MODE == MODE_GATED ? BN / 2 : BN;   // output columns of a tile
    const int n0 = n_first + place.n * BN_OUT;
    const int lane = threadIdx.x % XRT_WAVE, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / XRT_WAVE);
    const int wave_m = wave / WAVES_N, wave_n = wave % WAVES_N;
    const int quad = lane / 16;                                // which four rows of a 16 x 16 block of sums this lane holds
    const int upper_blocks = (height / 16 + 1) / 2;            // of 16 rows, of the wavefronts 0 to 3
    const int blocks = wave_m == 0 ? upper_blocks : height / 16 - upper_blocks;
    const int wave_row = m0 + wave_m * upper_blocks * 16, tile_end = min(m0 + height, M);

    // Row of w behind row r of the tile (w not packed). Gated: a wavefront's rows are half gate rows and half the up rows of
    // the same outputs. Rows beyond the operands are clamped to the last one: what they make is not written.
    auto w_row = [&](int r) -> int {
        if constexpr (MODE == MODE_GATED) {
            constexpr int HALF = WAVE_N / 2;
            const int within = r % WAVE_N;
            return min(n0 + (r / WAVE_N) * HALF + within % HALF, N - 1) + (within / HALF) * N;
        } else {
            return min(n0 + r, N - 1);
        }
    };
    // Piece c (16 bytes) of row r of 64 lies at place c ^ (r % 8) of the row. The sixteen lanes that a 16-byte read serves at
    // once are not neighbours (0 to 3, 12 to 15, 20 to 23 and 24 to 27, say): in this order they take 16 different groups of
    // banks (no conflicts counted, 2084 cycles a step; with the order of the smaller tiles 2470).
    auto swizzle_of = [](int r) { return r % 8; };
    // The kilobyte of LDS (8 rows of 64, or a packed tile of 16 rows and 32 columns) that load i of half h fills, for a
    // wavefront; rows: a wavefront's rows of the operand in the tile.
    auto block_of = [&](int h, int i, int rows, int blocks) {
        const int per = rows / 16, p = min(i * 8 + wave, blocks - 1);
        return (p / per * rows + h * (rows / 2)) / 8 + p % per;
    };
    const int row_a = lda > 0 ? lda : K, row_w = ldw > 0 ? ldw : K;
    const bool packed_b = is_packed(packing);
    const int first_packed = MODE == MODE_GATED ? 2 * n0 : n0;
    const int last_group = ((MODE == MODE_GATED ? 2 * N : N) + 15) / 16 - 1;
    unsigned off_a[2][LOADS_A], off_b[2][LOADS_B];             // bytes
    // (rows of the tile that no wavefront has: the last one again, not multiplied)
    const int missing = WAVE_M - upper_blocks * 16;
    const unsigned piece_of_lane = (unsigned)((lane % 8) ^ swizzle_of(lane / 8)) * 16u;        // (rows of further loads differ by multiples of 8)
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int i = 0; i < LOADS_A; ++i) {
            const int block = block_of(h, i, WAVE_M, BLOCKS_A), r = block * 8 + lane / 8;
            const int row = min(m0 + r - (block * 8 >= WAVE_M ? missing : 0), tile_end - 1);
            off_a[h][i] = (unsigned)row * (unsigned)row_a * 2u + piece_of_lane;
        }
    if (packed_b) {
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int i = 0; i < LOADS_B; ++i) {
                const int block = block_of(h, i, WAVE_N, BN / 16);
                const int group = min(first_packed / 16 + block / 2, last_group);          // groups beyond the matrix: the last one again
                off_b[h][i] = ((unsigned)group * (unsigned)(row_w / 32) + (unsigned)(block % 2)) * 1024u + (unsigned)lane * 16u;
            }
    } else {
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int i = 0; i < LOADS_B; ++i) {
                const int r = block_of(h, i, WAVE_N, BN / 16) * 8 + lane / 8;
                off_b[h][i] = (unsigned)w_row(r) * (unsigned)row_w * 2u + piece_of_lane;
            }
    }
    const unsigned w_step = packed_b ? 32u : 2u;               // bytes per column of k
    const unsigned lds_a0 = lds_address(stage_a), lds_b0 = lds_address(stage_b);
    auto issue_a = [&](int h, int stage, int k0) {
#pragma unroll
        for (int i = 0; i < LOADS_A; ++i)
            load_to_lds(a, off_a[h][i] + (unsigned)k0 * 2u, lds_a0 + (unsigned)(stage * BM * DK * 2 + block_of(h, i, WAVE_M, BLOCKS_A) * 1024));
    };
    auto issue_b = [&](int h, int stage, int k0) {
#pragma unroll
        for (int i = 0; i < LOADS_B; ++i)
            load_to_lds(w, off_b[h][i] + (unsigned)k0 * w_step, lds_b0 + (unsigned)(stage * BN * DK * 2 + block_of(h, i, WAVE_N, BN / 16) * 1024));
    };
    // where this lane finds its 16 bytes of block 0 of its wavefront, for either 32 columns of the tile
    const bf16* place_a[2];
    const bf16* place_b[2];
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
        const int piece = ((ks * 4 + quad) ^ swizzle_of(lane % 16)) * 8;                 // (rows of further blocks differ by multiples of 16)
        place_a[ks] = stage_a + (wave_m * WAVE_M + lane % 16) * DK + piece;
        place_b[ks] = stage_b + wave_n * WAVE_N * DK + (packed_b ? ks * 512 + lane * 8 : lane % 16 * DK + piece);
    }
    bf16x8 xa[2][2][HM], wb[2][2][HN];                         // [half][32 columns][block]
    // (T: the blocks of the wavefront, TM or somewhat fewer; they are missing from the second half)
    auto read_a = [&](auto t, int h, int stage) {
        constexpr int T = decltype(t)::value;
#pragma unroll
        for (int ks = 0; ks < 2; ++ks)
#pragma unroll
            for (int i = 0; i < HM; ++i)
                if (h * HM + i < T) xa[h][ks][i] = *reinterpret_cast<const bf16x8*>(place_a[ks] + stage * BM * DK + (h * HM + i) * 16 * DK);
    };
    auto read_b = [&](int h, int stage) {
#pragma unroll
        for (int ks = 0; ks < 2; ++ks)
#pragma unroll
            for (int j = 0; j < HN; ++j)
                wb[h][ks][j] = *reinterpret_cast<const bf16x8*>(place_b[ks] + stage * BN * DK + (h * HN + j) * 16 * DK);
    };
    floatx4 acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) acc[i][j] = floatx4{0.f, 0.f, 0.f, 0.f};
    auto multiply = [&](auto t, int h, int g) {
        constexpr int T = decltype(t)::value;
#pragma unroll
        for (int ks = 0; ks < 2; ++ks)
#pragma unroll
            for (int i = 0; i < HM; ++i)
#pragma unroll
                for (int j = 0; j < HN; ++j)
                    if (h * HM + i < T)
                        acc[h * HM + i][g * HN + j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wb[g][ks][j], xa[h][ks][i], acc[h * HM + i][g * HN + j], 0, 0, 0);
    };
    // part p of a product split along k takes k_per_split from p * k_per_split on (less at the end) and writes its sums to
    // the p-th copy of out
    const int k_begin = part * k_per_split;
    const int steps = min(k_per_split, K - k_begin) / DK;
    const int last_k = k_begin + (steps - 1) * DK;
    out += (long)part * M * N;
    auto k_of = [&](int t) { return min(k_begin + t * DK, last_k); };    // (tiles beyond the end: the last one again, into a place nobody reads)
#pragma unroll
    for (int t = 0; t < 2; ++t) {
        issue_a(0, t, k_of(t));
        issue_b(0, t, k_of(t));
        issue_b(1, t, k_of(t));
        issue_a(1, t, k_of(t));
    }
    // Loads that may stay in flight behind a quarter's reads: those of the six quarters after the next one.
    constexpr int ALL = 2 * (LOADS_A + LOADS_B);
    auto barrier = [] {
        __builtin_amdgcn_sched_barrier(0);
        asm volatile("s_barrier" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
    };
    auto walk = [&](auto t_blocks) {
        wait_loads_and_barrier<ALL + LOADS_A + LOADS_B>();     // x0 and w0 of tile 0 are in LDS
        read_a(t_blocks, 0, 0);
        wait_loads_and_barrier<ALL + LOADS_A + LOADS_B>();     // and x0 is read by all: the first turn fills its place again
        auto turn = [&](auto in_flight, int h, int g) {
            __builtin_amdgcn_sched_barrier(0);
            wait_loads_and_barrier<decltype(in_flight)::value>();  // this wavefront's reads are done: what it read may be overwritten
            __builtin_amdgcn_sched_barrier(0);
            multiply(t_blocks, h, g);
            barrier();
        };
        if (wave >= 4) barrier();
        for (int t = 0; t < steps; ++t) {
            const int now = t % 2, k_next = k_of(t + 2);
            read_b(0, now);
            issue_a(0, now, k_next);
            turn(std::integral_constant<int, ALL + 2 * LOADS_A>{}, 0, 0);           // in flight: x1 x0 w0 w1 x1 x0
            read_b(1, now);
            issue_b(0, now, k_next);
            turn(std::integral_constant<int, ALL + LOADS_A + LOADS_B>{}, 0, 1);     // x0 w0 w1 x1 x0 w0
            read_a(t_blocks, 1, now);
            issue_b(1, now, k_next);
            turn(std::integral_constant<int, ALL + 2 * LOADS_B>{}, 1, 1);           // w0 w1 x1 x0 w0 w1
            read_a(t_blocks, 0, now ^ 1);
            issue_a(1, now, k_next);
            turn(std::integral_constant<int, ALL + LOADS_A + LOADS_B>{}, 1, 0);     // w1 x1 x0 w0 w1 x1
        }
    };
    // (tiles of up to 128 rows always run the whole loop: the way round the others, cold code, took 0.3 us of 17, and fewer products gained none)
    if (BM == 128 || blocks == TM) walk(std::integral_constant<int, TM>{});
    else if (blocks == TM - 1) walk(std::integral_constant<int, TM - 1>{});
    else walk(std::integral_constant<int, TM - 2>{});          // (fewer than that: some products that nobody writes)
    if (wave < 4) barrier();
    wait_loads_and_barrier<0>();                               // nothing lands in LDS after this

    // ---- epilogue: element e of acc[i][j] is row i * 16 + lane % 16 of x and row j * 16 + quad * 4 + e of w
    const int row0 = wave_row + lane % 16;
    const int row_end = min(wave_row + blocks * 16, tile_end);           // of the wavefront's rows
    if (MODE == MODE_GATED && packed_b) {
        // A group of 16 packed rows holds the gate rows of 8 outputs, then their up rows: the lane with an output's up sum
        // is 32 lanes away. One exchange of half a register between the sums of two blocks of x leaves gate and up of
        // every output of both in one lane (lanes 0 to 31 the first block's outputs, the others the second's); for
        // bfloat16 another one between two groups of w brings eight neighbouring outputs together: 16 bytes a store.
        const long n_wave = n0 + wave_n * (WAVE_N / 2);
        const bool wide = N % 8 == 0 && (uintptr_t)out % 16 == 0;
#pragma unroll
        for (int i = 0; i < TM; i += 2) {
            const long m = row0 + i * 16 + lane / 32 * 16;
#pragma unroll
            for (int j = 0; j < TN; j += 2) {
                float made[2][4];
#pragma unroll
                for (int u = 0; u < 2; ++u)
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        float gate = acc[i][j + u][e], up = acc[i + 1][j + u][e];
                        exchange_halves(gate, up);
                        made[u][e] = gate_activation<sizeof(TO) == 2>(gate, activation) * up;
                    }
                if constexpr (sizeof(TO) == 2) {
                    if (wide) {
                        uint4v piece = join_rows<TO>(made[0], made[1]);
                        const long n = n_wave + (j + quad % 2) * 8;
                        if (m < row_end && n < N) *reinterpret_cast<uint4v*>(out + m * (long)N + n) = piece;
                        continue;
                    }
                }
#pragma unroll
                for (int u = 0; u < 2; ++u)
                    store_four<TO>(out, m, n_wave + (j + u) * 8 + quad % 2 * 4, row_end, N, made[u], wide);
            }
        }
    } else if constexpr (MODE == MODE_GATED) {
        const bool wide = N % 4 == 0 && (uintptr_t)out % 16 == 0;
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < HN; ++j) {
                float made[4];
#pragma unroll
                for (int e = 0; e < 4; ++e) made[e] = gate_activation<sizeof(TO) == 2>(acc[i][j][e], activation) * acc[i][j + HN][e];
                store_four<TO>(out, row0 + i * 16, n0 + wave_n * (WAVE_N / 2) + j * 16 + quad * 4, row_end, N, made, wide);
            }
    } else {
        const bool wide = N % 8 == 0 && (uintptr_t)out % 16 == 0;
        // The output column behind packed row q of w. Every order of packed rows keeps runs of eight together.
        auto column_of = [&](long q) -> long { return packed_b && q < N ? logical_row(packing, q) : q; };
        // Two neighbouring blocks of columns change eight lanes with each other, so that an instruction takes eight rows of
        // 128 bytes, whole cache lines, instead of sixteen of 64 (adding onto a float32 residual of 8192 x 4096: 54 instead of 17
        // microseconds a round of tiles without it).
        const long row8 = wave_row + lane % 8;
        const int upper = lane % 16 / 8;
        if constexpr (MODE == MODE_STORE && sizeof(TO) == 2) {
            if (wide) {
                static_assert(TN == 4, "two pieces of 32 columns");
                const long q = n0 + wave_n * WAVE_N + (2 * upper + quad % 2) * 16 + quad / 2 * 8, n = column_of(q);
#pragma unroll
                for (int i = 0; i < TM; ++i) {
                    uint4v piece[2];
#pragma unroll
                    for (int u = 0; u < 2; ++u) {
                        const floatx4 x = acc[i][2 * u], y = acc[i][2 * u + 1];
                        const float first[4] = {x[0], x[1], x[2], x[3]}, second[4] = {y[0], y[1], y[2], y[3]};
                        piece[u] = join_rows<TO>(first, second);
                    }
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        unsigned low = piece[0][e], high = piece[1][e];
                        exchange_eights(low, high);
                        piece[0][e] = low;
                        piece[1][e] = high;
                    }
#pragma unroll
                    for (int u = 0; u < 2; ++u) {
                        const long m = row8 + i * 16 + u * 8;
                        if (m < row_end && q < N) *reinterpret_cast<uint4v*>(out + m * (long)N + n) = piece[u];
                    }
                }
                return;
            }
        }
        constexpr int RUN = TM % 4 == 0 ? 4 : 3;               // blocks of x whose old values are read in one go, before any is written
#pragma unroll
        for (int i0 = 0; i0 < TM; i0 += RUN) {
            float before[RUN][TN][4];
            if constexpr (MODE == MODE_ACCUMULATE) {
#pragma unroll
                for (int i = 0; i < RUN; ++i)
#pragma unroll
                    for (int j = 0; j < TN; ++j)
                        load_four<TO>(out, row8 + (i0 + i) * 16 + j % 2 * 8, column_of(n0 + wave_n * WAVE_N + (j / 2 * 2 + upper) * 16 + quad * 4),
                                      row_end, N, before[i][j], wide);
            }
#pragma unroll
            for (int i = 0; i < RUN; ++i)
#pragma unroll
                for (int j = 0; j < TN; j += 2) {
                    float made[2][4];
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        made[0][e] = acc[i0 + i][j][e];
                        made[1][e] = acc[i0 + i][j + 1][e];
                        exchange_eights(made[0][e], made[1][e]);
                        if constexpr (MODE == MODE_ACCUMULATE) {
                            made[0][e] = before[i][j][e] + made[0][e];
                            made[1][e] = before[i][j + 1][e] + made[1][e];
                        }
                    }
                    const long q = n0 + wave_n * WAVE_N + (j + upper) * 16 + quad * 4;
                    if (q < N) {
                        const long n = column_of(q);
                        store_four<TO>(out, row8 + (i0 + i) * 16, n, row_end, N, made[0], wide);
                        store_four<TO>(out, row8 + (i0 + i) * 16 + 8, n, row_end, N, made[1], wide);
                    }
                }
        }
    }
}

// PARTS: k may be split (without it the way to the first loads is shorter).
template <int BM, int MODE, typename TO, bool PARTS>
__global__ void __launch_bounds__(8 * XRT_WAVE) gemm_large_kernel(
    const bf16* __restrict__ a, const bf16* __restrict__ w, TO* __restrict__ out, int M, int N, int K,
    int tiles_m, int tiles_n, int by_parts, int k_per_split, const Packing packing, int activation, int height) {
    const PartPlace place = PARTS ? part_place(blockIdx.x, blockIdx.y, tiles_m, tiles_n, by_parts) : PartPlace{tile_place(blockIdx.x, tiles_m, tiles_n), 0};
    if (place.tile.m < 0) return;
    gemm_large_tile<BM, MODE, TO>(a, w, out, M, N, K, place.tile, 0, place.part, k_per_split, packing, activation, height);
}

template <int BM, int BN, int WM, int WN, int MODE, int DK, int STAGES, typename TO, bool PAST_CACHES>
__global__ void __launch_bounds__(WM * WN * XRT_WAVE) gemm_mfma_kernel(
    const bf16* __restrict__ a, const bf16* __restrict__ w, TO* __restrict__ out, int M, int N, int K,
    int tiles_m, int tiles_n, int by_parts, int k_per_split, const Packing packing, const RowScale scale) {
    gemm_tile<BM, BN, WM, WN, MODE, DK, STAGES, TO, PAST_CACHES>(a, w, out, M, N, K, blockIdx.x, tiles_m, tiles_n, by_parts, k_per_split, packing, scale);
}

// Two tile shapes in one launch: the first `large_blocks` workgroups take 256 x 256 tiles of the
// output columns below `split`, the others 128 x 256 tiles of the columns from `split` on. The
// large tiles are handed out first and fill whole rounds over the compute units; the small ones
// follow as compute units become free, so the last round is full of half-sized work and there is
// no gap between the two.
template <int MODE, typename TO>
__global__ void __launch_bounds__(8 * XRT_WAVE) gemm_mfma_mixed_kernel(
    const bf16* __restrict__ a, const bf16* __restrict__ w, TO* __restrict__ out, int M, int N, int K,
    int large_blocks, int large_tiles_m, int large_tiles_n, int split, int small_tiles_m, int small_tiles_n,
    const Packing packing, int activation, int large_height, int small_height) {
    if ((int)blockIdx.x < large_blocks) {
        const TilePlace place = tile_place(blockIdx.x, large_tiles_m, large_tiles_n);
        if (place.m >= 0) gemm_large_tile<256, MODE, TO>(a, w, out, M, N, K, place, 0, 0, K, packing, activation, large_height);
    } else {
        const TilePlace place = tile_place(blockIdx.x - large_blocks, small_tiles_m, small_tiles_n);
        if (place.m >= 0) gemm_large_tile<128, MODE, TO>(a, w, out, M, N, K, place, split, 0, K, packing, activation, small_height);
    }
}

// Products of groups of rows with matrices of their own (experts): the rows of a stand sorted by group, every group's stretch
// filled up to whole tiles of BM rows (128, or 256 where the groups are long: the larger tile multiplies half as fast again,
// and fills up more), and tile_group[t] names the group of tile t (negative: the tile holds nothing and
// its workgroups leave). Group g multiplies with w + g * w_stride; a's rows lie lda apart, w's ldw (so a group's matrix can be
// some columns of a wider one), K is what is summed over. Grid: x the tiles along n (a whole number of rounds over the XCDs,
// so that all tiles of one n and one group, which share their w, run on one XCD), y the parts that k is split into (each
// writes its sums to a copy of the tile's outputs: out is [tiles][parts][BM][N] then), z the tiles of rows.
template <int BM, int MODE, typename TO>
__global__ void __launch_bounds__(8 * XRT_WAVE) gemm_grouped_kernel(
    const bf16* __restrict__ a, const bf16* __restrict__ w, long w_stride, TO* __restrict__ out, int N, int K, int lda, int ldw,
    int tiles_n, const int* __restrict__ tile_group, const Packing packing, int activation) {
    const int tile = blockIdx.z;
    const int group = tile_group == nullptr ? 0 : tile_group[tile];      // (no table: one matrix for all tiles)
    if (group < 0) return;
    // (grid rows split k among them, and the tile puts row y's sums BM * N elements further on: a tile's parts lie one
    // after the other, tile after tile)
    const TilePlace place = tile_place(blockIdx.x, 1, tiles_n);
    if (place.m < 0) return;
    gemm_large_tile<BM, MODE, TO>(a + (long)tile * BM * lda, w + (long)group * w_stride, out + (long)tile * gridDim.y * BM * N, BM, N, K, place,
                                  0, (int)blockIdx.y, K / (int)gridDim.y, packing, activation, BM, lda, ldw);
}

template <int BM, int MODE, typename TO>
int launch_grouped(const bf16* a, const bf16* w, long w_stride, TO* out, int tiles_m, int N, int K, int lda, int ldw, const int* tile_group,
                   const Packing& packing, int activation, int splits, hipStream_t s) {
    constexpr int BN_OUT = MODE == MODE_GATED ? LARGE_BN / 2 : LARGE_BN;
    constexpr size_t lds = (size_t)2 * (BM + LARGE_BN) * 64 * sizeof(bf16);
    auto kernel = gemm_grouped_kernel<BM, MODE, TO>;
    static bool configured = false;          // per instantiation
    if (!configured) {
        hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        XRT_REQUIRE(e == hipSuccess, "linear (groups): cannot reserve %zu bytes of LDS: %s", lds, hipGetErrorString(e));
        configured = true;
    }
    const int tiles_n = (N + BN_OUT - 1) / BN_OUT;
    XRT_REQUIRE(tiles_m > 0 && tiles_m <= 65535, "linear (groups): %d tiles of rows", tiles_m);
    XRT_REQUIRE(splits >= 1 && K % (64 * splits) == 0 && (splits == 1 || MODE == MODE_STORE), "linear (groups): k in %d parts", splits);
    kernel<<<dim3((unsigned)((tiles_n + 7) / 8 * 8), (unsigned)splits, (unsigned)tiles_m), 8 * XRT_WAVE, lds, s>>>(
        a, w, w_stride, out, N, K, lda, ldw, tiles_n, tile_group, packing, activation);
    XRT_LAUNCH_CHECK("linear (groups)");
    return 0;
}

template <int BM>
int launch_grouped_of(const bf16* x, const bf16* m, long w_stride, void* out, int out_dtype, int tiles_m, int N, int K, int lda, int ldw,
                      const int* tile_group, const Packing& packing, int mode, int activation, int splits, hipStream_t s) {
    if (mode == MODE_GATED) {
        if (out_dtype == XRT_F32) return launch_grouped<BM, MODE_GATED, float>(x, m, w_stride, (float*)out, tiles_m, N, K, lda, ldw, tile_group, packing, activation, splits, s);
        return launch_grouped<BM, MODE_GATED, bf16>(x, m, w_stride, (bf16*)out, tiles_m, N, K, lda, ldw, tile_group, packing, activation, splits, s);
    }
    if (out_dtype == XRT_F32) return launch_grouped<BM, MODE_STORE, float>(x, m, w_stride, (float*)out, tiles_m, N, K, lda, ldw, tile_group, packing, activation, splits, s);
    return launch_grouped<BM, MODE_STORE, bf16>(x, m, w_stride, (bf16*)out, tiles_m, N, K, lda, ldw, tile_group, packing, activation, splits, s);
}

// One row of tiles, k not split: every byte of w is read by one workgroup, in one long run, and is asked for past the caches
// where it cannot stay in the last one (256 MB) until the next step. (Among other matrices, 64 rows: gate/up of 28672 rows
// of w and k = 4096 46.6 -> 44.1 us, an output head of 128256 rows and k = 2048 105.0 -> 98.5. A w that does stay is read faster from
// there: 17408 rows and k = 1024, 214 MB of such matrices in turn, 11.3 us as it is, 12.8 past the caches.) A gated matrix counts one
// and a half times: a model has the one back from that width too. Split along k the runs are short, and so marked they are
// read more slowly (4096 x 4096 in eight parts 16.3 -> 18.1 us).
// The gated tiles of up to 256 rows of a in several stages the same (700 products drawn at random, past the caches against through them: a w too large to stay
// 0.95 to 0.99 with one row of tiles; matrices of 60 MB in turn 1.02 to 1.08 in tiles of 64 x 64, 1.09 to 1.25 in the others, up to 1.5; with two rows of
// tiles, the second of which reads what the first has brought, 1.03 to 1.2 whatever w).
constexpr long LAST_CACHE = 256L << 20;
bool cannot_stay(long rows_w, int K, int halves) { return rows_w * K * (long)sizeof(bf16) / 2 * halves > LAST_CACHE; }      // halves: what it counts, in half matrices
bool reads_past_caches(int rows_of_tile, int M, int N, int K, int mode) {
    return M <= rows_of_tile && (mode == MODE_GATED ? cannot_stay(2L * N, K, 3) : cannot_stay(N, K, 2));
}

// Whether the tiles and parts of a product are dealt by parts (part_place): where k is so long that reading all of a on every XCD costs (tiles of 256 rows
// of w read it less often, and gain from k = 3072 on: 0.95 of the time by columns beyond k = 6144, 0.97 to 0.98 below; narrower ones 0.97 beyond k = 6144, and 1.01
// below, where an XCD's parts touch the pages of all of w for little), and where it makes a round less (0.79 to 0.94 up to 64 rows of x).
// Not in narrower tiles where the rows of tiles are many, unless each XCD gets a part of its own (8 parts): several XCDs' runs of a part then go down all of a, whose slice their
// L2 does not hold, for few columns, and by columns they read an eighth of it each. 1300 products drawn, both ways timed: tiles of 64 rows of w up to 12 rows of tiles 0.93 (none above
// 1.05), beyond that 1.14 (up to 1.7); of 128 up to 16 rows 0.95 (2 above 1.05), beyond that 1.05 (up to 1.2: 4548 rows of x, 144 pairs, k = 14976 67 -> 80 us); with 8 parts 0.95
// there too; of 256 0.96 throughout.
bool deals_by_parts(int columns, long tiles_m, long tiles_n, int K, int parts) {
    if (parts < 2 || (columns < 256 && tiles_m > (columns == 64 ? 12 : 16) && parts % 8 != 0)) return false;
    auto rounds = [](long groups) { return (groups + XRT_COMPUTE_UNITS - 1) / XRT_COMPUTE_UNITS; };
    return K > (columns >= 256 ? 2048 : 6144) || rounds(part_ids(tiles_m * tiles_n, parts, false)) > rounds(part_ids(tiles_m * tiles_n, parts, true));
}

template <int BM, int BN, int WM, int WN, int MODE, int DK, int STAGES, typename TO, bool PAST_CACHES = false>
int launch_kernel(const bf16* a, const bf16* w, TO* out, int M, int N, int K, const Packing& packing,
                  hipStream_t s, int splits = 1, int k_per_split = 0, const RowScale scale = RowScale{}) {
    if constexpr ((BM <= 64 || (MODE == MODE_GATED && STAGES > 2)) && !PAST_CACHES)
        if (splits == 1 && reads_past_caches(BM, M, N, K, MODE))
            return launch_kernel<BM, BN, WM, WN, MODE, DK, STAGES, TO, true>(a, w, out, M, N, K, packing, s, splits, k_per_split, scale);
    constexpr int BN_OUT = MODE == MODE_GATED ? BN / 2 : BN;
    constexpr int THREADS = WM * WN * XRT_WAVE;
    constexpr size_t staging = DK != 0 ? (size_t)STAGES * (BM + BN) * DK * sizeof(bf16) : (size_t)2 * (BM + BN) * PITCH * sizeof(bf16);
    constexpr size_t lds = staging;
    static_assert(lds <= 160 * 1024, "tile does not fit the LDS of a compute unit");
    auto kernel = gemm_mfma_kernel<BM, BN, WM, WN, MODE, DK, STAGES, TO, PAST_CACHES>;
    static bool configured = false;          // per instantiation
    if (!configured) {
        hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        XRT_REQUIRE(e == hipSuccess, "linear (mfma): cannot reserve %zu bytes of LDS: %s", lds, hipGetErrorString(e));
        configured = true;
    }
    const int tiles_m = (M + BM - 1) / BM, tiles_n = (N + BN_OUT - 1) / BN_OUT;
    const bool by_parts = deals_by_parts(BN, tiles_m, tiles_n, K, splits);
    const long ids = part_ids((long)tiles_m * tiles_n, by_parts ? splits : 1, by_parts);         // a whole number of rounds over the XCDs
    XRT_REQUIRE(ids < (1L << 31), "linear (mfma): %ld tiles", ids);
    XRT_REQUIRE(splits == 1 || DK != 0, "linear (mfma): only whole tiles along k can be split");
    XRT_REQUIRE(scale.squares == nullptr || (BM <= 64 && splits == 1), "linear (mfma): rows are scaled by tiles of up to 64 rows that see all of k");
    kernel<<<dim3((unsigned)ids, by_parts ? 1 : splits), THREADS, lds, s>>>(a, w, out, M, N, K, tiles_m, tiles_n, by_parts ? splits : 0, splits == 1 ? K : k_per_split,
                                                                            packing, scale);
    XRT_LAUNCH_CHECK("linear (mfma)");
    return 0;
}

// The rows of a of each tile, where tiles of up to `most` rows (a multiple of 16) share M.
int even_height(int M, int most) {
    const int tiles = (M + most - 1) / most;
    return ((M + tiles - 1) / tiles + 15) / 16 * 16;
}

// The large tiles over all of w; splits > 1: k dealt out among grid rows, each with its copy of out.
template <int BM, int MODE, typename TO, bool PARTS = false>
int launch_large(const bf16* a, const bf16* w, TO* out, int M, int N, int K, const Packing& packing, int activation, hipStream_t s,
                 int splits = 1, int k_per_split = 0) {
    constexpr int BN_OUT = MODE == MODE_GATED ? LARGE_BN / 2 : LARGE_BN;
    constexpr size_t lds = (size_t)2 * (BM + LARGE_BN) * 64 * sizeof(bf16);
    auto kernel = gemm_large_kernel<BM, MODE, TO, PARTS>;
    static bool configured = false;          // per instantiation
    if (!configured) {
        hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        XRT_REQUIRE(e == hipSuccess, "linear (mfma): cannot reserve %zu bytes of LDS: %s", lds, hipGetErrorString(e));
        configured = true;
    }
    XRT_REQUIRE(K % 64 == 0 && (splits == 1 || (PARTS && k_per_split % 64 == 0)), "linear (mfma): the large tiles take whole steps of 64 along k (K=%d)", K);
    const int tiles_m = (M + BM - 1) / BM, tiles_n = (N + BN_OUT - 1) / BN_OUT;
    const bool by_parts = deals_by_parts(LARGE_BN, tiles_m, tiles_n, K, splits);
    const long ids = part_ids((long)tiles_m * tiles_n, by_parts ? splits : 1, by_parts);         // a whole number of rounds over the XCDs
    XRT_REQUIRE(ids < (1L << 31), "linear (mfma): %ld tiles", ids);
    kernel<<<dim3((unsigned)ids, by_parts ? 1 : splits), 8 * XRT_WAVE, lds, s>>>(a, w, out, M, N, K, tiles_m, tiles_n, by_parts ? splits : 0, splits == 1 ? K : k_per_split,
                                                                                 packing, activation, even_height(M, BM));
    XRT_LAUNCH_CHECK("linear (mfma, large tiles)");
    return 0;
}

// What a tile shape costs: a full round over `places` takes `products` microseconds for each 4096 of k and ends[kind] for its
// first loads and its epilogue. A last round that is partly filled takes `least` percent of a full one and its share of the
// rest: the chip is bound by its power, and with fewer compute units at work their clock rises. The numbers are fitted to 1985
// products (layers of seven sizes and sizes drawn at random, k from 64 to 25600, 129 to 8192 rows of x), every tile shape of
// each of them timed: what the estimate chooses is 0.6 % off the best of them on average, which is within the runs' differences. (The tiles of 192 rows came later,
// fitted to 90 gated products: 28672 rows of w, k = 4096, 333 rows of x 90 -> 76 us, 1100 rows 234 -> 213; 16384 rows, k = 2048, 540 rows 46 -> 38; 51200
// rows, k = 5120, 576 rows 317 -> 279. Of products of every kind drawn at random afterwards those that take them now take 0.92 of what they took, storing 46
// of them, 0.93, adding, 8, 0.9, gated, 17; none takes more than 1.02.)
enum { ENDS_BF16 = 0, ENDS_F32 = 1, ENDS_ADDING = 2, ENDS_GATED = 3 };
struct TileTime { int bm, bn, places, products, ends[4], least; };
constexpr TileTime LARGE_TILE = {256, 256, XRT_COMPUTE_UNITS, 88, {10, 16, 15, 16}, 55}, HALF_TILE = {128, 256, XRT_COMPUTE_UNITS, 54, {6, 8, 9, 9}, 62},
                   MIDDLE_TILE = {192, 256, XRT_COMPUTE_UNITS, 71, {8, 13, 12, 13}, 55}, NARROW_TILE = {256, 192, XRT_COMPUTE_UNITS, 81, {0, 11, 8, 0}, 55}, SMALL_TILE = {128, 128, 2 * XRT_COMPUTE_UNITS, 67, {7, 7, 5, 10}, 41};
long rounds_cost(long tiles, const TileTime& tile, int K, int kind) {        // in nanoseconds or so
    const long round = tile.products * 1000L * K / 4096 + tile.ends[kind] * 1000L;
    const long whole = tiles / tile.places, rest = tiles % tile.places;
    return whole * round + (rest == 0 ? 0 : (tile.least * (long)tile.places + (100 - tile.least) * rest) * round / (100L * tile.places));
}

// The tiles of a product without a split along k: rows of a by rows of w, and beside them the stages where there is more than one choice.
enum TileShape { TILES_256, TILES_192, TILES_128, TILES_256_AND_128, TILES_256_BY_192, TILES_128_BY_128, TILES_128_BY_128_THREE_STAGES, TILES_128_BY_64_FOUR_STAGES,
                 TILES_RAGGED_256, TILES_RAGGED_128 };
// whole_columns: of TILES_256_AND_128, the tiles along the columns that are 256 rows high.
template <int MODE, typename TO>
TileShape tile_shape(int M, int N, int K, int* whole_columns) {
    // output columns per tile are half the tile's w rows in the gated mode
    constexpr int DIV = MODE == MODE_GATED ? 2 : 1;
    auto tiles = [&](int bm, int bn) { return (long)((M + bm - 1) / bm) * ((N + bn / DIV - 1) / (bn / DIV)); };
    if (K % 64 != 0) {                 // a ragged last tile along k: the path through registers
        const long large = ((tiles(256, 256) + XRT_COMPUTE_UNITS - 1) / XRT_COMPUTE_UNITS) * 100;
        const long small = ((tiles(128, 128) + 2 * XRT_COMPUTE_UNITS - 1) / (2 * XRT_COMPUTE_UNITS)) * 59;
        return large <= small ? TILES_RAGGED_256 : TILES_RAGGED_128;
    }
    // Up to 256 rows of a, gated: tiles that fit one round and are bound by reading w, in three or four stages, which keep more of it on
    // its way than the two that the tiles below have. (Split along k with a second kernel: 3072 pairs, k = 1024, 100 rows 14.6 us, so 9.5, 256 rows
    // 17.8 -> 9.9; 8192 pairs, k = 2048, 100 rows 24.4 -> 19.9, 200 rows 31.2 -> 24.7; 12288 pairs, k = 4096, 100 rows 59.6 -> 50.9; 5000 pairs,
    // k = 3072, 65 rows 28.8 -> 21.8. Tiles of 128 x 64 beyond one round lose to one of 128 x 128: 12288 pairs, 100 rows 55.7.)
    if constexpr (MODE == MODE_GATED) {
        if (M <= 256 && tiles(128, 64) <= XRT_COMPUTE_UNITS) return TILES_128_BY_64_FOUR_STAGES;
        if (M <= 128 || (M <= 256 && tiles(128, 128) <= XRT_COMPUTE_UNITS)) return TILES_128_BY_128_THREE_STAGES;
    }
    // 256 x 256 tiles cost the least energy a product, and tiles of half the height somewhat more (2048 rows of x, 4096 rows of
    // w, k = 4096: 128 tiles of the one 85 us, 256 of the other 58; 6144 rows of w: 82 and 102); tiles of 128 x 128, two to a compute
    // unit, where neither fills the chip, or where k is so short that one's epilogue wants another's products beside it (200 rows of x,
    // 9632 rows of w, k = 1728, adding: 25 against 31 us). The tiles of 256 x 192, which are gemm_tile's, where they make one round that
    // the large ones leave half empty and those of half the height need two for, and results are float32, which they write faster
    // (adding, 3072 rows of w, k = 3072, 2816 rows of x: 63 against 73 and 90 us; 4096 rows, k = 14336, 2300 rows of x: 250, 259 and
    // 327; bfloat16 results, 3072 rows, k = 2048, 2048 rows of x: 53 against 46 us). They read their operands more often, which a w
    // beyond the caches does not stand (5120 rows of w, k = 25600, 2048 rows of x: 572 against 447 us; 13536 rows, k = 10624,
    // 724 rows of x: 240 against 188).
    constexpr long NARROW_W = 150L * 1000 * 1000;              // bytes
    constexpr int KIND = MODE == MODE_GATED ? ENDS_GATED : MODE == MODE_ACCUMULATE ? ENDS_ADDING : sizeof(TO) == 4 ? ENDS_F32 : ENDS_BF16;
    auto cost = [&](const TileTime& tile) { return rounds_cost(tiles(tile.bm, tile.bn), tile, K, KIND); };
    const long large = cost(LARGE_TILE), middle = cost(MIDDLE_TILE), half = cost(HALF_TILE), small = cost(SMALL_TILE);
    constexpr bool NARROW = MODE != MODE_GATED && sizeof(TO) == 4;
    const long narrow = NARROW && (long)N * K * (long)sizeof(bf16) <= NARROW_W ? cost(NARROW_TILE) : LONG_MAX;
    // Large tiles for as many columns as make whole rounds, and tiles of half the height for the rest, if those then fit
    // one round: the last round is full of half-sized work instead of half empty (28672 rows of w, k = 4096, 2048 rows of x:
    // 366 against 372 us).
    const int tiles_m = (M + 255) / 256, tiles_n = (N + 256 / DIV - 1) / (256 / DIV);
    *whole_columns = (int)((long)tiles_m * tiles_n / XRT_COMPUTE_UNITS * XRT_COMPUTE_UNITS / tiles_m);     // n-tiles that run in full rounds
    const long rest_tiles = (long)((M + 127) / 128) * (tiles_n - *whole_columns);
    long mixed = LONG_MAX;
    if (*whole_columns > 0 && *whole_columns < tiles_n && rest_tiles <= XRT_COMPUTE_UNITS)
        mixed = rounds_cost((long)tiles_m * *whole_columns, LARGE_TILE, K, KIND) + rounds_cost(rest_tiles, HALF_TILE, K, KIND);
    if (mixed < large && mixed <= middle && mixed <= half && mixed <= small && mixed <= narrow) return TILES_256_AND_128;
    if (large <= middle && large <= half && large <= small && large <= narrow) return TILES_256;
    if (middle <= half && middle <= small && middle <= narrow) return TILES_192;
    if (half <= small && half <= narrow) return TILES_128;
    if (NARROW && narrow <= small) return TILES_256_BY_192;
    return TILES_128_BY_128;           // (four stages of 32 keep a load in flight for longer but meet at twice as many barriers, and measured slower)
}

template <int MODE, typename TO>
int launch_mode(const bf16* a, const bf16* w, TO* out, int M, int N, int K, const Packing& packing, int activation, hipStream_t s) {
    constexpr int DIV = MODE == MODE_GATED ? 2 : 1;
    const RowScale plain = {nullptr, 0, 0, 0.f, activation};
    int whole_columns = 0;
    switch (tile_shape<MODE, TO>(M, N, K, &whole_columns)) {
        case TILES_RAGGED_256: return launch_kernel<256, 256, 2, 4, MODE, 0, 0, TO>(a, w, out, M, N, K, packing, s, 1, 0, plain);
        case TILES_RAGGED_128: return launch_kernel<128, 128, 2, 2, MODE, 0, 0, TO>(a, w, out, M, N, K, packing, s, 1, 0, plain);
        case TILES_128_BY_64_FOUR_STAGES:
            if constexpr (MODE == MODE_GATED) return launch_kernel<128, 64, 4, 1, MODE, 64, 4, TO>(a, w, out, M, N, K, packing, s, 1, 0, plain);
            break;
        case TILES_128_BY_128_THREE_STAGES:
            // (eight wavefronts: 66 such products drawn at random take 0.92 of what they take in four, the slowest 1.02; 14336 pairs, k = 4096, 100 rows 51.6
            // -> 50.1 us, 25600 pairs, k = 5120 121 -> 118)
            if constexpr (MODE == MODE_GATED) return launch_kernel<128, 128, 4, 2, MODE, 64, 3, TO>(a, w, out, M, N, K, packing, s, 1, 0, plain);
            break;
        case TILES_256: return launch_large<256, MODE, TO>(a, w, out, M, N, K, packing, activation, s);
        case TILES_192: return launch_large<192, MODE, TO>(a, w, out, M, N, K, packing, activation, s);
        case TILES_128: return launch_large<128, MODE, TO>(a, w, out, M, N, K, packing, activation, s);
        case TILES_256_BY_192:
            if constexpr (MODE != MODE_GATED && sizeof(TO) == 4) return launch_kernel<256, 192, 4, 2, MODE, 64, 2, TO>(a, w, out, M, N, K, packing, s, 1, 0, plain);
            break;
        case TILES_128_BY_128: return launch_kernel<128, 128, 2, 2, MODE, 64, 2, TO>(a, w, out, M, N, K, packing, s, 1, 0, plain);
        case TILES_256_AND_128: break;
    }
    const int tiles_m = (M + 255) / 256, tiles_n = (N + 256 / DIV - 1) / (256 / DIV);
    const int split = whole_columns * (256 / DIV);
    const int small_tiles_m = (M + 127) / 128, small_tiles_n = tiles_n - whole_columns;
    const int large_blocks = (tiles_m * whole_columns + 7) / 8 * 8;      // whole rounds over the XCDs
    const int small_blocks = (small_tiles_m * small_tiles_n + 7) / 8 * 8;
    constexpr size_t lds = (size_t)2 * (256 + 256) * 64 * sizeof(bf16);
    auto kernel = gemm_mfma_mixed_kernel<MODE, TO>;
    static bool configured = false;      // per instantiation
    if (!configured) {
        hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        XRT_REQUIRE(e == hipSuccess, "linear (mfma): cannot reserve %zu bytes of LDS: %s", lds, hipGetErrorString(e));
        configured = true;
    }
    kernel<<<large_blocks + small_blocks, 8 * XRT_WAVE, lds, s>>>(a, w, out, M, N, K, large_blocks, tiles_m, whole_columns,
                                                                  split, small_tiles_m, small_tiles_n, packing, activation, even_height(M, 256), even_height(M, 128));
    XRT_LAUNCH_CHECK("linear (mfma, two tile shapes)");
    return 0;
}

template <typename TO>
int launch_shape(const bf16* a, const bf16* w, TO* out, int M, int N, int K, int mode, int activation, const Packing& packing, hipStream_t s) {
    if (mode == MODE_STORE) return launch_mode<MODE_STORE, TO>(a, w, out, M, N, K, packing, activation, s);
    if (mode == MODE_ACCUMULATE) return launch_mode<MODE_ACCUMULATE, TO>(a, w, out, M, N, K, packing, activation, s);
    return launch_mode<MODE_GATED, TO>(a, w, out, M, N, K, packing, activation, s);
}

// ---- 17 to 64 rows of x: too many for the kernel that streams w through registers (it would read
// x from L2 up to four times as often as w from HBM), too few for the tiles above to fill the chip.
// Tiles of 64 x 128 take their x through LDS; k is split among workgroups as far as every compute
// unit still gets at most one of them (one long stream per unit pulls w faster than several short
// ones, measured); each writes float32 sums of its part of k to a workspace, and a second kernel
// adds the parts in order and applies the epilogue. Where w has tiles enough without a split, the
// tiles apply the epilogue themselves and there is no second kernel.
// With more rows of x (up to a few hundred) the tiles of 128 x 128 do the same when they are too
// few to fill the chip: such products are still bound by reading w.
constexpr int SPLIT_BM = 64, SPLIT_BN = 128;

struct SplitPlan { int splits, k_per_split; long rows_w; int tile, columns; };      // tile: rows of x per tile (64, 128, 192 or 256), columns: rows of w

// What a product of some hundred rows of x takes (nanoseconds) in parts along k, if it is gated (of others: the plan of few parts, and what the estimate
// below has to beat): tiles of 128 rows of x and `columns` rows of w, `places` of them to a compute unit. A step of 64 along k takes `step`, `share` more
// for each tile that a compute unit has on average, and `beside` more where some have two; `once` is start, end and the second kernel's start, `part` what a
// further part costs it, `sums` what a million partial sums cost to write and to read again. (Fitted to products of every kind, 512 to 8192 rows of w, k
// from 512 to 14336, 65 to 1700 rows of x; of 2686 gated products drawn at random afterwards what it chooses is 0.9 % off the best of 27 on average.)
// Workgroups are counted as the fullest die has them when they are dealt by columns, as all were when this was fitted: their number alone put two rounds on
// seven of the eight dies where the tiles are no multiple of eight (298 rows of x, 5328 rows of w in pairs, k = 9664: 77 us, 55 by the rule before this
// estimate). Dealt by parts they would make one now, and are still charged two. Charged as they are dealt, with the figures as they are, 300 gated products
// whose cut that changes took 0.99 of their time, but 85 of them over 1.05 (up to 1.21: tiles of 128 where parts of 192 rows are better), so it stays.
struct PartTime { int columns, places, once, step, share, beside, part, sums; };
constexpr int DIES = 8;
// Tiles dealt to the dies by columns come in equal runs, the same in every part: what the largest run comes to on all of them.
long dealt(long tiles) { return (tiles + DIES - 1) / DIES * DIES; }
constexpr PartTime NARROW_PARTS = {64, 2, 5950, 256, 166, 95, 250, 1540}, WIDE_PARTS = {128, 1, 6630, 445, 200, 0, 251, 1720},
                   WIDE_PARTS_TWO = {128, 2, 7190, 592, 237, 0, 268, 1050};          // (two stages instead of three: two to a compute unit, beyond 256 rows)
long parts_time(const PartTime& shape, int M, long rows_w, int steps, int parts) {
    const long groups = dealt((long)((M + 127) / 128) * ((rows_w + shape.columns - 1) / shape.columns)) * parts, places = (long)shape.places * XRT_COMPUTE_UNITS;
    const long whole = groups / places, rest = groups % places;
    const long full = shape.step + shape.share * shape.places + shape.beside;
    const long last = rest == 0 ? 0 : shape.step + shape.share * rest / XRT_COMPUTE_UNITS + (rest > XRT_COMPUTE_UNITS ? shape.beside : 0);
    return shape.once + shape.part * parts + steps * (whole * full + last) + shape.sums * parts * ((long)M * rows_w / 1000) / 1000;
}
// The same of the tiles without a split (a fit to the same products: their own estimate counts a warm chip's rounds alone).
long unsplit_time(int M, long rows_w, int K, int mode) {
    const int kind = mode == MODE_GATED ? ENDS_GATED : mode == MODE_ACCUMULATE ? ENDS_ADDING : ENDS_BF16;
    auto tiles = [&](int bm, int bn) { return (long)((M + bm - 1) / bm) * ((rows_w + bn - 1) / bn); };
    if (mode == MODE_GATED && M <= 256) {                      // one round of tiles in several stages
        if (tiles(128, 64) <= XRT_COMPUTE_UNITS) return 5000 + (NARROW_PARTS.step + NARROW_PARTS.share * tiles(128, 64) / XRT_COMPUTE_UNITS) * (K / 64);
        if (tiles(128, 128) <= XRT_COMPUTE_UNITS) return 5000 + (WIDE_PARTS.step + WIDE_PARTS.share * tiles(128, 128) / XRT_COMPUTE_UNITS) * (K / 64);
    }
    auto cost = [&](const TileTime& tile) { return rounds_cost(tiles(tile.bm, tile.bn), tile, K, kind); };
    const long least = min(min(cost(LARGE_TILE), cost(MIDDLE_TILE)), min(cost(HALF_TILE), cost(SMALL_TILE)));
    return 1000 + (mode == MODE_GATED ? least : least * 127 / 100);
}
struct Cut { int splits, tile, columns; };
// Tiles of 128 x 64 or 128 x 128 and the number of parts by the estimates, against the product without a split, which saves a gated one the sums of both
// halves. (Narrow tiles read x twice as often, which does not stay in a die's L2 when k is long: 4096 rows of w, k = 14336, 100 rows of x 34.7 us in wide
// tiles, 40.3 in narrow ones.)
Cut cut_by_parts_time(int M, long rows_w, int K, int mode, bool whole_norm = false) {
    const int units = K / 64;
    auto per_part = [&](int parts) { return (units + parts - 1) / parts; };
    auto some = [&](int parts) { return parts <= units && (units + per_part(parts) - 1) / per_part(parts) == parts; };     // (otherwise: as many pieces a part with fewer parts)
    Cut cut{1, 128, 128};
    const long large_tiles = (long)((M + 255) / 256) * ((rows_w + 255) / 256);
    if (large_tiles <= 128 && M >= 512 && mode != MODE_GATED && units >= (whole_norm ? 64 : 128)) return Cut{max(1, min(min((int)(XRT_COMPUTE_UNITS / large_tiles), 8), units / 24)), 256, 256};
    if ((long)((M + 127) / 128) * ((rows_w + SPLIT_BN - 1) / SPLIT_BN) > (M <= 256 ? 2 * XRT_COMPUTE_UNITS : XRT_COMPUTE_UNITS)) return cut;      // (they fill the chip as they are)
    long best = unsplit_time(M, rows_w, K, mode);
    for (const PartTime& shape : {NARROW_PARTS, M <= 256 ? WIDE_PARTS : WIDE_PARTS_TWO}) {
        if (shape.columns == 64 && K >= 8192 && rows_w > 2048) continue;
        for (int parts = 2; parts <= 16; ++parts) {
            if (!some(parts)) continue;
            const long time = parts_time(shape, M, rows_w, per_part(parts), parts);
            if (time < best) { best = time; cut = Cut{parts, 128, shape.columns}; }
        }
    }
    // Large tiles of 192 rows, in parts that make one round in either order: fewer operands read a product, more at the ends (150 rows of x, 10240 rows of w, k = 5120
    // 43 -> 34 us beside the best of the others).
    const long large = dealt((long)((M + 191) / 192) * ((rows_w + 255) / 256));
    for (int parts = 2; M > 128 && parts <= 16 && parts * large <= XRT_COMPUTE_UNITS; ++parts) {
        if (!some(parts)) continue;
        const long time = 10000 + 1200L * per_part(parts) + 1400L * parts * (M * rows_w / 1000) / 1000;
        if (time < best) { best = time; cut = Cut{parts, 192, 256}; }
    }
    return cut;
}

// What every other product of more than 64 rows of x takes, in microseconds, cut or not. A step of 64 along k takes `step`, `share` more for each workgroup
// that a compute unit has on average (up to `places` of them side by side), and `beside` where some have two; reading w, and `again` of what is read of x on
// all dies (on one, where the parts are dealt so), takes `bytes` a megabyte; the larger of the two counts, smoothly. `part` and `sums` are what a part and a
// million partial sums cost the second kernel and the first; once and outs (a million results) go by what the product does: store, add with the norm behind
// it (cut: in the second kernel; not cut: a kernel of its own), add.
// Fitted to 8000 products (65 to 2100 rows of x, 256 to 16384 rows of w, k from 256 to 25600, half of them of widths that models have), every tile with
// every number of parts from 2 to 16 of each timed, 150000 times in all: of 2400 others what it chooses is 1.5 % off the best of all on average, where the
// estimates above, which know the tiles of 128 and, for k from 4096 on and 512 rows, of 256 rows, and of 192 as a rule of thumb, were 4.5 % off: 520 rows of
// x, 4096 rows of w, k = 14336 84 -> 67 us, 2048 rows, k = 8192 45 -> 34, 200 rows, 5120 rows, k = 25600 97 -> 72, 1100 rows, 4096 rows, k = 4096 63 -> 51.
// Two shapes are fitted anew to 2500 products where cut and uncut are near each other (k up to 5000), timed with w from memory, as a model's layers find it:
// uncut in tiles of 128 x 128 (the last of WHOLE; adding, it was taken for 25 % dearer than it is) and 128 x 64 of a short k, alone on its compute unit (14
// % dearer). By the figures before, adding products of a short k went in two parts where the workgroups then shared compute units (300 rows of x, 4096 rows
// of w, k = 256 13.2 us, uncut 9.4; 788 rows, 2048, k = 768 17.1, uncut 14.6). Of 700 products drawn whose cut is another than before the estimate none
// takes more than 1.01 of what it took then (by the figures before 20 took over 1.05), and all of them 0.75.
enum { KIND_STORE, KIND_NORMED, KIND_ADD };
struct TileCost { double step, share, beside, part, bytes, again, sums, once[3], outs[3]; };
struct CutShape { int rows, columns, places; TileCost cost; };
constexpr CutShape CUT_128_BY_64 = {128, 64, 2, {0.295, 0.101, 0.149, 0.174, 0.203, 0.075, 1.385, {6.003, 6.308, 6.525}, {0.075, 1.864, 0.000}}},
                   // (at most one to a compute unit: four stages; of a short k eight wavefronts)
                   CUT_128_BY_64_ALONE = {128, 64, 2, {0.329, 0.000, 0.000, 0.219, 0.198, 0.185, 1.762, {5.174, 5.018, 5.524}, {0.169, 3.266, 0.312}}},
                   CUT_128_BY_64_SHORT = {128, 64, 2, {0.276, 0.012, 0.000, 0.233, 0.165, 0.389, 1.754, {4.364, 5.403, 4.433}, {1.168, 2.526, 1.469}}},
                   CUT_128_BY_128 = {128, 128, 2, {0.706, 0.122, 0.003, 0.147, 0.314, 0.105, 1.035, {6.869, 7.672, 6.806}, {0.169, 1.672, 0.754}}},
                   CUT_128_BY_128_THREE_STAGES = {128, 128, 1, {0.543, 0.000, 0.000, 0.204, 0.162, 0.161, 1.942, {5.855, 6.164, 5.901}, {0.694, 0.947, 0.788}}},
                   CUT_192 = {192, 256, 1, {0.759, 0.209, 0.000, 0.093, 0.165, 0.646, 0.850, {12.673, 13.490, 12.186}, {0.052, 1.386, 0.922}}},
                   CUT_256 = {256, 256, 1, {0.778, 0.441, 0.000, 0.069, 0.181, 0.632, 0.698, {15.312, 16.178, 14.564}, {0.247, 1.626, 1.237}}},
                   WHOLE[] = {{256, 256, 1, {0.842, 0.410, 0.000, 0.000, 0.001, 0.196, 0.000, {7.279, 26.096, 21.168}, {0.429, 1.205, 0.632}}},
                              {192, 256, 1, {0.763, 0.224, 0.000, 0.000, 0.372, 0.000, 0.000, {5.708, 18.654, 14.700}, {0.527, 1.509, 0.977}}},
                              {128, 256, 1, {0.676, 0.106, 0.000, 0.000, 0.377, 0.000, 0.000, {4.336, 13.687, 9.568}, {0.572, 1.724, 1.275}}},
                              {128, 128, 2, {0.592, 0.272, 0.000, 0.000, 0.457, 0.163, 0.000, {7.491, 8.395, 6.122}, {0.020, 2.493, 0.649}}}};
// Whether the parts of tiles of 128 x 64 have a compute unit each, as they are dealt: four stages then (counted as dealt by columns, 39 tiles in six parts had
// none left: 150 x 2664, k = 5504 19.5 -> 16.9 us, 98 x 5320, k = 6464 23.7 -> 22.2; 150 such products drawn 0.93 of their time, the worst 1.01).
bool narrow_alone(int M, long rows_w, int K, int parts) {
    const long tiles_m = (M + 127) / 128, tiles_n = (rows_w + 63) / 64;
    return part_ids(tiles_m * tiles_n, parts, deals_by_parts(64, tiles_m, tiles_n, K, parts)) <= XRT_COMPUTE_UNITS;
}
double cut_time(const CutShape& shape, int M, int N, int K, int steps, int parts, int kind) {
    const TileCost& c = shape.cost;
    const long tiles_m = (M + shape.rows - 1) / shape.rows, tiles_n = (N + shape.columns - 1) / shape.columns;
    const bool by_parts = deals_by_parts(shape.columns, tiles_m, tiles_n, K, parts);
    const long groups = part_ids(tiles_m * tiles_n, parts, by_parts), places = (long)shape.places * XRT_COMPUTE_UNITS;
    const long whole = groups / places, rest = groups % places;
    const double full = c.step + c.share * shape.places + c.beside;
    const double last = rest == 0 ? 0. : c.step + c.share * rest / XRT_COMPUTE_UNITS + (rest > XRT_COMPUTE_UNITS ? c.beside : 0.);
    const double loop = steps * (whole * full + last), results = 1e-6 * M * N;
    const double memory = c.bytes * 2e-6 * K * (N + c.again * M * (by_parts ? 1 : DIES));
    const double loop2 = loop * loop, memory2 = memory * memory;
    return c.once[kind] + c.part * parts + sqrt(sqrt(loop2 * loop2 + memory2 * memory2)) + (parts > 1 ? c.sums * parts * results : 0.) + c.outs[kind] * results;
}

// Gated products of 17 to 64 rows of x (nanoseconds): unsplit in one round of tiles of 64 x 64, every workgroup all of k, or in parts of 64 x 128 as many as
// the compute units take, and a second kernel. A step of 64 along k takes its time however few the tiles, so a long k with few of them wants parts (64 rows of
// x, 1408 rows of w, k = 4096 20.4 us unsplit, 13.2 in parts; 512 rows, k = 8192 36.4, 12.4; 10240 rows, k = 3072 21.2, 20.1) and a short one none (6144 rows
// of w, k = 1024, 24 rows of x 8.4 us, 10.1 in parts; 16384 rows, k = 2048, 64 rows 17.7, 21.0). Fitted to 3841 products drawn at random (128 to 16384 rows of
// w, k of 128 to 16384, 17 to 64 rows of x, a third of them of widths that are multiples of 256): what the estimates choose is 0.1 % off the better of the two
// on average and takes 0.91 of what parts alone do, 34 above 1.03, up to 1.17.
long narrow_gated_time(int M, long rows_w, int units) {
    const long share = dealt((rows_w + 63) / 64);              // (of the compute units; at most all of them)
    return 3970 + units * (243 + (77 * 64 + 33 * M) * share / (64 * XRT_COMPUTE_UNITS)) + 2510 * (M * rows_w / 1000) / 1000;
}
long few_rows_parts_time(int M, long rows_w, int per, int parts) {
    const long groups = dealt((rows_w + SPLIT_BN - 1) / SPLIT_BN) * parts;
    return 5330 + 94 * parts + per * (328 + 318 * groups / XRT_COMPUTE_UNITS + (groups > XRT_COMPUTE_UNITS ? 250 : 0)) + 2490 * parts * (M * rows_w / 1000) / 1000;
}

// Products of 17 to 64 rows of x that are not gated, in tiles of 64 x 128 and `parts` parts: microseconds, as above. Fitted to 6500 products (256 to 16384 rows
// of w, k from 256 to 20000); of 2700 others the choice by it is 0.9 % off the best number of parts (61 rows, 4096 rows of w, k = 1024 12.2 -> 10.4 us, 3072
// rows, k = 2048 12.2 -> 11.9). 454 whose number of parts it changes take 0.87 of as many as leave every compute unit one workgroup, the worst 1.01.
double few_rows_cut_time(int M, int N, int K, int steps, int parts) {
    const long tiles = (N + SPLIT_BN - 1) / SPLIT_BN;
    const long groups = part_ids(tiles, parts, deals_by_parts(SPLIT_BN, 1, tiles, K, parts));
    constexpr double STEP = 0.367, SHARE = 0.292, BESIDE = 0.313;
    const long whole = groups / XRT_COMPUTE_UNITS, rest = groups % XRT_COMPUTE_UNITS;
    const double share = SHARE * rest / XRT_COMPUTE_UNITS;
    double step = whole * (STEP + SHARE) + (rest > 0 ? STEP + share : 0.);
    if (whole == 1 && rest > 0) step = STEP + SHARE + BESIDE + share;      // two side by side
    const double loop = steps * step, memory = 0.051 * 2e-6 * K * N, loop2 = loop * loop, memory2 = memory * memory;
    return 5.287 + 0.051 * parts + sqrt(sqrt(loop2 * loop2 + memory2 * memory2)) + 2.444e-6 * parts * M * N;
}

// fixed: the plan of few parts, which xrt_linear_static takes where the sums of the product's own do not fit its array.
SplitPlan plan_of(int M, int N, int K, int mode, bool whole_norm, bool fixed) {
    const long rows_w = mode == MODE_GATED ? 2L * N : N;
    const long tiles_n = (rows_w + SPLIT_BN - 1) / SPLIT_BN;
    const int units = K / 64;                                  // k is dealt out in pieces of 64
    int splits = 1, tile = SPLIT_BM, columns = SPLIT_BN;
    double best = 0;
    auto per_part = [&](int parts) { return (units + parts - 1) / parts; };
    auto some = [&](int parts) { return parts <= units && (units + per_part(parts) - 1) / per_part(parts) == parts; };     // (otherwise: as many pieces a part with fewer parts)
    if (M <= SPLIT_BM && mode == MODE_GATED) {
        splits = (int)(XRT_COMPUTE_UNITS / tiles_n);                         // one workgroup per compute unit, or fewer
        if ((rows_w + 63) / 64 <= XRT_COMPUTE_UNITS) {
            // one round of tiles of half the width is there for the taking, without a second kernel: by the estimates of both
            const int parts = max(1, min(min(splits, 16), units)), per = per_part(parts);
            if (parts == 1 || narrow_gated_time(M, rows_w, units) < few_rows_parts_time(M, rows_w, per, (units + per - 1) / per)) { splits = 1; columns = 64; }
        }
    } else if (M <= SPLIT_BM) {
        // As many parts as leave every compute unit one workgroup, or fewer that are a twentieth better by the estimate. (More, for a w so wide that they leave units idle: with w
        // from memory, which bounds such a product, 346 drawn took 1.01 of the time, 124 of them over 1.03 and up to 1.12: 20 rows, 12288 rows of w, k = 8192 39.0 us in two
        // parts, 42.0 in five.) A product whose tiles leave no room for two parts is not cut, and what the parts sum up fits the fixed array of xrt_linear_static.
        splits = min((int)(XRT_COMPUTE_UNITS / tiles_n), min(16, units));
        if (splits > 1) {
            splits = (units + per_part(splits) - 1) / per_part(splits);
            best = 0.95 * few_rows_cut_time(M, N, K, per_part(splits), splits);
        }
        for (int parts = 2; splits > 1 && parts <= 16; ++parts) {
            if (!some(parts) || parts * tiles_n > XRT_COMPUTE_UNITS || (long)parts * M * N > XRT_LINEAR_STATIC_FLOATS) continue;
            const double time = few_rows_cut_time(M, N, K, per_part(parts), parts);
            if (time < best) { best = time; splits = parts; }
        }
    } else if (mode == MODE_GATED || fixed || M > (N < 1024 ? 2100 : 4608) || N > 16384) {
        // Gated products, and others where the estimate below is not good for more rows or columns than it was fitted to. Drawn products whose cut it changes:
        // of 185 with more than 16384 rows of w 24 took over 1.05 of the time by it (74 rows of x, 25600, k = 1024 22.5 -> 26.0 us), of 103 with more than 4608
        // rows of x 12 (5500 rows, 1024, k = 3072 46 -> 50), of 230 with more than 2100 and fewer than 1024 of w 17 (3763 rows, 256, k = 7168 27.6 -> 36.9).
        // Within the line: 2100 to 4608 rows 3 of 359, and 0.91 on average (2600 rows, 2048, k = 8192 92 -> 84; 4300 rows, 1024, k = 3072 45 -> 43); k below
        // 256 or above 25600 none of 223, 0.71; fewer than 256 rows of w 1 of 240, 0.55.
        const Cut cut = cut_by_parts_time(M, rows_w, K, mode, whole_norm);
        splits = cut.splits;
        tile = cut.tile;
        columns = cut.columns;
    } else {
        // The best of all cuts by the estimate, where it is a twentieth less than what the two older estimates choose (what it finds below that is as often slower as
        // faster: of 2400 products 157 take more than 1.05 of their time without this, 20 with it, and all of them 0.97 either way).
        const int kind = mode == MODE_STORE ? KIND_STORE : whole_norm ? KIND_NORMED : KIND_ADD;
        auto time_of = [&](int rows, int wide, int parts) {
            const CutShape& shape = rows == 256 ? CUT_256 : rows == 192 ? CUT_192 : wide == 128 ? (M <= 256 ? CUT_128_BY_128_THREE_STAGES : CUT_128_BY_128)
                : !narrow_alone(M, N, K, parts) ? CUT_128_BY_64 : K < 4096 ? CUT_128_BY_64_SHORT : CUT_128_BY_64_ALONE;
            return cut_time(shape, M, N, K, per_part(parts), parts, kind);
        };
        double whole = 1e30;
        for (const CutShape& shape : WHOLE) whole = fmin(whole, cut_time(shape, M, N, K, units, 1, kind));
        const Cut cut = cut_by_parts_time(M, rows_w, K, mode, whole_norm);
        splits = cut.splits;
        tile = cut.tile;
        columns = cut.columns;
        best = 0.95 * (splits == 1 ? whole : time_of(tile, columns, splits));
        if (splits > 1 && whole < best) { best = whole; splits = 1; tile = columns = 128; }
        for (const Cut& shape : {Cut{0, 128, 64}, Cut{0, 128, 128}, Cut{0, 192, 256}, Cut{0, 256, 256}}) {
            // (tiles that are mostly empty, and more than a round of the large ones or about two of the others, were not timed)
            if ((shape.tile == 192 && M <= 96) || (shape.tile == 256 && M < 200)) continue;
            const long tiles = (long)((M + shape.tile - 1) / shape.tile) * ((N + shape.columns - 1) / shape.columns);
            for (int parts = 2; parts <= 16 && (shape.columns == 256 ? parts * dealt(tiles) <= XRT_COMPUTE_UNITS : parts * tiles <= 600); ++parts) {
                if (!some(parts)) continue;
                const double time = time_of(shape.tile, shape.columns, parts);
                if (time < best) { best = time; splits = parts; tile = shape.tile; columns = shape.columns; }
            }
        }
    }
    splits = max(1, min(min(splits, 16), units));
    const int per = per_part(splits);
    splits = (units + per - 1) / per;                          // no empty part
    return SplitPlan{splits, per * 64, rows_w, tile, columns};
}
// whole_norm: an RMSNorm follows that the second kernel can do outright.
// A step asks for the same plans again and again, several times a product (what it takes, its workspace, its launch): each thread keeps the last ones it has worked out.
SplitPlan split_plan(int M, int N, int K, int mode, bool whole_norm = false, bool fixed = false) {
    struct Kept { int M, N, K, kind; SplitPlan plan; };
    constexpr int PLANS = 64;
    static thread_local Kept kept[PLANS] = {};                 // (M = 0: none)
    const int kind = mode * 4 + whole_norm * 2 + fixed;
    Kept& k = kept[((unsigned)M * 2654435761u ^ (unsigned)N * 2246822519u ^ (unsigned)K * 3266489917u ^ (unsigned)kind * 668265263u) >> 26];
    if (k.M != M || k.N != N || k.K != K || k.kind != kind) k = Kept{M, N, K, kind, plan_of(M, N, K, mode, whole_norm, fixed)};
    return k.plan;
}

// The sums over the parts, in order, of one output, or (BOTH) of it and the one `apart` columns behind; part p lies p * stride floats
// behind `first`. Two, four or eight parts are asked for at once, then added (those beyond the last: that one again; with eight
// at a time whatever their number, two parts of 512 rows and 6144 columns took 1.0 us longer).
template <bool BOTH>
__device__ __forceinline__ float2 sum_of_parts(const float* __restrict__ first, long stride, int splits, long apart) {
    float2 sum = make_float2(0.f, 0.f);
    auto add = [&](auto at_once) {
        for (int p0 = 0; p0 < splits; p0 += at_once) {
            float of[at_once], behind[at_once];
#pragma unroll
            for (int u = 0; u < at_once; ++u) {
                const float* part = first + min(p0 + u, splits - 1) * stride;
                of[u] = part[0];
                if constexpr (BOTH) behind[u] = part[apart];
            }
#pragma unroll
            for (int u = 0; u < at_once; ++u) {
                sum.x = p0 + u < splits ? sum.x + of[u] : sum.x;
                if constexpr (BOTH) sum.y = p0 + u < splits ? sum.y + behind[u] : sum.y;
            }
        }
    };
    if (splits <= 2) add(std::integral_constant<int, 2>{});
    else if (splits <= 4) add(std::integral_constant<int, 4>{});
    else add(std::integral_constant<int, 8>{});
    return sum;
}

// NORM 1: the rows of a came without their RMSNorm's division (norm.squares_in): the sums are multiplied by
// 1 / rms of their row first. NORM 2 (accumulating): bfloat16(out * gain) and the sums of squares of out per
// tile of 16 columns are written as well (N a multiple of 16: the 16 lanes of a tile then share a row).
template <int MODE, typename TO, int NORM = 0>
__global__ void __launch_bounds__(256) split_reduce_kernel(const float* __restrict__ parts, int splits, int M, int N,
                                                            TO* __restrict__ out, const xrt_linear_norm norm, int activation) {
    __shared__ float wave_sums[256 / XRT_WAVE];
    const long rows_w = MODE == MODE_GATED ? 2L * N : N;
    const long index = (long)blockIdx.x * blockDim.x + threadIdx.x;
    const bool inside = index < (long)M * N;
    const long m = inside ? index / N : M - 1, n = inside ? index % N : 0;
    // the row's sums of squares are asked for before the partial sums and used after them. A block lies
    // within one row if N is a multiple of 256: then its threads share the work; else every thread adds
    // up its row's sums itself, in the order of the tiles.
    float mine = 0.f;
    if constexpr (NORM == 1) {
        if (N % 256 == 0)
            for (int t = threadIdx.x; t < norm.tiles_in; t += 256) mine += norm.squares_in[(long)t * XRT_SQUARES_STRIDE + m];
        else
            for (int t = 0; t < norm.tiles_in; ++t) mine += norm.squares_in[(long)t * XRT_SQUARES_STRIDE + m];
    }
    float sum = 0.f, up = 0.f;
    if (inside) {
        const float2 sums = sum_of_parts<MODE == MODE_GATED>(parts + m * rows_w + n, M * rows_w, splits, N);
        sum = sums.x;
        up = sums.y;
    }
    float by = 1.0f;
    if constexpr (NORM == 1) {
        float total = mine;
        if (N % 256 == 0) {
            mine = whole_wave_sum(mine);
            if (threadIdx.x % XRT_WAVE == 0) wave_sums[threadIdx.x / XRT_WAVE] = mine;
            __syncthreads();
            total = 0.f;
            for (int w = 0; w < 256 / XRT_WAVE; ++w) total += wave_sums[w];
        }
        by = 1.0f / sqrtf(total / (float)norm.width_in + norm.eps);
    }
    sum *= by;
    up *= by;
    float fresh = 0.f;
    if (inside) {
        if constexpr (MODE == MODE_STORE) out[index] = from_float<TO>(sum);
        else if constexpr (MODE == MODE_ACCUMULATE) { fresh = to_float(out[index]) + sum; out[index] = from_float<TO>(fresh); }
        else out[index] = from_float<TO>(gate_activation<sizeof(TO) == 2>(sum, activation) * up);
    }
    if constexpr (NORM == 2) {
        float squares = fresh * fresh;
        squares += __shfl_xor(squares, 1, XRT_WAVE);
        squares += __shfl_xor(squares, 2, XRT_WAVE);
        squares += __shfl_xor(squares, 4, XRT_WAVE);
        squares += __shfl_xor(squares, 8, XRT_WAVE);
        if (inside) {
            if (n % 16 == 0) norm.squares_out[(n / 16) * XRT_SQUARES_STRIDE + m] = squares;
            const float gain = norm.gain_dtype == XRT_F32 ? ((const float*)norm.gain)[n] : to_float(((const bf16*)norm.gain)[n]);
            ((bf16*)norm.scaled_out)[index] = from_float<bf16>(fresh * gain);
        }
    }
}

// The same for store and accumulate without a norm, four neighbouring columns a thread (N a multiple of 4):
// what products of many rows use, whose partial sums are tens of megabytes.
template <int MODE, typename TO>
__global__ void __launch_bounds__(256) split_reduce_wide_kernel(const float* __restrict__ parts, int splits, long count, TO* __restrict__ out) {
    const long index = ((long)blockIdx.x * blockDim.x + threadIdx.x) * 4;
    if (index >= count) return;
    float4 sum = *reinterpret_cast<const float4*>(parts + index);
    for (int p = 1; p < splits; ++p) {
        const float4 part = *reinterpret_cast<const float4*>(parts + p * count + index);
        sum.x += part.x; sum.y += part.y; sum.z += part.z; sum.w += part.w;
    }
    if constexpr (MODE == MODE_ACCUMULATE) {
        static_assert(sizeof(TO) == 4, "accumulation needs a float32 output");
        const float4 before = *reinterpret_cast<const float4*>(out + index);
        // the order of the one-column kernel: the parts first, in order, then onto what was there
        sum.x = before.x + sum.x; sum.y = before.y + sum.y; sum.z = before.z + sum.z; sum.w = before.w + sum.w;
    }
    if constexpr (sizeof(TO) == 4) {
        *reinterpret_cast<float4*>(out + index) = sum;
    } else {
        Four<TO> four;
        four.e[0] = from_float<TO>(sum.x); four.e[1] = from_float<TO>(sum.y); four.e[2] = from_float<TO>(sum.z); four.e[3] = from_float<TO>(sum.w);
        *reinterpret_cast<Four<TO>*>(out + index) = four;
    }
}

// The second kernel of an accumulating product of many rows that an RMSNorm follows: a workgroup takes a whole row, adds the
// parts onto the residual and writes the row's norm as well. The norm is the norm kernel's (elementwise.hip) to the bit: the same
// four columns a thread, the same order of the sum of squares, (x * 1/rms) * gain.
constexpr int NORM_THREADS = 256, NORM_QUADS = 8;       // of the norm kernel, and the four-column pieces a thread of it holds: rows of up to 8 * 256 * 4 columns
// THREADS: 256, or 1024 where the rows are too few to fill the chip with workgroups of 256 (a thread then holds a quarter of the
// pieces, and 256 threads add up the squares from LDS, in the norm kernel's order).
// Instead of a kernel that adds the parts and one that norms the rows (3.5 + 3.3 us for 100 rows of 2048, 6.3 + 4.9 for 333 of 4096). With the same for
// q, k and v (qkv_prepare.hip): logits of 100 tokens at the Llama-3.2-1B sizes 1549 -> 1366 us, 333 tokens on 3001 at the 8B sizes (6 layers) 1706 -> 1623.
template <typename TW, int THREADS>
__global__ void __launch_bounds__(THREADS) split_reduce_rmsnorm_kernel(const float* __restrict__ parts, int splits, long count, int N,
                                                                    float* __restrict__ out, const TW* __restrict__ gain, float eps,
                                                                    bf16* __restrict__ normed) {
    typedef float floatx4 __attribute__((ext_vector_type(4)));
    constexpr int QUADS = NORM_QUADS * NORM_THREADS / THREADS, AT_ONCE = THREADS == NORM_THREADS ? 1 : 4;     // parts asked for at once
    __shared__ float scratch[32];
    __shared__ floatx4 row_quads[THREADS == NORM_THREADS ? 1 : NORM_QUADS * NORM_THREADS];
    const long row = (long)blockIdx.x * N;
    const int quads = N / 4;
    floatx4 kept[QUADS];
    Four<TW> weight[QUADS];
#pragma unroll
    for (int i = 0; i < QUADS; ++i) {
        const int q = threadIdx.x + i * THREADS;
        kept[i] = floatx4{0.f, 0.f, 0.f, 0.f};
        weight[i] = Four<TW>{};
        if (q < quads) {
            const long index = row + 4L * q;
            const floatx4 before = *reinterpret_cast<const floatx4*>(out + index);
            weight[i] = *reinterpret_cast<const Four<TW>*>(gain + 4 * q);
            auto part_of = [&](int p) {                        // read once, by nobody else; few rows' parts still lie in the last cache
                const floatx4* from = reinterpret_cast<const floatx4*>(parts + p * count + index);
                return THREADS == NORM_THREADS ? __builtin_nontemporal_load(from) : *from;
            };
            floatx4 sum = part_of(0);
            for (int p0 = 1; p0 < splits; p0 += AT_ONCE) {
                floatx4 part[AT_ONCE];
#pragma unroll
                for (int u = 0; u < AT_ONCE; ++u)
                    part[u] = part_of(min(p0 + u, splits - 1));
#pragma unroll
                for (int u = 0; u < AT_ONCE; ++u)
                    if (p0 + u < splits) sum += part[u];
            }
            kept[i] = before + sum;
            *reinterpret_cast<floatx4*>(out + index) = kept[i];
        }
    }
    float squares = 0.f;
    auto add_squares = [&](const floatx4& v) { squares = fmaf(v[0], v[0], fmaf(v[1], v[1], fmaf(v[2], v[2], fmaf(v[3], v[3], squares)))); };
    if constexpr (THREADS == NORM_THREADS) {
#pragma unroll
        for (int i = 0; i < QUADS; ++i) add_squares(kept[i]);
    } else {
#pragma unroll
        for (int i = 0; i < QUADS; ++i) row_quads[threadIdx.x + i * THREADS] = kept[i];
        __syncthreads();
        if (threadIdx.x < NORM_THREADS) {
#pragma unroll
            for (int i = 0; i < NORM_QUADS; ++i) add_squares(row_quads[threadIdx.x + i * NORM_THREADS]);
        }
    }
    squares = block_sum(squares, scratch);                     // (wavefronts beyond the norm kernel's four add zeros behind theirs)
    const float inv_rms = 1.0f / sqrtf(squares / (float)N + eps);
#pragma unroll
    for (int i = 0; i < QUADS; ++i) {
        const int q = threadIdx.x + i * THREADS;
        if (q < quads) {
            Four<bf16> r;
#pragma unroll
            for (int e = 0; e < 4; ++e) r.e[e] = from_float<bf16>((kept[i][e] * inv_rms) * to_float(weight[i].e[e]));
            *reinterpret_cast<Four<bf16>*>(normed + row + 4L * q) = r;
        }
    }
}
template <typename TW>
void launch_reduce_rmsnorm(const float* parts, int splits, int M, int N, float* out, const void* gain, float eps, void* normed, hipStream_t s) {
    if (M < 2 * XRT_COMPUTE_UNITS)
        split_reduce_rmsnorm_kernel<TW, 1024><<<M, 1024, 0, s>>>(parts, splits, (long)M * N, N, out, (const TW*)gain, eps, (bf16*)normed);
    else
        split_reduce_rmsnorm_kernel<TW, NORM_THREADS><<<M, NORM_THREADS, 0, s>>>(parts, splits, (long)M * N, N, out, (const TW*)gain, eps, (bf16*)normed);
}

// The second kernel of a q/k/v projection split along k (no head norms, the rotation over the whole head):
// a thread adds up the two outputs that the rotation pairs (dims d and d + head_dim / 2 of one head), for
// NORM 1 scales them by the row's 1 / rms, rotates q and k by the token's position, writes bfloat16 q/k/v and
// puts k and v into the cache. One thread per (token, head, d).
template <int NORM>
__global__ void __launch_bounds__(256) split_reduce_qkv_kernel(const float* __restrict__ parts, int splits, int M, int N,
                                                                bf16* __restrict__ qkv, const xrt_linear_norm norm,
                                                                const QkvAfter after) {
    __shared__ float wave_sums[256 / XRT_WAVE];
    const int half = after.head_dim / 2;
    const long per_token = (long)(N / 2);
    const long index = (long)blockIdx.x * blockDim.x + threadIdx.x;
    const bool inside = index < (long)M * per_token;
    const long m = inside ? index / per_token : M - 1;
    const int pair = inside ? (int)(index % per_token) : 0;
    const int head = pair / half, d = pair % half;
    const long n = (long)head * after.head_dim + d;
    float mine = 0.f;
    if constexpr (NORM == 1) {
        // a block lies within one token if a token's pairs are a multiple of 256: then its threads share the work
        if (per_token % 256 == 0)
            for (int t = threadIdx.x; t < norm.tiles_in; t += 256) mine += norm.squares_in[(long)t * XRT_SQUARES_STRIDE + m];
        else
            for (int t = 0; t < norm.tiles_in; ++t) mine += norm.squares_in[(long)t * XRT_SQUARES_STRIDE + m];
    }
    const float2 sums = sum_of_parts<true>(parts + m * N + n, (long)M * N, splits, half);
    float lower = sums.x, upper = sums.y;
    const int pos = after.positions[m];
    const bool is_q = head < after.n_heads, is_v = head >= after.n_heads + after.n_kv_heads;
    float sine = 0.f, cosine = 1.f;
    if (after.rope_theta != nullptr && !is_v) sincosf((float)pos * after.rope_scale / after.rope_theta[d], &sine, &cosine);
    if constexpr (NORM == 1) {
        float total = mine;
        if (per_token % 256 == 0) {
            mine = whole_wave_sum(mine);
            if (threadIdx.x % XRT_WAVE == 0) wave_sums[threadIdx.x / XRT_WAVE] = mine;
            __syncthreads();
            total = 0.f;
            for (int w = 0; w < 256 / XRT_WAVE; ++w) total += wave_sums[w];
        }
        const float by = 1.0f / sqrtf(total / (float)norm.width_in + norm.eps);
        lower *= by;
        upper *= by;
    }
    if (!inside) return;
    // rounded as the product alone would have stored them, then rotated: the same values as from two kernels
    lower = to_float(from_float<bf16>(lower));
    upper = to_float(from_float<bf16>(upper));
    const bf16 out_lower = from_float<bf16>(lower * cosine - upper * sine);
    const bf16 out_upper = from_float<bf16>(lower * sine + upper * cosine);
    qkv[m * N + n] = out_lower;
    qkv[m * N + n + half] = out_upper;
    if (is_q || after.k_cache == nullptr) return;
    const int kv_head = head - after.n_heads - (is_v ? after.n_kv_heads : 0);
    const long base = cache_block_base(after.block_table, after.table_stride, after.n_blocks, after.slots[m], pos,
                                       after.n_kv_heads, kv_head, after.head_dim);
    if (base < 0) return;
    const int within = pos % XRT_BLOCK_TOKENS;
    if (is_v) {
        after.v_cache[base + cache_value_offset(d, within, after.head_dim)] = out_lower;
        after.v_cache[base + cache_value_offset(d + half, within, after.head_dim)] = out_upper;
    } else {
        after.k_cache[base + cache_key_offset(within, d, after.head_dim)] = out_lower;
        after.k_cache[base + cache_key_offset(within, d + half, after.head_dim)] = out_upper;
    }
}

// Parts of up to 64 rows of x: w past the caches where it cannot stay in them and k is long, which makes the runs of the parts long again. Ungated, so long a k
// is a feed-forward's width, and the matrix back from it counts three times: the gated one of twice its size stands beside it. (700 products drawn at random,
// past the caches against through them: such a w 0.97, 5120 rows, k = 25600, 32 rows of x 48.6 against 52.9 us; as large and k of 4096 to 16384 0.99, up to
// 1.08 with more than 48 rows of x; smaller and among more than the caches hold 0.97 to 1.04, 60 MB of them in turn 1.03 to 1.25.)
bool parts_read_past_caches(long rows_w, int K, bool gated) { return K >= 16384 && cannot_stay(rows_w, K, gated ? 3 : 6); }

// The product of all rows of w, ungated, into the workspace: [splits][M][rows_w]
int launch_parts(const bf16* a, const bf16* w, float* workspace, int M, int K, bool gated, const Packing& packing, const SplitPlan& plan, hipStream_t s) {
    const int rows_w = (int)plan.rows_w;
    if (M <= SPLIT_BM) {
        // Eight wavefronts, two to a SIMD: one reads its operands while the other multiplies (with four: 3 to 6 % longer, the second kernel included; 1024 rows of w,
        // k = 2048, 24 rows of x 8.8 -> 8.2 us, 10240 rows, k = 5120 26.7 -> 26.3).
        const bool past = parts_read_past_caches(plan.rows_w, K, gated);
        if (past) return launch_kernel<SPLIT_BM, SPLIT_BN, 2, 4, MODE_STORE, 64, 3, float, true>(a, w, workspace, M, rows_w, K, packing, s, plan.splits, plan.k_per_split);
        return launch_kernel<SPLIT_BM, SPLIT_BN, 2, 4, MODE_STORE, 64, 3, float>(a, w, workspace, M, rows_w, K, packing, s, plan.splits, plan.k_per_split);
    }
    if (plan.tile == 192)
        return launch_large<192, MODE_STORE, float, true>(a, w, workspace, M, rows_w, K, packing, XRT_ACT_SILU, s, plan.splits, plan.k_per_split);
    if (plan.tile == 256)
        return launch_large<256, MODE_STORE, float, true>(a, w, workspace, M, rows_w, K, packing, XRT_ACT_SILU, s, plan.splits, plan.k_per_split);
    if (plan.columns == 64) {
        // a fourth stage where a compute unit has one workgroup anyway (2048 rows of w, k = 8192, 65 / 200 rows of x 16.0 / 22.5 -> 14.7 / 20.5 us with its
        // second kernel; k = 2048, 3072 rows, 100 rows of x 12.0 -> 11.5)
        if (narrow_alone(M, rows_w, K, plan.splits)) {
            // eight wavefronts where k is short (2048 rows of w, k = 2048, 72 / 160 rows of x 11.1 / 13.0 -> 10.6 / 12.7 us with its second kernel, 3072 rows
            // 12.9 / 14.9 -> 12.4 / 14.4; 4096 rows, k = 4096, 72 / 100 rows 16.6 / 17.6 in four, 17.3 / 18.6 in eight)
            if (K < 4096) return launch_kernel<128, 64, 4, 2, MODE_STORE, 64, 4, float>(a, w, workspace, M, rows_w, K, packing, s, plan.splits, plan.k_per_split);
            return launch_kernel<128, 64, 4, 1, MODE_STORE, 64, 4, float>(a, w, workspace, M, rows_w, K, packing, s, plan.splits, plan.k_per_split);
        }
        return launch_kernel<128, 64, 2, 2, MODE_STORE, 64, 3, float>(a, w, workspace, M, rows_w, K, packing, s, plan.splits, plan.k_per_split);
    }
    if (M <= 256)           // (one workgroup to a compute unit anyway: a third stage keeps more of w on its way; with more, two share a unit)
        return launch_kernel<128, 128, 2, 2, MODE_STORE, 64, 3, float>(a, w, workspace, M, rows_w, K, packing, s, plan.splits, plan.k_per_split);
    return launch_kernel<128, 128, 2, 2, MODE_STORE, 64, 2, float>(a, w, workspace, M, rows_w, K, packing, s, plan.splits, plan.k_per_split);
}

template <typename TO>
int launch_split(const bf16* a, const bf16* w, TO* out, int M, int N, int K, int mode, int activation, const Packing& packing,
                 float* workspace, const xrt_linear_norm* norm, const QkvAfter* after, hipStream_t s, bool fixed = false) {
    // the whole norm after an accumulating product of many rows: normed rows asked for, and no sums of squares
    const bool whole_norm = norm && norm->scaled_out && !norm->squares_out && !norm->squares_in;
    const SplitPlan plan = split_plan(M, N, K, mode, whole_norm, fixed);
    const bool scaled = norm && norm->squares_in, emits = norm && norm->squares_out;
    XRT_REQUIRE(!norm || M <= SPLIT_BM || whole_norm, "linear (mfma): the halves of a norm around a product take at most %d rows here", SPLIT_BM);
    if (whole_norm)
        XRT_REQUIRE(M > SPLIT_BM && mode == MODE_ACCUMULATE && sizeof(TO) == 4 && plan.splits > 1 && N % 4 == 0 &&
                    N <= NORM_QUADS * 256 * 4 && norm->gain && (uintptr_t)out % 16 == 0 && (uintptr_t)norm->scaled_out % 8 == 0,
                    "linear (mfma): M=%d N=%d K=%d is not a product whose second kernel does the norm after it", M, N, K);
    const RowScale scale = scaled ? RowScale{norm->squares_in, norm->tiles_in, norm->width_in, norm->eps, activation}
                                  : RowScale{nullptr, 0, 0, 0.f, activation};
    XRT_REQUIRE(!after || (plan.splits > 1 && mode == MODE_STORE && sizeof(TO) == 2),
                "linear (mfma): only a bfloat16 product split along k does what follows a q/k/v projection");
    if (M <= SPLIT_BM && plan.splits == 1) {                   // tiles enough: each applies the epilogue itself
        XRT_REQUIRE(!emits, "linear (mfma): only a product split along k writes what the norm after it needs");
        if (mode == MODE_STORE) return launch_kernel<SPLIT_BM, SPLIT_BN, 1, 4, MODE_STORE, 64, 3, TO>(a, w, out, M, N, K, packing, s, 1, 0, scale);
        if (mode == MODE_GATED && plan.columns == 64) return launch_kernel<SPLIT_BM, 64, 2, 1, MODE_GATED, 64, 4, TO>(a, w, out, M, N, K, packing, s, 1, 0, scale);
        if (mode == MODE_GATED) return launch_kernel<SPLIT_BM, SPLIT_BN, 2, 2, MODE_GATED, 64, 3, TO>(a, w, out, M, N, K, packing, s, 1, 0, scale);
        if constexpr (sizeof(TO) == 4)
            return launch_kernel<SPLIT_BM, SPLIT_BN, 1, 4, MODE_ACCUMULATE, 64, 3, TO>(a, w, out, M, N, K, packing, s, 1, 0, scale);
        XRT_REQUIRE(false, "linear (mfma): accumulation needs a float32 output");
    }
    XRT_REQUIRE(workspace != nullptr, "linear (mfma): a product split along k needs its workspace");
    if (launch_parts(a, w, workspace, M, K, mode == MODE_GATED, packing, plan, s) != 0) return 1;
    const unsigned blocks = (unsigned)(((long)M * N + 255) / 256);
    const xrt_linear_norm none = {};
    const xrt_linear_norm& around = norm ? *norm : none;
    XRT_REQUIRE(!(scaled && emits), "linear (mfma): one product does one half of a norm");
    if (after != nullptr) {
        if constexpr (sizeof(TO) == 2) {
            const unsigned pair_blocks = (unsigned)(((long)M * (N / 2) + 255) / 256);
            if (scaled) split_reduce_qkv_kernel<1><<<pair_blocks, 256, 0, s>>>(workspace, plan.splits, M, N, out, around, *after);
            else split_reduce_qkv_kernel<0><<<pair_blocks, 256, 0, s>>>(workspace, plan.splits, M, N, out, around, *after);
            XRT_LAUNCH_CHECK("linear (split reduce, q/k/v)");
        }
        return 0;
    }
    if (whole_norm) {
        if constexpr (sizeof(TO) == 4) {
            if (norm->gain_dtype == XRT_F32) launch_reduce_rmsnorm<float>(workspace, plan.splits, M, N, out, norm->gain, norm->eps, norm->scaled_out, s);
            else launch_reduce_rmsnorm<bf16>(workspace, plan.splits, M, N, out, norm->gain, norm->eps, norm->scaled_out, s);
            XRT_LAUNCH_CHECK("linear (split reduce with the norm after it)");
        }
        return 0;
    }
    if (!scaled && !emits && mode != MODE_GATED && N % 4 == 0 && M > SPLIT_BM && (uintptr_t)out % 16 == 0) {
        const long count = (long)M * N;
        const unsigned wide_blocks = (unsigned)((count / 4 + 255) / 256);
        if (mode == MODE_STORE) split_reduce_wide_kernel<MODE_STORE, TO><<<wide_blocks, 256, 0, s>>>(workspace, plan.splits, count, out);
        else if constexpr (sizeof(TO) == 4) split_reduce_wide_kernel<MODE_ACCUMULATE, TO><<<wide_blocks, 256, 0, s>>>(workspace, plan.splits, count, out);
        else XRT_REQUIRE(false, "linear (mfma): accumulation needs a float32 output");
        XRT_LAUNCH_CHECK("linear (split reduce, four columns a thread)");
        return 0;
    }
#define XRT_REDUCE(MODE_, NORM_) split_reduce_kernel<MODE_, TO, NORM_><<<blocks, 256, 0, s>>>(workspace, plan.splits, M, N, out, around, activation)
    if (mode == MODE_STORE) { if (scaled) XRT_REDUCE(MODE_STORE, 1); else XRT_REDUCE(MODE_STORE, 0); }
    else if (mode == MODE_GATED) { if (scaled) XRT_REDUCE(MODE_GATED, 1); else XRT_REDUCE(MODE_GATED, 0); }
    else if (scaled) XRT_REDUCE(MODE_ACCUMULATE, 1);
    else if (emits) {
        XRT_REQUIRE(N % 16 == 0, "linear (mfma): sums of squares per 16 columns need N = %d to be a multiple of 16", N);
        XRT_REDUCE(MODE_ACCUMULATE, 2);
    } else XRT_REDUCE(MODE_ACCUMULATE, 0);
#undef XRT_REDUCE
    XRT_LAUNCH_CHECK("linear (split reduce)");
    return 0;
}

}  // namespace

bool xrt_linear_mfma_accepts(const void* a, const void* w, int M, int N, int K, int mode) {
    const long rows_w = mode == MODE_GATED ? 2L * N : N;     // operands are addressed with 32-bit element offsets
    return K % 8 == 0 && (uintptr_t)a % 16 == 0 && (uintptr_t)w % 16 == 0 && (long)M * K < (1L << 31) && (rows_w + 15) * K < (1L << 31);
}

int xrt_linear_mfma(const void* a, const void* w, void* out, int out_dtype, int M, int N, int K, int mode, int activation,
                    const Packing& packing, hipStream_t s) {
    if (out_dtype == XRT_F32) return launch_shape<float>((const bf16*)a, (const bf16*)w, (float*)out, M, N, K, mode, activation, packing, s);
    return launch_shape<bf16>((const bf16*)a, (const bf16*)w, (bf16*)out, M, N, K, mode, activation, packing, s);
}

// Groups of rows of a, each with a matrix of its own (gemm_grouped_kernel). The rows of a tile: 256 where a group has some
// hundred rows on average (the filling of its last tile is then a small part), 128 otherwise.
int xrt_linear_groups_tile(long rows, int groups) { return groups > 0 && rows / groups >= 384 ? 256 : 128; }

bool xrt_linear_groups_mfma_accepts(const void* a, int lda, const void* w, int ldw, int N, int K, int mode, const Packing& packing) {
    const long rows_w = mode == MODE_GATED ? 2L * N : N;
    if (mode != MODE_STORE && mode != MODE_GATED) return false;
    if (mode == MODE_GATED && (!is_packed(packing) ? true : packing.kind != XRT_PACK_GATED || packing.gated_n != N || N % 8 != 0)) return false;
    if (mode == MODE_STORE && is_packed(packing) && packing.kind != XRT_PACK_TILES) return false;
    return K > 0 && K % 64 == 0 && lda >= K && lda % 8 == 0 && ldw >= K && ldw % (is_packed(packing) ? 32 : 8) == 0 && (uintptr_t)a % 16 == 0 &&
           (uintptr_t)w % 16 == 0 && 256L * lda < (1L << 31) && (rows_w + 15) * ldw < (1L << 31);
}

// How many parts k is best split into: two where the tiles are too few to fill the chip twice over (a last round that is mostly
// empty costs a whole one), one otherwise. Only plain sums can be split (their parts are added by whoever reads them).
int xrt_linear_groups_splits(int tiles_m, int N, int K, int mode) {
    const int tiles_n = (N + LARGE_BN - 1) / LARGE_BN;
    return mode == MODE_STORE && K % 128 == 0 && (long)tiles_m * tiles_n < 2L * XRT_COMPUTE_UNITS ? 2 : 1;
}

int xrt_linear_groups_mfma(const void* a, int lda, const void* w, long w_stride, int ldw, void* out, int out_dtype, int tile, int tiles_m, int N,
                           int K, int mode, int activation, const int* tile_group, const Packing& packing, int splits, hipStream_t s) {
    XRT_REQUIRE(tile == 128 || tile == 256, "linear (groups): tiles of %d rows", tile);
    if (tile == 256)
        return launch_grouped_of<256>((const bf16*)a, (const bf16*)w, w_stride, out, out_dtype, tiles_m, N, K, lda, ldw, tile_group, packing, mode,
                                      activation, splits, s);
    return launch_grouped_of<128>((const bf16*)a, (const bf16*)w, w_stride, out, out_dtype, tiles_m, N, K, lda, ldw, tile_group, packing, mode,
                                  activation, splits, s);
}

// The same by the plan of few parts (xrt_linear_static): how many floats its partial sums are (0: not cut along k), and the product.
long xrt_linear_split_fixed_floats(const void* a, const void* w, int M, int N, int K, int mode) {
    if (M <= 16 || K % 64 != 0 || K < 128 || !xrt_linear_mfma_accepts(a, w, M, N, K, mode)) return 0;
    const SplitPlan plan = split_plan(M, N, K, mode, false, true);
    return plan.splits == 1 || plan.rows_w * (long)M >= (1L << 31) ? 0 : (long)plan.splits * M * plan.rows_w;
}
int xrt_linear_split_fixed(const void* a, const void* w, void* out, int out_dtype, int M, int N, int K, int mode, int activation, float* workspace, hipStream_t s) {
    const Packing plain = {XRT_PACK_NONE, 0, 0, 0};
    if (out_dtype == XRT_F32) return launch_split<float>((const bf16*)a, (const bf16*)w, (float*)out, M, N, K, mode, activation, plain, workspace, nullptr, nullptr, s, true);
    return launch_split<bf16>((const bf16*)a, (const bf16*)w, (bf16*)out, M, N, K, mode, activation, plain, workspace, nullptr, nullptr, s, true);
}

// Whether a product runs through the tiles of this section (17 to 64 rows of x, or more rows and few
// tiles), and the floats of workspace it then needs (0 where k is not split).
bool xrt_linear_split_takes(const void* a, const void* w, int M, int N, int K, int mode, long* workspace_floats) {
    *workspace_floats = 0;
    if (M <= 16 || K % 64 != 0 || K < 128 || !xrt_linear_mfma_accepts(a, w, M, N, K, mode)) return false;
    const SplitPlan plan = split_plan(M, N, K, mode);
    if (plan.splits == 1) return M <= SPLIT_BM;               // more rows and enough tiles without a split: the kernels above
    if (plan.rows_w * (long)M >= (1L << 31)) return false;
    *workspace_floats = (long)plan.splits * M * plan.rows_w;
    return true;
}

// Whether an accumulating product of more than 64 rows runs as tiles that split k, so that its second kernel can do the
// RMSNorm that follows it outright; and the floats of workspace it then needs.
bool xrt_linear_split_takes_whole_norm(const void* a, const void* w, int M, int N, int K, int mode, long* workspace_floats) {
    *workspace_floats = 0;
    if (mode != MODE_ACCUMULATE || M <= SPLIT_BM || K % 64 != 0 || N % 4 != 0 || N > NORM_QUADS * 256 * 4 ||
        !xrt_linear_mfma_accepts(a, w, M, N, K, mode))
        return false;
    const SplitPlan plan = split_plan(M, N, K, mode, true);
    if (plan.splits < 2 || (long)M * N >= (1L << 31)) return false;
    *workspace_floats = (long)plan.splits * M * N;
    return true;
}

// Whether a product of 17 to 64 rows can do its half of an RMSNorm: take rows that come without the
// division (any mode), or, accumulating and split along k, write what the norm after it needs, provided
// the product after the norm (same rows, N columns of a) will run through these tiles too.
bool xrt_linear_split_takes_norm(const void* a, const void* w, int M, int N, int K, int mode) {
    long unused = 0;
    if (M <= 16 || M > SPLIT_BM || !xrt_linear_split_takes(a, w, M, N, K, mode, &unused)) return false;
    if (mode != MODE_ACCUMULATE) return true;
    return split_plan(M, N, K, mode).splits > 1 && N % 64 == 0 && N >= 128;
}

int xrt_linear_split(const void* a, const void* w, void* out, int out_dtype, int M, int N, int K, int mode, int activation,
                     const Packing& packing, float* workspace, const xrt_linear_norm* norm, hipStream_t s) {
    if (out_dtype == XRT_F32) return launch_split<float>((const bf16*)a, (const bf16*)w, (float*)out, M, N, K, mode, activation, packing, workspace, norm, nullptr, s);
    return launch_split<bf16>((const bf16*)a, (const bf16*)w, (bf16*)out, M, N, K, mode, activation, packing, workspace, norm, nullptr, s);
}

// Whether the q/k/v projection of a step of 17 to 64 tokens can also do what follows it (rotation over the
// whole head or none, no head norms, cache write) in the kernel that adds up its partial sums.
bool xrt_linear_split_takes_qkv(const void* a, const void* w, int M, int N, int K, const QkvAfter& after, long* workspace_floats) {
    *workspace_floats = 0;
    if (M > SPLIT_BM || after.head_dim % 2 != 0 || N != (after.n_heads + 2 * after.n_kv_heads) * after.head_dim) return false;
    if (after.rope_theta != nullptr && after.rope_dim != after.head_dim) return false;
    return xrt_linear_split_takes(a, w, M, N, K, MODE_STORE, workspace_floats) && *workspace_floats > 0;
}

int xrt_linear_split_qkv(const void* a, const void* w, void* qkv, int M, int N, int K, const Packing& packing, float* workspace,
                         const xrt_linear_norm* norm, const QkvAfter& after, hipStream_t s) {
    return launch_split<bf16>((const bf16*)a, (const bf16*)w, (bf16*)qkv, M, N, K, MODE_STORE, XRT_ACT_SILU, packing, workspace, norm, &after, s);
}

// The tiles of a product that is not cut along k, more than 64 rows of x.
extern "C" int xrt_linear_tiles(int out_dtype, int M, int N, int K, int mode) {
    int unused = 0;
    if (M <= 0 || N <= 0 || K <= 0 || mode < MODE_STORE || mode > MODE_GATED) return -1;
    if (mode == MODE_GATED) return out_dtype == XRT_F32 ? tile_shape<MODE_GATED, float>(M, N, K, &unused) : tile_shape<MODE_GATED, bf16>(M, N, K, &unused);
    if (mode == MODE_ACCUMULATE) return tile_shape<MODE_ACCUMULATE, float>(M, N, K, &unused);
    return out_dtype == XRT_F32 ? tile_shape<MODE_STORE, float>(M, N, K, &unused) : tile_shape<MODE_STORE, bf16>(M, N, K, &unused);
}

// How a product is cut that runs through the tiles of this section: the number of parts along k (1: not cut, another kernel's if M > 64), a tile's rows of x and of w.
extern "C" int xrt_linear_parts(int M, int N, int K, int mode, int whole_norm, int* rows, int* columns) {
    if (M <= 16 || N <= 0 || K < 64 || K % 64 != 0 || mode < MODE_STORE || mode > MODE_GATED || !rows || !columns) return -1;
    const SplitPlan plan = split_plan(M, N, K, mode, whole_norm != 0);
    *rows = plan.tile;
    *columns = plan.columns;
    return plan.splits;
}

// The order in which the workgroups of one that is not cut take its tiles.
extern "C" int xrt_linear_tile_order(int tiles_m, int tiles_n, int K, int* places, int room) {
    if (tiles_m <= 0 || tiles_n <= 0 || (long)tiles_m * tiles_n >= (1L << 30) || K <= 0 || (room > 0 && !places)) return -1;
    const int groups = (tiles_m * tiles_n + 7) / 8 * 8;
    for (int i = 0; i < min(groups, room); ++i) {
        const TilePlace place = tile_place(i, tiles_m, tiles_n, K % 64 != 0);
        places[i] = place.m < 0 ? -1 : place.m * tiles_n + place.n;
    }
    return groups;
}

// The order in which the workgroups of a product cut along k take its tiles and parts.
extern "C" int xrt_linear_part_order(int M, int N, int K, int mode, int whole_norm, int* by_parts, int* places, int room) {
    int rows = 0, columns = 0;
    const int parts = xrt_linear_parts(M, N, K, mode, whole_norm, &rows, &columns);
    if (parts < 2 || !by_parts || (room > 0 && !places)) return -1;
    const long tiles_m = (M + rows - 1) / rows, tiles_n = ((mode == MODE_GATED ? 2L * N : N) + columns - 1) / columns;
    *by_parts = deals_by_parts(columns, tiles_m, tiles_n, K, parts);
    const long groups = part_ids(tiles_m * tiles_n, parts, *by_parts), in_a_row = *by_parts ? groups : groups / parts;
    if (groups >= (1L << 31)) return -1;
    for (long i = 0; i < min(groups, (long)room); ++i) {
        const PartPlace place = part_place((int)(i % in_a_row), (int)(i / in_a_row), (int)tiles_m, (int)tiles_n, *by_parts ? parts : 0);
        places[i] = place.tile.m < 0 ? -1 : (int)(place.part * tiles_m * tiles_n + place.tile.m * tiles_n + place.tile.n);
    }
    return (int)groups;
}

// Whether a product of 17 to 256 rows of x asks for w past the caches (k a multiple of 64).
extern "C" int xrt_linear_past_caches(int M, int N, int K, int mode) {
    if (M <= 16 || M > 256 || N <= 0 || K < (M <= SPLIT_BM ? 128 : 64) || K % 64 != 0 || mode < MODE_STORE || mode > MODE_GATED) return -1;
    const SplitPlan plan = split_plan(M, N, K, mode);
    if (plan.splits > 1) return M <= SPLIT_BM && parts_read_past_caches(plan.rows_w, K, mode == MODE_GATED);
    if (M > SPLIT_BM) {
        const int shape = xrt_linear_tiles(XRT_BF16, M, N, K, mode);
        if (shape != TILES_128_BY_64_FOUR_STAGES && shape != TILES_128_BY_128_THREE_STAGES) return 0;
    }
    return reads_past_caches(M <= SPLIT_BM ? SPLIT_BM : 128, M, N, K, mode);
}

// The first kernel alone of a bfloat16 product split along k (xrt_linear_split_takes says so and asks for a workspace): the sums of the parts,
// [parts][M][N], for a kernel that adds them itself. Returns the number of parts, or 0 on failure.
int xrt_linear_split_parts(const void* a, const void* w, int M, int N, int K, const Packing& packing, float* workspace, hipStream_t s) {
    const SplitPlan plan = split_plan(M, N, K, MODE_STORE);
    return launch_parts((const bf16*)a, (const bf16*)w, workspace, M, K, false, packing, plan, s) == 0 ? plan.splits : 0;
}
