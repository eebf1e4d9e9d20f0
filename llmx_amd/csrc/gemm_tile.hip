// LDS-tiled bf16 product for many rows (prompt portions): C[M,N] (+)= A[M,K] * W[N,K]^T on the matrix cores.
//
// A workgroup of 4 waves computes 64 rows x 128 features (each wave 32 rows x 64 features as 2 x 4 products of 16x16x32, so
// that the accumulators of the current run of K and of the runs before it fit in registers twice over); K is walked
// 64 at a time: the next A and W tiles travel from global memory into registers while the current ones are multiplied out
// of LDS (rows padded to 144 bytes so that the 16-byte operand reads of 8 consecutive rows fall into different banks).
// Grouped form: blockIdx.y walks the (expert, row tile) pairs of the experts that have rows; A's rows are gathered
// through the expert-sorted pair list and C's rows scattered to the pairs.  SwiGLU form: the tile's 128 weight rows
// are 64 gate rows and the 64 up rows of the same features, and silu(gate) * up is stored.
//
// Three forms of the lean loop share this arithmetic: 4 waves on 64 x 128 (three workgroups a CU), 4 waves on 128 x 128
// (each wave 64 x 64: fewer operand reads a product) and the wide form of 8 waves on 128 x 256 further down; the
// launcher says which runs when.
//
// The arithmetic of an output element is the weight-streaming kernel's, bit for bit: the same 16x16x32 instruction with
// the weights as its A operand and the same k-slots, K cut into the same `ks` runs of 32-wide steps, each run summed
// from zero in step order, the runs' sums added in run order.  So a row's result does not depend on whether its step
// held few rows or many.
#include "common.h"
#include "tile_choice.h"
#include <type_traits>

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));

enum : int { TL_STORE = 0, TL_ADD = 1, TL_SWIGLU = 2 };

#define TL_BN 128
#define TL_BK 64
#define TL_LD 72  // padded row length in bf16 elements (144 bytes)
// Dense products of fewer 64 x 128 tiles than this multiply K's runs in workgroups of their own (runs_apart_below).  One row tile: always
// while there are fewer tiles than CUs (the other kernel of up to 64 rows reads them again for every 16 features: 24,576 features of 4,096
// values, 48 rows 56 against 75 us; 28,672 of 6,144, 64 rows 82 against 167).  More rows: until the deep form below, which walks all of K
// in one workgroup, has enough tiles; long K and few rows in the last tile favour the runs (3,072 features of 6,144 values, runs apart
// against deep: 144 tiles 40 and 47 us, 192 tiles 47.4 and 45.5; of 8,192: 192 tiles 55 and 59; 8,192 features, 192 tiles: of 3,072 30.2 and
// 27.7, of 6,144 47.5 and 51.7; 65 rows of 8,192 features of 2,048: 16.3 and 17.7; 2,048 of 2,048: 64 tiles 14.3 and 15.4, 128 tiles 17.6 and
// 15.0; 4,096 of 16,384, 256 tiles: 134 and 123).
#define TILE_RUNS_APART_MOST 256
static int runs_apart_below(int M, int K) {
    if (M <= 64 || (M <= 192 && K >= 4096)) return TILE_RUNS_APART_MOST;
    const int tiles = 100 + K / (M <= 128 ? 64 : 80);
    return tiles < TILE_RUNS_APART_MOST ? tiles : TILE_RUNS_APART_MOST;
}
#define TL_DEEP_STAGES 3  // ... where no CU gets more than two workgroups (72 KB each): a tile asked for one ahead then arrives a whole trip to memory later, with nobody else to work meanwhile
#define TL_DEEP_MOST 512  // (K 8,192, 2,048 features: 512 rows 89 -> 55 us, 1,024 rows 92 -> 59, 2,048 rows 98 -> 87; four stages, one workgroup a CU: 53, 56, 104; 800 tiles of K 2,048, three a CU with two stages: 47 against 40, the wide form 34)
// Fewer rows: what bounds them is the weights' way from memory, which three workgroups a CU keep busier (two and three stages: 128 rows, 352
// tiles of 6,144 values 96 and 101 us, 368 of 12,288 187 and 206, 480 of 8,192 132 and 164, but 320 tiles of 8,192 109 and 88; 256 rows, 480 tiles of
// 12,288 170 and 180, 512 of 6,144 88 and 94, but 384 of 8,192 107 and 86).
static int deep_most(int M) { return M <= 128 ? 320 : M <= 256 ? 384 : TL_DEEP_MOST; }
#define TL_STAGES 2  // tiles in LDS in the lean loop: one being multiplied, the other on its way (48 KB: three workgroups a CU; measured better than deeper stages with fewer workgroups)

// Lane l of the wave: 16 bytes from base + offset (bytes, per lane) to LDS at lds + 16 l (lds the same for the whole
// wave).  Written as an instruction of its own so that waiting for it is the kernel's business: the loop below keeps
// two tiles' loads in flight and waits by count.
__device__ __forceinline__ void load_to_lds(const void* base, uint32_t offset, void* lds) {
    const uint32_t at = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) void*)lds;
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(at), "v"(offset), "s"(base) : "memory", "m0");
}
// The same for bytes that are read once: the caches are told not to keep them.
__device__ __forceinline__ void stream_to_lds(const void* base, uint32_t offset, void* lds) {
    const uint32_t at = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) void*)lds;
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2 nt" ::"s"(at), "v"(offset), "s"(base) : "memory", "m0");
}

// Four neighbouring features of one output row (n a multiple of 4): one 16-byte (float) or 8-byte (bfloat16) access
// when the row allows it, element by element at a ragged edge.  ADD: the values join what the row holds.
template <bool ADD, typename TC>
__device__ __forceinline__ void store_quad(TC* crow, int n, int N, bool rows_aligned, const float (&v)[4]) {
    if (rows_aligned && n + 3 < N) {
        if constexpr (std::is_same<TC, float>::value) {
            f32x4_t x = {v[0], v[1], v[2], v[3]};
            if (ADD) {
                const f32x4_t old = *reinterpret_cast<const f32x4_t*>(crow + n);
                x = f32x4_t{old[0] + x[0], old[1] + x[1], old[2] + x[2], old[3] + x[3]};
            }
            *reinterpret_cast<f32x4_t*>(crow + n) = x;
        } else {
            typedef uint32_t u32x2_t __attribute__((ext_vector_type(2)));
            const u32x2_t x = {(uint32_t)f32_to_bf16(v[0]) | ((uint32_t)f32_to_bf16(v[1]) << 16),
                               (uint32_t)f32_to_bf16(v[2]) | ((uint32_t)f32_to_bf16(v[3]) << 16)};
            *reinterpret_cast<u32x2_t*>(crow + n) = x;
        }
        return;
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        if (n + i >= N) continue;
        float x = v[i];
        if (ADD) x = ld(crow + n + i) + x;
        st(crow + n + i, x);
    }
}

// Which float32 results leave past the caches.  Kept, they are written back between the reads of weights that stream from memory and cost several times
// their bytes (down of 256 experts, 3,072 features of 1,536 values, us, half lines kept, whole lines kept, half lines streamed, whole lines streamed:
// 52 rows an expert 511, 510, 493, 477; 100 rows 608, 606, 575, 542).  Streamed, their reader finds them in memory instead of the last cache (256 MB), so
// both count.
// Routed, from 8 MB on.  Down and combine together, kept and streamed, us: 256 experts 6 MB 328 and 326, 8 MB 368 and 366, 31 MB 435 and 417, 60 MB 472 and
// 453, 117 MB 514 and 491, 156 MB 537 and 508 (503 + 34 and 470 + 38), 309 MB 658 and 611; 55 of 256 experts 60 MB 149 and 143, 192 MB 332 and 333;
// 64 experts (2,048 of 512) 12 MB 44 and 42, 48 MB 67 and 64, 96 MB 105 and 104; 16 experts (4,096 of 2,048) 8 MB 73 and 74; 8 experts nothing.
// Dense, where the results are a fifth of the last cache (48 MB), or the weights twice as large as it and the results 10 MB.  Whole passes of a model with
// its other results as they are, kept and streamed, us: 8,192 features of 3,072 values in four layers, 2,048 rows (64 MB) 6,267 and 6,195,
// 1,745 rows 7,163 and 7,132; 9,216 of 2,048 (72 MB) 5,477 and 5,373, but 900 rows (32 MB) 3,428 and 3,446; 3,072 of 2,048, 900 and 1,999
// rows 3,374 and 3,388, 5,532 and 5,538; 2,048 of 2,048, 1,999 rows 5,532 and 5,546; smaller results go either way (520 rows of 8,192 of 3,072 4,103
// and 4,088, 900 rows of 4,096 of 128 3,374 and 3,390).  A product and a copy of its results: 65,536 features of 2,048 values 25 MB 74 and 76, 50 MB
// 159 and 135; 28,672 of 4,096 22 MB 79 and 82, 56 MB 162 and 153, 224 MB 554 and 568; 16,384 of 8,192 32 MB 147 and 149, 64 MB 290 and 287; a
// head of 200,064 of 3,072 (1.2 GB) 13 MB 229 and 223, 49 MB 264 and 254, 76 MB 295 and 269, of 151,936 of 2,048 (0.6 GB) 7 MB 122 and 124,
// 14 MB 135 and 131, of 131,072 of 2,048 (0.54 GB) 5 MB 129 and 130, 12 MB 139 and 138.
// Only whole lines: rows that begin within one lose (9,220 of 3,072, 1,024 rows 99 and 106; 256 experts, 3,076 features, 192 MB 585 and 614).
#define TILE_STREAM_ROUTED (8L << 20)
#define TILE_STREAM_DENSE (48L << 20)
#define TILE_STREAM_HEAD (10L << 20)
#define TILE_STREAM_HEAD_WEIGHTS (512L << 20)
extern "C" int llmx_gemm_tile_streams_out(const void* C, int M, int N, int K, int ldc, int n_groups) {
    const long results = (long)M * N * (long)sizeof(float), weights = (long)N * K * (long)sizeof(bf16_t);
    if (N % 4 || ldc % 32 || ((uintptr_t)C & 127)) return 0;
    if (n_groups > 0) return results >= TILE_STREAM_ROUTED;
    return results >= TILE_STREAM_DENSE || (results >= TILE_STREAM_HEAD && weights >= TILE_STREAM_HEAD_WEIGHTS);
}

// Sixteen rows of two neighbouring tiles of 16 features, float32 (a lane: row lane % 16, features 4 (lane / 16) .. of either), stored as whole
// lines of 128 bytes that the caches do not keep: lanes 8 apart exchange quads (as weight_lines.h's do), so that an instruction stores 32
// features of eight rows.  line(0) and line(8) are the lane's rows lane % 8 and 8 + lane % 8 of C, null where the tile has none; n: of the even tile.
template <typename Line>
__device__ __forceinline__ void store_lines(const f32x4_t& even, const f32x4_t& odd, int n, int N, Line line) {
    f32x4_t lo, hi;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        lo[i] = __uint_as_float((uint32_t)__builtin_amdgcn_update_dpp((int)__float_as_uint(even[i]), (int)__float_as_uint(odd[i]), 0x128, 0xf, 0xc, false));
        hi[i] = __uint_as_float((uint32_t)__builtin_amdgcn_update_dpp((int)__float_as_uint(odd[i]), (int)__float_as_uint(even[i]), 0x128, 0xf, 0x3, false));
    }
    n += 2 * (threadIdx.x & 8);
    if (n >= N) return;
    float* const first = line(0);
    float* const second = line(8);
    if (first) __builtin_nontemporal_store(lo, reinterpret_cast<f32x4_t*>(first + n));
    if (second) __builtin_nontemporal_store(hi, reinterpret_cast<f32x4_t*>(second + n));
}

struct TileArgs {
    const bf16_t* A;
    const bf16_t* W;
    void* C;
    int M, N, K;
    int lda, ldc;
    const int* group_offsets;  // grouped: [G+1]
    const int* list;
    int n_groups, a_div;
    long w_group_stride;
    int up_offset;
    int m_tiles;  // dense: number of row tiles
    int ks;       // runs K is cut into (the weight-streaming kernel's waves per strip for this shape)
    int bm;       // rows a workgroup covers: 64 or 128
    const int* tile_stats;  // grouped, optional: the sum over groups of ceil(rows / 128); with choice_bit >= 0 the grouping's choice
    int choice_bit;         // ... whose bit this is: set where this product takes tiles of 128 rows
    int choice_without;     // ... where the grouping chose for tickets and this product takes none
    int run_if_big;         // with tile_stats: 1: this launch works only if the product takes tiles of 128 rows, 0: only if not
    int strip_runs;         // dense: XCDs take contiguous runs of tiles, strip after strip (see tile_place)
    int run_tiles;          // dense lean form, > 0: workgroup z multiplies only K's run z (this many 64-wide tiles) and stores its sums at C + z * M * ldc
    int act;                // TL_STORE, TL_ADD: an activation applied to the product (LLMX_ACT_*; a launch of runs' sums leaves it to the kernel that adds them)
    const float* act_params;
    GluArgs glu;            // TL_SWIGLU: the gated unit and its per-row values
    int stream_out;         // float32 results that go past the caches (see store_lines)
    int* ticket;            // grouped wide form, optional: 0, and 0 again afterwards; workgroups take tile after tile by it
};

// Whether this launch is the one that works: the grouping's own choice says which tiles the product takes; for a caller
// that brings the bare count, tiles of 128 rows where they hold at most 1.6 times the rows (measured on
// the prompt's routing on one machine: a 2,048-token step takes 30.9 ms with the bound at 1.25, 30.3 ms at 1.6, 30.2 ms at 2).  The launcher
// cannot know (the counts are on the device), so it launches the form for either case and one of them leaves at once.
__device__ __forceinline__ bool tile_launch_runs(const TileArgs& g) {
    if (!g.tile_stats) return true;
    const int stat = g.tile_stats[0];
    const bool big = g.choice_bit >= 0 ? ((g.choice_without ? stat ^ stat >> 4 : stat) >> g.choice_bit) & 1 : (long)stat * 128 * 5 <= (long)g.M * 8;
    return big == (g.run_if_big != 0);
}

// Which tile a workgroup takes.  Workgroups go round the 8 XCDs in launch order, each with an L2 of its own.  Strips of weights in a
// multiple of 8 stay on one XCD each as they are launched; any other number of them moves on from row tile to row tile: an odd one
// shows every XCD every strip, 2 more than a multiple of 4 half of them, 4 more than a multiple of 8 a quarter.  With strip_runs an XCD
// takes a contiguous run of tiles in the order strip after strip instead, a strip's row tiles together, and reads the rows' whole
// activations for every strip.
#define TILE_XCDS 8
#define TILE_CUS 256
template <bool GROUPED>
__device__ __forceinline__ void tile_place(const TileArgs& g, int at, int gx, int gy, int& strip, int& rows) {
    if (GROUPED || !g.strip_runs) {
        rows = at / gx;
        strip = at - rows * gx;
        return;
    }
    const int total = gx * gy;
    const int xcd = at % TILE_XCDS, share = total / TILE_XCDS, more = total % TILE_XCDS;
    const int tile = xcd * share + min(xcd, more) + at / TILE_XCDS;
    strip = tile / gy;
    rows = tile - strip * gy;
}
// Whether a dense product's strips go in runs, by their number and the row tiles' (wide: strips of 256 features, row tiles of 128; else 128
// and 64).  Odd numbers of strips gain at every size of several row tiles (2,048 rows of 2,048 values: 21 wide strips 67 -> 62 us, 35
// 119 -> 99, 43 127 -> 114; 1,024 rows, narrow: 21 28.8 -> 21.3, 27 34 -> 25).  Even ones lose while they are few (4,096 rows of 3,072, launch
// order and runs: 12 wide strips 89 and 92, 28 184 and 207, 30 197 and 216, 52 349 and 384, but 50 410 and 376, 84 640 and 590, 100 781 and 700;
// 1,024 rows of 4,096: 20 narrow ones 38 and 45, 28 41 and 52; 512 of 2,048: 84 36 and 46; 256 of 3,072: 100 43 and 48, but 114 56 and 47, 130 74
// and 56).  With one row tile nothing is shared and the order costs the division (48 rows: 0.3 of 10 us), until the strips are very many
// (5 rows of 2,048 values: 514 68 and 71, 1,188 143 and 129, 1,562 194 and 162; 65 rows: 594 wide 159 and 140).  Routed products keep
// the launch order: an expert's strips, side by side, stream one stretch of memory (256 experts of 3,072 x 3,072, 52 rows each: 916 us,
// strip after strip 1,010).
extern "C" int llmx_gemm_tile_strip_runs(int strips, int row_tiles, int wide) {
    if (strips % TILE_XCDS == 0) return 0;
    if (row_tiles == 1) return strips >= (wide ? 512 : 1024);
    if (strips % 2) return 1;
    if (wide) return strips >= (strips % 4 ? 48 : 80);
    return strips % 4 && strips >= 96 && row_tiles > 2;
}

// FAST: K is a multiple of 64 and the runs end on multiples of 64, so nothing in the loop needs a bound: the tiles are
// loaded without conditions (a row past the tile's rows reads the first row, a feature past N the last; what they
// produce is never stored, and a column of the product never touches another), straight into LDS, STAGES deep,
// one barrier a tile.
template <int EPI, typename TC, bool GROUPED, bool SPLIT, bool FAST, int BM, int STAGES = TL_STAGES>
__global__ void __launch_bounds__(256) gemm_tile_kernel(TileArgs g) {
    // FAST: STAGES tiles of unpadded 128-byte rows whose 16-byte chunks are swizzled; else one tile of padded rows
    __shared__ __attribute__((aligned(1024))) bf16_t As[FAST ? STAGES * BM * TL_BK : BM * TL_LD];
    __shared__ __attribute__((aligned(1024))) bf16_t Ws[FAST ? STAGES * TL_BN * TL_BK : TL_BN * TL_LD];
    __shared__ int rows_a[BM];
    __shared__ int rows_c[BM];
    __shared__ int tile_info[4];
    __shared__ int scan_waves[4];

    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    const bool runs = !GROUPED || tile_launch_runs(g);   // looked at below, once the first offsets are asked for too
    constexpr int FEATS = (EPI == TL_SWIGLU) ? 64 : 128;  // output features a workgroup covers
    int strip, row_tile;
    if (GROUPED || !g.strip_runs) {
        strip = blockIdx.x;
        row_tile = blockIdx.y;
    } else {
        tile_place<GROUPED>(g, (int)(blockIdx.y * gridDim.x + blockIdx.x), gridDim.x, gridDim.y, strip, row_tile);
    }
    const int n0 = strip * FEATS;
    const bf16_t* W = g.W;
    int row_begin, row_end;
    if (GROUPED) {
        // which (expert, row tile) this workgroup has: experts in order, each with ceil(rows / 64) tiles
        // found by all threads together: 256 experts a round, their tile counts scanned within waves and across them
        if (tid == 0) tile_info[0] = -1;
        int base = 0;
        for (int e0 = 0; e0 < g.n_groups; e0 += 256) {
            const int e = e0 + tid;
            const int begin = e < g.n_groups ? g.group_offsets[e] : 0;
            const int end = e < g.n_groups ? g.group_offsets[e + 1] : 0;
            if (!runs) return;   // the whole workgroup: the other tile size has this product
            const int tiles = (end - begin + BM - 1) / BM;
            int incl = tiles;
#pragma unroll
            for (int d = 1; d < 64; d <<= 1) {
                const int o = __shfl_up(incl, d, 64);
                if (lane >= d) incl += o;
            }
            if (lane == 63) scan_waves[wave] = incl;
            __syncthreads();
            int before = base;
            for (int w = 0; w < wave; ++w) before += scan_waves[w];
            const int round_total = scan_waves[0] + scan_waves[1] + scan_waves[2] + scan_waves[3];
            const int first = before + incl - tiles;
            if (row_tile >= first && row_tile < first + tiles) {
                tile_info[0] = e;
                tile_info[1] = begin + (row_tile - first) * BM;
                tile_info[2] = end;
                tile_info[3] = tiles;
            }
            base += round_total;
            __syncthreads();
            if (row_tile < base) break;
        }
        __syncthreads();
        const int e = tile_info[0];
        if (e < 0) return;
        row_begin = tile_info[1];
        row_end = min(tile_info[2], row_begin + BM);
        W += (size_t)e * g.w_group_stride;
    } else {
        row_begin = row_tile * BM;
        row_end = min(g.M, row_begin + BM);
    }
    if (tid < BM) {
        const int m = row_begin + tid;
        int ra = -1, rc = -1;
        if (m < row_end) {
            if (GROUPED) {
                const int p = g.list[m];
                ra = p / g.a_div;
                rc = p;
            } else {
                ra = rc = m;
            }
        }
        rows_a[tid] = ra;
        rows_c[tid] = rc;
    }
    __syncthreads();

    // global -> register staging in chunks of 16 bytes: W 1024 chunks (4 a thread), A 512 (2 a thread); chunk c: row c/8, k offset (c%8)*8
    const int K = g.K;
    const bf16_t* a_src[4];
    const bf16_t* w_src[4];
    uint32_t a_off[4], w_off[4];   // the same places as byte offsets from A and W (the lean loop adds them to a uniform base)
    bool a_ok[4], w_ok[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int c = tid + 256 * i;
        const int row = c >> 3, kc = (c & 7) * 8;
        a_ok[i] = false;
        a_src[i] = g.A;
        a_off[i] = 0;
        if (i < BM / 32) {
            const int ra = rows_a[row];
            a_ok[i] = ra >= 0;
            a_src[i] = g.A + (size_t)(ra >= 0 ? ra : 0) * g.lda + kc;
            a_off[i] = (uint32_t)(((size_t)(ra >= 0 ? ra : 0) * g.lda + kc) * sizeof(bf16_t));
        }
        int wr;
        if (EPI == TL_SWIGLU) {
            const int f = n0 + (row & 63);
            w_ok[i] = f < g.N;
            wr = (row < 64 ? 0 : g.up_offset) + min(f, g.N - 1);
        } else {
            const int f = n0 + row;
            w_ok[i] = f < g.N;
            wr = min(f, g.N - 1);
        }
        w_src[i] = W + (size_t)wr * K + kc;
        w_off[i] = (uint32_t)(((size_t)wr * K + kc) * sizeof(bf16_t));
    }
    u32x4_t a_reg[4], w_reg[4];
    auto load_global = [&](int k0) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int kc = ((tid + 256 * i) & 7) * 8;
            const bool in = k0 + kc < K;
            if (FAST) {
                const char* a_base = reinterpret_cast<const char*>(g.A + k0);
                const char* w_base = reinterpret_cast<const char*>(W + k0);
                if (i < BM / 32) a_reg[i] = *reinterpret_cast<const u32x4_t*>(a_base + a_off[i]);
                w_reg[i] = *reinterpret_cast<const u32x4_t*>(w_base + w_off[i]);
            } else {
                if (i < BM / 32) a_reg[i] = (in && a_ok[i]) ? *reinterpret_cast<const u32x4_t*>(a_src[i] + k0) : u32x4_t{0u, 0u, 0u, 0u};
                w_reg[i] = (in && w_ok[i]) ? *reinterpret_cast<const u32x4_t*>(w_src[i] + k0) : u32x4_t{0u, 0u, 0u, 0u};
            }
        }
    };
    auto store_lds = [&](int buf = 0) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int c = tid + 256 * i;
            const int row = c >> 3, kc = (c & 7) * 8;
            if (i < BM / 32) *reinterpret_cast<u32x4_t*>(&As[buf * BM * TL_LD + row * TL_LD + kc]) = a_reg[i];
            *reinterpret_cast<u32x4_t*>(&Ws[buf * TL_BN * TL_LD + row * TL_LD + kc]) = w_reg[i];
        }
    };

    // wave (wm, wn): rows 32*wm .. (2 tiles of 16 rows), features: 4 tiles of 16 weight rows
    const int wm = wave >> 1, wn = wave & 1;
    const int lr = lane & 15, lk = (lane >> 4) * 8;
    int w_row[4];  // LDS rows of the wave's 4 feature tiles
#pragma unroll
    for (int f = 0; f < 4; ++f) {
        if (EPI == TL_SWIGLU)
            w_row[f] = (f < 2 ? 0 : 64) + 32 * wn + 16 * (f & 1) + lr;   // tiles 0,1: gate rows; tiles 2,3: the up rows of the same features
        else
            w_row[f] = 64 * wn + 16 * f + lr;
    }
    constexpr int TT = BM / 32;   // 16-row tiles a wave holds
    f32x4_t acc[4][TT], total[SPLIT ? 4 : 1][SPLIT ? TT : 1];
#pragma unroll
    for (int f = 0; f < 4; ++f)
#pragma unroll
        for (int t = 0; t < TT; ++t) acc[f][t] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
    const int steps_total = (K + 31) >> 5;
    const int per = (steps_total + g.ks - 1) / g.ks;   // 32-wide steps in a run
    int until_fold = per;                                // steps left in the current run
    bool first_run = true;

    if constexpr (FAST) {
        // Tiles travel from global memory straight into LDS (no registers in between), STAGES deep: while tile t
        // is multiplied, the tiles after it are on their way.  A wave's load instruction fills 1 KB of LDS, lane after
        // lane: 8 rows of 128 bytes.  Rows are not padded; instead chunk c (16 bytes) of row r sits at place
        // c ^ ((r >> 1) & 7) of the row, so that the operand reads of 16 rows at one k fall into different banks.  The
        // lane that fills place p of row r therefore fetches chunk p ^ ((r >> 1) & 7) of that row.
        constexpr int A_LOADS = BM / 32, LOADS = 4 + A_LOADS;   // load instructions a wave issues per tile
        // the 64-wide tiles of K this workgroup multiplies: all of them, or one run's (run_tiles > 0: the runs lie apart)
        const int t_first = g.run_tiles > 0 ? (int)blockIdx.z * g.run_tiles : 0;
        const int n_tiles = g.run_tiles > 0 ? min(K / TL_BK, t_first + g.run_tiles) : K / TL_BK;
        const int tiles_per_run = SPLIT ? per / 2 : n_tiles;
        uint32_t w_at[4], a_at[A_LOADS];
        const int place = lane & 7;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int r = 32 * wave + 8 * j + (lane >> 3);           // row of the W tile
            const int ch = place ^ ((r >> 1) & 7);
            int wr;
            if (EPI == TL_SWIGLU) wr = (r < 64 ? 0 : g.up_offset) + min(n0 + (r & 63), g.N - 1);
            else wr = min(n0 + r, g.N - 1);
            w_at[j] = (uint32_t)(((size_t)wr * K + 8 * ch) * sizeof(bf16_t));
        }
#pragma unroll
        for (int j = 0; j < A_LOADS; ++j) {
            const int r = (BM / 4) * wave + 8 * j + (lane >> 3);     // row of the A tile
            const int ch = place ^ ((r >> 1) & 7);
            const int ra = rows_a[r];
            a_at[j] = (uint32_t)(((size_t)(ra >= 0 ? ra : 0) * g.lda + 8 * ch) * sizeof(bf16_t));
        }
        const int wave_u = __builtin_amdgcn_readfirstlane(wave);
        // a tile of few rows, weights that no other row tile reads: see the wide form
        const bool read_once = __builtin_amdgcn_readfirstlane(GROUPED ? tile_info[3] : g.m_tiles) == 1;
        const int rows_here = row_end - row_begin;
        const bool brings_rows = (BM / 4) * wave_u < rows_here, works = BM / 2 * __builtin_amdgcn_readfirstlane(wm) < rows_here;
        auto issue = [&](int t, int stage) {
            const bf16_t* wb = W + (size_t)t * TL_BK;
            const bf16_t* ab = g.A + (size_t)t * TL_BK;
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                void* to = &Ws[(stage * TL_BN + 32 * wave_u + 8 * j) * TL_BK];
                if (read_once) stream_to_lds(wb, w_at[j], to);
                else load_to_lds(wb, w_at[j], to);
            }
            if (STAGES > 2 || brings_rows) {
#pragma unroll
                for (int j = 0; j < A_LOADS; ++j) load_to_lds(ab, a_at[j], &As[(stage * BM + (BM / 4) * wave_u + 8 * j) * TL_BK]);
            }
        };
        // operand reads: row `row` of a stage, chunk kk/8 + lane/16
        int w_rd[4], a_rd[TT], w_swz[4], a_swz[TT];
#pragma unroll
        for (int f = 0; f < 4; ++f) {
            w_rd[f] = w_row[f] * TL_BK;
            w_swz[f] = (w_row[f] >> 1) & 7;
        }
#pragma unroll
        for (int q = 0; q < TT; ++q) {
            const int r = BM / 2 * wm + 16 * q + lr;
            a_rd[q] = r * TL_BK;
            a_swz[q] = (r >> 1) & 7;
        }
        const int kg = lane >> 4;
        auto multiply = [&](int stage) {
            const bf16_t* ws = &Ws[stage * TL_BN * TL_BK];
            const bf16_t* as = &As[stage * BM * TL_BK];
            // the operands of both halves of the tile are asked for at once; the second half's arrive while the first is multiplied
            bf16x8_t wf[2][4], af[2][TT];
#pragma unroll
            for (int hk = 0; hk < 2; ++hk) {
                const int kk = 32 * hk;
#pragma unroll
                for (int f = 0; f < 4; ++f)
                    wf[hk][f] = __builtin_bit_cast(bf16x8_t, *reinterpret_cast<const u32x4_t*>(&ws[w_rd[f] + 8 * ((kk / 8 + kg) ^ w_swz[f])]));
#pragma unroll
                for (int q = 0; q < TT; ++q)
                    af[hk][q] = __builtin_bit_cast(bf16x8_t, *reinterpret_cast<const u32x4_t*>(&as[a_rd[q] + 8 * ((kk / 8 + kg) ^ a_swz[q])]));
            }
#pragma unroll
            for (int hk = 0; hk < 2; ++hk)
#pragma unroll
                for (int f = 0; f < 4; ++f)
#pragma unroll
                    for (int q = 0; q < TT; ++q) acc[f][q] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[hk][f], af[hk][q], acc[f][q], 0, 0, 0);
            // order: the first half's reads, then a read of the second half after every multiplication while they last
            __builtin_amdgcn_sched_group_barrier(0x100, 4 + TT, 0);
#pragma unroll
            for (int sg = 0; sg < 4 + TT; ++sg) {
                __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
            }
            __builtin_amdgcn_sched_group_barrier(0x008, 8 * TT - (4 + TT), 0);
        };
        issue(t_first, 0);
#pragma unroll
        for (int ahead = 1; ahead < STAGES - 1; ++ahead)
            if (t_first + ahead < n_tiles) issue(t_first + ahead, ahead);
        int t = t_first, stage = 0;
        for (int run_end = tiles_per_run;; run_end += tiles_per_run) {
            const int stop = min(run_end, n_tiles);
            for (; t < stop; ++t) {
                // tile t has arrived when at most the loads of tile t+1 are still out; then everybody's have, and
                // everybody is done with the stage that tile t+2 goes into
                constexpr int OUT = LOADS * (STAGES - 2);   // loads of the tiles after t that may still be out
                if (t + STAGES - 2 < n_tiles) __builtin_amdgcn_s_waitcnt(0x0F70 | (OUT & 15) | ((OUT >> 4) << 14));
                else __builtin_amdgcn_s_waitcnt(0x0F70);
                __syncthreads();
                if (t + STAGES - 1 < n_tiles) issue(t + STAGES - 1, stage == 0 ? STAGES - 1 : stage - 1);
                if (works) multiply(stage);
                stage = stage == STAGES - 1 ? 0 : stage + 1;
            }
            if (t >= n_tiles) break;
            if (SPLIT) {
                // a run of K ends: its sum joins the runs before it, in run order
#pragma unroll
                for (int f = 0; f < 4; ++f)
#pragma unroll
                    for (int q = 0; q < TT; ++q) {
                        if (first_run) total[f][q] = acc[f][q];
                        else total[f][q] = f32x4_t{total[f][q][0] + acc[f][q][0], total[f][q][1] + acc[f][q][1],
                                                   total[f][q][2] + acc[f][q][2], total[f][q][3] + acc[f][q][3]};
                        acc[f][q] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
                    }
                first_run = false;
            }
        }
    } else {
    load_global(0);
    store_lds();
    __syncthreads();
    for (int k0 = 0; k0 < K; k0 += TL_BK) {
        const bool more = k0 + TL_BK < K;
        if (more) load_global(k0 + TL_BK);
#pragma unroll
        for (int kk = 0; kk < TL_BK; kk += 32) {
            if (k0 + kk < K) {
                if (SPLIT && until_fold == 0) {
                    // a run of K ends: its sum joins the runs before it, in run order
#pragma unroll
                    for (int f = 0; f < 4; ++f)
#pragma unroll
                        for (int t = 0; t < TT; ++t) {
                            if (first_run) total[f][t] = acc[f][t];
                            else total[f][t] = f32x4_t{total[f][t][0] + acc[f][t][0], total[f][t][1] + acc[f][t][1],
                                                       total[f][t][2] + acc[f][t][2], total[f][t][3] + acc[f][t][3]};
                            acc[f][t] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
                        }
                    first_run = false;
                    until_fold = per;
                }
                bf16x8_t wf[4], af[TT];
#pragma unroll
                for (int f = 0; f < 4; ++f) wf[f] = __builtin_bit_cast(bf16x8_t, *reinterpret_cast<const u32x4_t*>(&Ws[w_row[f] * TL_LD + kk + lk]));
#pragma unroll
                for (int t = 0; t < TT; ++t)
                    af[t] = __builtin_bit_cast(bf16x8_t, *reinterpret_cast<const u32x4_t*>(&As[(BM / 2 * wm + 16 * t + lr) * TL_LD + kk + lk]));
#pragma unroll
                for (int f = 0; f < 4; ++f)
#pragma unroll
                    for (int t = 0; t < TT; ++t) acc[f][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[f], af[t], acc[f][t], 0, 0, 0);
                --until_fold;
            }
        }
        __syncthreads();
        if (more) {
            store_lds();
            __syncthreads();
        }
    }
    }
    if (SPLIT && !first_run) {
#pragma unroll
        for (int f = 0; f < 4; ++f)
#pragma unroll
            for (int t = 0; t < TT; ++t)
                acc[f][t] = f32x4_t{total[f][t][0] + acc[f][t][0], total[f][t][1] + acc[f][t][1], total[f][t][2] + acc[f][t][2],
                                    total[f][t][3] + acc[f][t][3]};
    }

    // acc[f][t][i]: feature (tile f) 4*(lane/16) + i, row 32*wm + 16*t + lane%16
    const int fq = 4 * (lane >> 4);
    const bool rows_aligned = g.ldc % 4 == 0 && ((uintptr_t)g.C & 15) == 0;   // a lane's four features make one access
    const ActFn act(EPI == TL_STORE ? g.act : LLMX_ACT_NONE, g.act_params);      // formed once, as in the wide form
    if constexpr (FAST && EPI == TL_STORE && std::is_same<TC, float>::value) {
        if (g.stream_out) {
#pragma unroll
            for (int t = 0; t < TT; ++t) {
                float* at[2];
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    const int rc = rows_c[BM / 2 * wm + 16 * t + 8 * h + (lr & 7)];
                    at[h] = rc >= 0 ? (float*)g.C + (size_t)rc * g.ldc : nullptr;
                }
#pragma unroll
                for (int f = 0; f < 4; f += 2) store_lines(acc[f][t], acc[f + 1][t], n0 + 64 * wn + 16 * f + fq, g.N, [&](int d) { return at[d >> 3]; });
            }
            return;
        }
    }
#pragma unroll
    for (int t = 0; t < TT; ++t) {
        const int rc = rows_c[BM / 2 * wm + 16 * t + lr];
        if (rc < 0) continue;
        TC* crow = (TC*)g.C + (size_t)rc * g.ldc + (g.run_tiles > 0 ? (size_t)blockIdx.z * g.M * g.ldc : 0);
        if (EPI == TL_SWIGLU) {
            const GluRow glu(g.glu, rc);
#pragma unroll
            for (int f = 0; f < 2; ++f) {
                float v[4];
#pragma unroll
                for (int i = 0; i < 4; ++i) v[i] = glu(acc[f][t][i], acc[f + 2][t][i]);
                store_quad<false>(crow, n0 + 32 * wn + 16 * f + fq, g.N, rows_aligned, v);
            }
        } else {
#pragma unroll
            for (int f = 0; f < 4; ++f) {
                float v[4] = {acc[f][t][0], acc[f][t][1], acc[f][t][2], acc[f][t][3]};
                if (llmx_act_reads_vector(g.act)) {
#pragma unroll
                    for (int i = 0; i < 4; ++i) v[i] = biased_act(g.act, v[i], act_feature(g.act, g.act_params, n0 + 64 * wn + 16 * f + fq + i, g.N));
                } else if (EPI == TL_STORE && g.act != LLMX_ACT_NONE) {
#pragma unroll
                    for (int i = 0; i < 4; ++i) v[i] = act(v[i]);
                }
                store_quad<EPI == TL_ADD>(crow, n0 + 64 * wn + 16 * f + fq, g.N, rows_aligned, v);
            }
        }
    }
}

// The wide form of the lean loop, for products with many rows a group: a workgroup of 8 waves computes 128 rows x 256
// weight rows (each wave 64 x 64 as 4 x 4 products), three tiles deep in LDS (144 KB: one workgroup a CU, two waves a
// SIMD).  What bounds the 4-wave form is the tiles' way into LDS: a 64 x 128 tile needs 24 KB per 1 MFLOP and a tile is
// asked for only one multiplication ahead, far less than the memory's latency; here 48 KB serve 4 MFLOP and two tiles
// (96 KB) are on their way while one is multiplied.  Per output element nothing differs from the other forms: the same
// instruction, the same k-slots, the same runs.
#define WD_BM 128
#define WD_BN 256
#define WD_STAGES 3
// The order within half a tile: an operand read after every two multiplications, so the reads are early and spread out.
#define WD_INTERLEAVE()                                      \
    do {                                                     \
        _Pragma("unroll") for (int sg = 0; sg < 8; ++sg) {   \
            __builtin_amdgcn_sched_group_barrier(0x100, 1, 0); \
            __builtin_amdgcn_sched_group_barrier(0x008, 2, 0); \
        }                                                    \
    } while (0)
//
// With one workgroup a CU nothing else works while a tile's place is looked up, its first weights are on their way and its sums are stored.
// So, for routed products whose caller brings a ticket counter, a workgroup stays on its CU and takes tile after tile: the next one is
// looked up while this one is multiplied, and its first K tiles are asked for as stages of LDS fall free; only the stores and one wait stand
// between two tiles.  The tiles are handed out in order by tickets, not in strides: the row tiles of one expert have to stay close in
// time for its weights to be found in the caches (strides, 256 experts of 300 rows, 3,072 features of 3,072 values: 2,423 -> 2,664 us), and
// a tile is drawn as late as it can be, when the one before the present is done (drawn a tile earlier 2,333 -> 2,436).
// A workgroup a tile and tickets, gate_up of these sizes, 256 experts: 64 rows an expert 865 -> 839 us, 100 941 -> 893, 130 1,287 -> 1,260,
// 170 1,599 -> 1,555, but 300 2,079 -> 2,333; 55 experts of 130 302 -> 294, of 200 395 -> 364, but of 100 211 -> 220, of 300 461 -> 497.
// BARE: nothing is applied to the sums but, gated, silu(gate) * up.  With the other units and activations in the loop over tiles their
// constants take the registers the sums need; those products launch a workgroup a tile, and dense ones too (nothing gained).
#define WD_MAX_GROUPS 1536      // groups whose row tiles and places are kept in LDS beside the stages
template <int EPI, typename TC, bool GROUPED, bool SPLIT, bool BARE>
__global__ void __launch_bounds__(512) gemm_wide_kernel(TileArgs g) {
    __shared__ __attribute__((aligned(1024))) bf16_t As[WD_STAGES * WD_BM * TL_BK];
    __shared__ __attribute__((aligned(1024))) bf16_t Ws[WD_STAGES * WD_BN * TL_BK];
    __shared__ int tiles_before[GROUPED ? WD_MAX_GROUPS + 1 : 1], places[GROUPED ? WD_MAX_GROUPS + 1 : 1];
    __shared__ int pairs[3][GROUPED ? WD_BM : 1];        // of the tile before (its sums may still be stored), this one and the next
    __shared__ int scan_waves[8];
    __shared__ int drawn;                                // the tile after this one

    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
    const bool runs = !GROUPED || tile_launch_runs(g);   // looked at below, once the first offsets are asked for too
    constexpr int HALF = WD_BN / 2;                               // SwiGLU: gate rows, then the up rows of the same features
    constexpr int FEATS = (EPI == TL_SWIGLU) ? HALF : WD_BN;      // output features a tile covers
    const int strips = (g.N + FEATS - 1) / FEATS;
    int row_tiles = g.m_tiles;
    if (GROUPED) {
        // experts in order, each with ceil(rows / 128) row tiles: how many lie before each expert's, and where its rows begin
        int base = 0;
        for (int e0 = 0; e0 < g.n_groups; e0 += 512) {
            const int e = e0 + tid;
            const int begin = e < g.n_groups ? g.group_offsets[e] : 0;
            const int end = e < g.n_groups ? g.group_offsets[e + 1] : 0;
            if (!runs) return;   // the whole workgroup: the other tile size has this product
            const int tiles = (end - begin + WD_BM - 1) / WD_BM;
            int incl = tiles;
#pragma unroll
            for (int d = 1; d < 64; d <<= 1) {
                const int o = __shfl_up(incl, d, 64);
                if (lane >= d) incl += o;
            }
            if (lane == 63) scan_waves[wave] = incl;
            __syncthreads();
            int before = base, round_total = 0;
            for (int w = 0; w < 8; ++w) {
                if (w < wave) before += scan_waves[w];
                round_total += scan_waves[w];
            }
            if (e < g.n_groups) {
                tiles_before[e] = before + incl - tiles;
                places[e] = begin;
                if (e == g.n_groups - 1) {
                    tiles_before[e + 1] = before + incl;
                    places[e + 1] = end;
                }
            }
            base += round_total;
            __syncthreads();
        }
        row_tiles = __builtin_amdgcn_readfirstlane(base);
    }
    const int total = strips * row_tiles;

    // a tile of the product: which weights, which rows (places in the list, if grouped)
    struct Tile {
        const bf16_t* W;
        int n0, row_begin, row_end, tiles;      // tiles: row tiles that read these weights
    };
    auto tile_at = [&](int at) {
        Tile t;
        int strip, row_tile;
        tile_place<GROUPED>(g, at, strips, row_tiles, strip, row_tile);
        t.n0 = strip * FEATS;
        t.W = g.W;
        if (GROUPED) {
            // the last expert with at most this many row tiles before its own (one without rows has as many as the next)
            int found = 0;
            for (int e0 = 0; e0 < g.n_groups; e0 += 64) found += __popcll(__ballot(e0 + lane < g.n_groups && tiles_before[min(e0 + lane, g.n_groups)] <= row_tile));
            const int e = __builtin_amdgcn_readfirstlane(found) - 1;
            const int first = __builtin_amdgcn_readfirstlane(tiles_before[e]), end = __builtin_amdgcn_readfirstlane(places[e + 1]);
            t.tiles = __builtin_amdgcn_readfirstlane(tiles_before[e + 1]) - first;
            t.row_begin = __builtin_amdgcn_readfirstlane(places[e]) + (row_tile - first) * WD_BM;
            t.row_end = min(end, t.row_begin + WD_BM);
            t.W += (size_t)e * g.w_group_stride;
        } else {
            t.tiles = g.m_tiles;
            t.row_begin = row_tile * WD_BM;
            t.row_end = min(g.M, t.row_begin + WD_BM);
        }
        return t;
    };

    const int K = g.K;
    // wave (wm, wn): rows 64 * wm .. (4 tiles of 16), 4 tiles of 16 weight rows
    const int wm = wave >> 2, wn = wave & 3;
    const int lr = lane & 15;
    constexpr int TT = 4;
    const int steps_total = (K + 31) >> 5;
    const int per = (steps_total + g.ks - 1) / g.ks;   // 32-wide steps in a run

    // the same unpadded, swizzled rows as the 4-wave form: chunk c (16 bytes) of row r sits at place c ^ ((r >> 1) & 7)
    constexpr int W_LOADS = 4, A_LOADS = 2, LOADS = W_LOADS + A_LOADS;   // load instructions a wave issues per tile
    const int n_tiles = K / TL_BK, last = n_tiles - 1;
    const int tiles_per_run = SPLIT ? per / 2 : n_tiles;
    const int place = lane & 7;
    // What the loads are of: weights from a base the workgroup shares, A's rows (those of the wave, where the tile has them).
    // A tile of few rows (an expert's last, or its only one) is not multiplied out to 128: a wave whose 16 rows of A lie past the tile's
    // rows leaves them unread, and with at most 64 rows the waves of the upper half only bring weights.  What LDS holds for such rows makes
    // columns of the product that are never stored.  Weights that no other row tile reads come as bytes read once, which the caches do not
    // keep; where several do, the later ones find them in the caches (all as read once: down of 2,048 rows 596 -> 719 us).  Both, gate_up (256
    // experts or some 60, 3,072 features of 3,072 values): 2,048 rows in 64 an expert 1,037 -> 984 us, in 300 602 -> 535; 37 prompts of 45
    // 1,050 -> 952; 64-row tiles: 64 rows in 221 experts 669 -> 601 (6.9 TB/s), 520 rows 752 -> 700, down of 64 rows 345 -> 318.
    const bf16_t* w_base;
    uint32_t w_at[W_LOADS], a_at[A_LOADS];
    bool brings_rows, read_once;
    auto rows_in = [&](const Tile& t) { return 16 * wave < t.row_end - t.row_begin; };
    auto ask_pairs = [&](const Tile& t, int slot) {
        if (GROUPED && tid < WD_BM) pairs[slot][tid] = g.list[min(t.row_begin + tid, t.row_end - 1)];
    };
    auto row_of = [&](const Tile& t, int slot, int r) { return GROUPED ? pairs[slot][r] : min(t.row_begin + r, t.row_end - 1); };
    auto adopt = [&](const Tile& t, int slot) {
        w_base = t.W;
        read_once = t.tiles == 1;
        brings_rows = rows_in(t);
#pragma unroll
        for (int j = 0; j < W_LOADS; ++j) {
            const int r = 32 * wave + 8 * j + (lane >> 3);           // row of the W tile
            int wr;
            if (EPI == TL_SWIGLU) wr = (r < HALF ? 0 : g.up_offset) + min(t.n0 + (r & (HALF - 1)), g.N - 1);
            else wr = min(t.n0 + r, g.N - 1);
            w_at[j] = (uint32_t)(((size_t)wr * K + 8 * (place ^ ((r >> 1) & 7))) * sizeof(bf16_t));
        }
#pragma unroll
        for (int j = 0; j < A_LOADS; ++j) {
            const int r = 16 * wave + 8 * j + (lane >> 3);           // row of the A tile
            const int ra = GROUPED ? row_of(t, slot, r) / g.a_div : row_of(t, slot, r);
            a_at[j] = (uint32_t)(((size_t)ra * g.lda + 8 * (place ^ ((r >> 1) & 7))) * sizeof(bf16_t));
        }
    };
    auto issue = [&](int t, int stage) {
        const bf16_t* wb = w_base + (size_t)t * TL_BK;
        const bf16_t* ab = g.A + (size_t)t * TL_BK;
        bf16_t* to = &Ws[(stage * WD_BN + 32 * wave) * TL_BK];
        if (read_once) {
#pragma unroll
            for (int j = 0; j < W_LOADS; ++j) stream_to_lds(wb, w_at[j], to + 8 * j * TL_BK);
        } else {
#pragma unroll
            for (int j = 0; j < W_LOADS; ++j) load_to_lds(wb, w_at[j], to + 8 * j * TL_BK);
        }
        if (brings_rows) {
#pragma unroll
            for (int j = 0; j < A_LOADS; ++j) load_to_lds(ab, a_at[j], &As[(stage * WD_BM + 16 * wave + 8 * j) * TL_BK]);
        }
    };
    // operand reads: rows 16 apart are swizzled alike, so a lane's places differ by constants.  SwiGLU: feature tiles 0,1: gate rows; 2,3:
    // the up rows of the same features
    const int kg = lane >> 4, swizzle = (lr >> 1) & 7;
    const int w_lane = ((EPI == TL_SWIGLU ? 32 : 64) * wn + lr) * TL_BK, a_lane = (64 * wm + lr) * TL_BK;
    f32x4_t acc[4][TT], sum[SPLIT ? 4 : 1][SPLIT ? TT : 1];
    // the operands of one half (32 of k) of a stage's tile
    auto read_half = [&](int stage, int kk, bf16x8_t (&wf)[4], bf16x8_t (&af)[TT]) {
        const int chunk = 8 * ((kk / 8 + kg) ^ swizzle);
        const bf16_t* ws = &Ws[stage * WD_BN * TL_BK + w_lane + chunk];
        const bf16_t* as = &As[stage * WD_BM * TL_BK + a_lane + chunk];
#pragma unroll
        for (int f = 0; f < 4; ++f) {
            const int row = EPI == TL_SWIGLU ? (f < 2 ? 0 : HALF) + 16 * (f & 1) : 16 * f;
            wf[f] = __builtin_bit_cast(bf16x8_t, *reinterpret_cast<const u32x4_t*>(&ws[row * TL_BK]));
        }
#pragma unroll
        for (int q = 0; q < TT; ++q) af[q] = __builtin_bit_cast(bf16x8_t, *reinterpret_cast<const u32x4_t*>(&as[16 * q * TL_BK]));
    };
    auto multiply_half = [&](const bf16x8_t (&wf)[4], const bf16x8_t (&af)[TT]) {
#pragma unroll
        for (int f = 0; f < 4; ++f)
#pragma unroll
            for (int q = 0; q < TT; ++q) acc[f][q] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[f], af[q], acc[f][q], 0, 0, 0);
    };
    const int fq = 4 * (lane >> 4);
    const bool rows_aligned = g.ldc % 4 == 0 && ((uintptr_t)g.C & 15) == 0;   // a lane's four features make one access
    // The activation's numbers formed once: behind the stores, which may write what it reads, they were formed for every tile
    // (a softplus pair 16 times a thread: 2,048 rows, 2,048 -> 8,192 features with xIELU 126 -> 101 us).
    const ActFn act(!BARE && EPI == TL_STORE ? g.act : LLMX_ACT_NONE, g.act_params);

    // Three K tiles in LDS; while a tile's first half is multiplied its second half's operands are read, and while the
    // second half is multiplied the next tile's first: the matrix cores and LDS work at the same time, also within a
    // wave.  One barrier a tile, in its middle: by then a wave has all operands of tile t in registers, so after the
    // barrier tile t's stage takes tile t+3 (past K's end: the next tile of the product's first ones), and tile t+1
    // (awaited before the barrier) can be read by everybody.
    if ((int)blockIdx.x >= total) return;
    // A workgroup's first tile is its number's; the others it draws, each when the tile before the present is stored, until one is none.  So every
    // workgroup draws one that is none, and who draws the last of all puts the counter back.
    const bool tickets = BARE && GROUPED && g.ticket != nullptr && total > (int)gridDim.x;       // (K of at least four K tiles: TILE_TICKETS_MIN_K)
    const int firsts = min((int)gridDim.x, total);
    int ticket = 0;
    if (tid == 0 && tickets) ticket = atomicAdd(g.ticket, 1);
    Tile tile = tile_at(blockIdx.x), next = tile;
    int stage = 0, slot = 0;
    ask_pairs(tile, 0);
    if (GROUPED) __syncthreads();
    adopt(tile, 0);
    for (int t = 0; t < min(3, n_tiles); ++t) issue(t, t);
    for (;;) {
        const int rows_here = tile.row_end - tile.row_begin;
        const bool works = 64 * wm < rows_here;
        __builtin_amdgcn_s_waitcnt(0x0070);     // the first three K tiles, the stores of the tile before, the ticket
        if (tid == 0) {
            if (tickets && ticket == total - 1) atomicExch(g.ticket, 0);
            drawn = tickets ? firsts + ticket : total;
        }
        __syncthreads();
        const int following = __builtin_amdgcn_readfirstlane(drawn);
        const bool more = BARE && GROUPED && following < total;
        const bool brings_now = brings_rows;
        const int slot_next = slot == 2 ? 0 : slot + 1;
        if (more) {
            next = tile_at(following);
            ask_pairs(next, slot_next);
        }
        const bool brings_next = rows_in(next);
        auto ask = [&](int t, int into) {
            if (t < n_tiles) {
                issue(t, into);
            } else if (more) {
                if (t == n_tiles) adopt(next, slot_next);
                issue(t - n_tiles, into);
            }
        };
        // until at most the loads of tile t are on their way (LDS reads awaited too where the wave makes any)
        auto wait_but = [&](int t) {
            if (t >= n_tiles && !more) __builtin_amdgcn_s_waitcnt(0x0070);
            else if (t < n_tiles ? brings_now : brings_next) __builtin_amdgcn_s_waitcnt(0x0070 | LOADS);
            else __builtin_amdgcn_s_waitcnt(0x0070 | W_LOADS);
        };
        auto last_stage_read = [&]() {          // by this wave, then by all: the stage takes one more K tile of the next tile
            __builtin_amdgcn_s_waitcnt(0xC07F);
            __syncthreads();
            ask(n_tiles + 2, stage);
            stage = stage == 2 ? 0 : stage + 1;
        };
        if (!works) {
            for (int t = 0; t < last; ++t) {
                wait_but(t + 2);
                __syncthreads();
                ask(t + 3, stage);
                stage = stage == 2 ? 0 : stage + 1;
            }
            last_stage_read();
        } else {
#pragma unroll
            for (int f = 0; f < 4; ++f)
#pragma unroll
                for (int q = 0; q < TT; ++q) {
                    acc[f][q] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
                    if (SPLIT) sum[f][q] = acc[f][q];        // (written before it is read anyway: said here, it need not live from tile to tile)
                }
            bool first_run = true;
            bf16x8_t wf_a[4], af_a[TT], wf_b[4], af_b[TT];
            read_half(stage, 0, wf_a, af_a);
            auto step = [&](int t, auto inside) {       // inside: K tile t + 3 is one of this tile's
                read_half(stage, 32, wf_b, af_b);
                multiply_half(wf_a, af_a);
                WD_INTERLEAVE();
                const int after = stage == 2 ? 0 : stage + 1;
                // this wave's operand reads of tile t are done, and its part of tile t+1 has arrived (tile t+2's may be out)
                if (!decltype(inside)::value) wait_but(t + 2);
                else if (brings_now) __builtin_amdgcn_s_waitcnt(0x0070 | LOADS);
                else __builtin_amdgcn_s_waitcnt(0x0070 | W_LOADS);
                __syncthreads();
                if (decltype(inside)::value) issue(t + 3, stage);
                else ask(t + 3, stage);
                read_half(after, 0, wf_a, af_a);
                multiply_half(wf_b, af_b);
                WD_INTERLEAVE();
                stage = after;
            };
            int t = 0;      // the last tile has no tile after it: it runs after the loop, so the loop's body has no branch around its reads
            for (int run_end = tiles_per_run;; run_end += tiles_per_run) {
                const int stop = min(run_end, last);
                for (; t < min(stop, n_tiles - 3); ++t) step(t, std::true_type{});
                for (; t < stop; ++t) step(t, std::false_type{});
                if (SPLIT && t == run_end && t < n_tiles) {
                    // a run of K ends: its sum joins the runs before it, in run order
#pragma unroll
                    for (int f = 0; f < 4; ++f)
#pragma unroll
                        for (int q = 0; q < TT; ++q) {
                            if (first_run) sum[f][q] = acc[f][q];
                            else sum[f][q] = f32x4_t{sum[f][q][0] + acc[f][q][0], sum[f][q][1] + acc[f][q][1], sum[f][q][2] + acc[f][q][2],
                                                     sum[f][q][3] + acc[f][q][3]};
                            acc[f][q] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
                        }
                    first_run = false;
                }
                if (t >= last) break;
            }
            read_half(stage, 32, wf_b, af_b);
            multiply_half(wf_a, af_a);
            multiply_half(wf_b, af_b);
            if (SPLIT && !first_run) {
#pragma unroll
                for (int f = 0; f < 4; ++f)
#pragma unroll
                    for (int q = 0; q < TT; ++q)
                        acc[f][q] = f32x4_t{sum[f][q][0] + acc[f][q][0], sum[f][q][1] + acc[f][q][1], sum[f][q][2] + acc[f][q][2],
                                            sum[f][q][3] + acc[f][q][3]};
            }
            last_stage_read();

            // acc[f][q][i]: feature (tile f) 4*(lane/16) + i, row 64*wm + 16*q + lane%16
            const bool lines = BARE && EPI == TL_STORE && std::is_same<TC, float>::value && g.stream_out;
            if (lines) {
#pragma unroll
                for (int q = 0; q < TT; ++q) {
                    float* at[2];
#pragma unroll
                    for (int h = 0; h < 2; ++h) {
                        const int m = 64 * wm + 16 * q + 8 * h + (lr & 7);
                        at[h] = m < rows_here ? (float*)g.C + (size_t)row_of(tile, slot, m) * g.ldc : nullptr;
                    }
#pragma unroll
                    for (int f = 0; f < 4; f += 2) {
                        // (copies, as below)
                        f32x4_t even = acc[f][q], odd = acc[f + 1][q];
#pragma unroll
                        for (int i = 0; i < 4; ++i) {
                            float x = even[i], y = odd[i];
                            asm volatile("" : "+v"(x), "+v"(y));
                            even[i] = x;
                            odd[i] = y;
                        }
                        store_lines(even, odd, tile.n0 + 64 * wn + 16 * f + fq, g.N, [&](int d) { return at[d >> 3]; });
                    }
                }
            }
#pragma unroll
            for (int q = 0; q < TT; ++q) {
                if (lines) break;
                if (64 * wm + 16 * q + lr >= rows_here) continue;
                const int rc = row_of(tile, slot, 64 * wm + 16 * q + lr);
                TC* crow = (TC*)g.C + (size_t)rc * g.ldc;
                if (EPI == TL_SWIGLU) {
                    const GluRow glu(BARE ? GluArgs{LLMX_GLU_SILU, 0.0f, nullptr, nullptr, 0} : g.glu, rc);
#pragma unroll
                    for (int f = 0; f < 2; ++f) {
                        float v[4];
#pragma unroll
                        for (int i = 0; i < 4; ++i) v[i] = glu(acc[f][q][i], acc[f + 2][q][i]);
                        store_quad<false>(crow, tile.n0 + 32 * wn + 16 * f + fq, g.N, rows_aligned, v);
                    }
                } else {
#pragma unroll
                    for (int f = 0; f < 4; ++f) {
                        const int n = tile.n0 + 64 * wn + 16 * f + fq;
                        float v[4] = {acc[f][q][0], acc[f][q][1], acc[f][q][2], acc[f][q][3]};
                        // a copy of the sums: stored as they are, the compiler lays them out for the stores from the first product on
                        // (and spills a hundred registers in the loop)
#pragma unroll
                        for (int i = 0; i < 4; ++i) asm volatile("" : "+v"(v[i]));
                        if (!BARE && llmx_act_reads_vector(g.act)) {
#pragma unroll
                            for (int i = 0; i < 4; ++i) v[i] = biased_act(g.act, v[i], act_feature(g.act, g.act_params, n + i, g.N));
                        } else if (!BARE && EPI == TL_STORE && g.act != LLMX_ACT_NONE) {
#pragma unroll
                            for (int i = 0; i < 4; ++i) v[i] = act(v[i]);
                        }
                        store_quad<EPI == TL_ADD>(crow, n, g.N, rows_aligned, v);
                    }
                }
            }
        }
        if (!BARE || !more) return;
        if (tid == 0) ticket = atomicAdd(g.ticket, 1);
        tile = next;
        slot = slot_next;
    }
}

// form: which kernel takes the product.  The lean forms need whole 64-wide tiles of K, runs that end on them, and
// operands whose byte offsets fit 32 bits (llmx_gemm_tile_offsets_fit).
enum : int { FORM_64 = 0, FORM_128 = 1, FORM_WIDE = 2, FORM_BOUNDED = 3, FORM_64_DEEP = 4 };
// Routed products' tiles of 128 rows: the wide form for long K and wherever tiles are taken by tickets (256 experts, 3,072 features of 1,536 values, four
// waves a tile and the wide form, us: 64 rows an expert 558 and 524, 100 612 and 575, 130 731 and 709, 170 855 and 861; of 1,792 170 964 and
// 998, 199 1,024 and 1,004; 55 experts of 300 rows, some 60 a group, 281 and 287; 2,048 features of 1,024 values, 100 rows 319 and 277).
static bool wide_routed(int K, const int* ticket) { return K >= 2048 || ticket; }

// The sums are stored as they are or, gated, as silu(gate) * up.
static bool nothing_applied(const TileArgs& g, int epi) {
    return epi == TL_SWIGLU ? g.glu.kind == LLMX_GLU_SILU && !g.glu.row_scale && !g.glu.row_gate : g.act == LLMX_ACT_NONE;
}

template <int EPI, typename TC, bool GROUPED, bool SPLIT>
static void tile_launch_form(const TileArgs& g, int form, dim3 grid, hipStream_t stream) {
    if (form == FORM_WIDE) {
        const unsigned tiles = grid.x * grid.y;
        if (nothing_applied(g, EPI)) hipLaunchKernelGGL((gemm_wide_kernel<EPI, TC, GROUPED, SPLIT, true>), dim3(g.ticket && tiles > TILE_CUS ? TILE_CUS : tiles), dim3(512), 0, stream, g);
        else hipLaunchKernelGGL((gemm_wide_kernel<EPI, TC, GROUPED, SPLIT, false>), dim3(tiles), dim3(512), 0, stream, g);
        return;
    }
    if (form == FORM_128) hipLaunchKernelGGL((gemm_tile_kernel<EPI, TC, GROUPED, SPLIT, true, 128>), grid, dim3(256), 0, stream, g);
    else if (form == FORM_64) hipLaunchKernelGGL((gemm_tile_kernel<EPI, TC, GROUPED, SPLIT, true, 64>), grid, dim3(256), 0, stream, g);
    else if (form == FORM_64_DEEP && !GROUPED) hipLaunchKernelGGL((gemm_tile_kernel<EPI, TC, false, SPLIT, true, 64, TL_DEEP_STAGES>), grid, dim3(256), 0, stream, g);
    else hipLaunchKernelGGL((gemm_tile_kernel<EPI, TC, GROUPED, SPLIT, false, 64>), grid, dim3(256), 0, stream, g);
}

template <int EPI, typename TC>
static void tile_launch(const TileArgs& g, int form, dim3 grid, bool grouped, hipStream_t stream) {
    if (grouped) {
        if (g.ks > 1) tile_launch_form<EPI, TC, true, true>(g, form, grid, stream);
        else tile_launch_form<EPI, TC, true, false>(g, form, grid, stream);
    } else {
        if (g.ks > 1) tile_launch_form<EPI, TC, false, true>(g, form, grid, stream);
        else tile_launch_form<EPI, TC, false, false>(g, form, grid, stream);
    }
}

static int tile_launch_typed(const TileArgs& g, int form, dim3 grid, bool grouped, int epi, int c_dtype, hipStream_t stream) {
    if (epi == TL_SWIGLU) {
        if (c_dtype == LLMX_BF16) tile_launch<TL_SWIGLU, bf16_t>(g, form, grid, grouped, stream);
        else tile_launch<TL_SWIGLU, float>(g, form, grid, grouped, stream);
    } else if (epi == TL_ADD) {
        if (c_dtype != LLMX_F32) return -2;
        tile_launch<TL_ADD, float>(g, form, grid, grouped, stream);
    } else if (epi == TL_STORE) {
        if (c_dtype == LLMX_BF16) tile_launch<TL_STORE, bf16_t>(g, form, grid, grouped, stream);
        else tile_launch<TL_STORE, float>(g, form, grid, grouped, stream);
    } else {
        return -2;
    }
    return 0;
}

// The lean forms keep each thread's places in A and in a group's W as 32-bit byte offsets from a base the whole wave
// shares.  Whether every such offset fits: the last row of a group's weights (2 N rows under SwiGLU) and the last row of
// A that can be read.  Host arithmetic only; products that do not fit take the bounded form, which carries pointers.
extern "C" int llmx_gemm_tile_offsets_fit(int M, int N, int K, int lda, int epi, int n_groups, int a_div, int up_offset) {
    const size_t w_rows = (size_t)N + (epi == TL_SWIGLU ? (size_t)up_offset : 0);
    const size_t a_rows = n_groups > 0 ? ((size_t)M + (a_div > 0 ? a_div : 1) - 1) / (a_div > 0 ? a_div : 1) : (size_t)M;
    const size_t limit = (size_t)1 << 32;
    return w_rows * (size_t)K * sizeof(bf16_t) < limit && a_rows * (size_t)lda * sizeof(bf16_t) < limit ? 1 : 0;
}

// The runs' sums of a product whose runs were multiplied apart (TileArgs::run_tiles), added in run order as the kernel
// that holds all runs adds them, then stored as the epilogue says.  Four neighbouring features a thread.
template <bool ADD, typename TC>
__global__ void __launch_bounds__(256) gemm_runs_sum_kernel(const float* __restrict__ partial, TC* __restrict__ C, int M, int N, int ldc, int runs,
                                                          int act_kind, const float* __restrict__ act_params) {
    const int quads = (N + 3) / 4;
    const long at = (long)blockIdx.x * 256 + threadIdx.x;
    if (at >= (long)M * quads) return;
    const int m = (int)(at / quads), n = (int)(at % quads) * 4;
    const bool whole = n + 3 < N && N % 4 == 0;
    float v[4] = {0.0f, 0.0f, 0.0f, 0.0f};
    for (int r = 0; r < runs; ++r) {
        const float* src = partial + ((size_t)r * M + m) * N + n;
        float x[4] = {0.0f, 0.0f, 0.0f, 0.0f};
        if (whole) {
            const f32x4_t q = *reinterpret_cast<const f32x4_t*>(src);
            x[0] = q[0], x[1] = q[1], x[2] = q[2], x[3] = q[3];
        } else {
#pragma unroll
            for (int i = 0; i < 4; ++i)
                if (n + i < N) x[i] = src[i];
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) v[i] = r == 0 ? x[i] : v[i] + x[i];
    }
    if (llmx_act_reads_vector(act_kind)) {
#pragma unroll
        for (int i = 0; i < 4; ++i) v[i] = biased_act(act_kind, v[i], act_feature(act_kind, act_params, n + i, N));
    } else if (!ADD && act_kind != LLMX_ACT_NONE) {
        const ActFn act(act_kind, act_params);
#pragma unroll
        for (int i = 0; i < 4; ++i) v[i] = act(v[i]);
    }
    store_quad<ADD>(C + (size_t)m * ldc, n, N, ldc % 4 == 0 && ((uintptr_t)C & 15) == 0, v);
}

static int form_rows(int form) { return form == FORM_WIDE || form == FORM_128 ? 128 : 64; }
static int form_feats(int form, int epi) { return (epi == TL_SWIGLU ? 64 : 128) * (form == FORM_WIDE ? 2 : 1); }

// A and W bfloat16, K a multiple of 8.  n_groups == 0: dense over M rows.  n_groups > 0: grouped over the n_pairs = M
// rows of `list`; `max_tiles` bounds the (expert, row tile) pairs of 64-row tiles (at most min(groups, pairs) + pairs / 64).
// ks: the runs K is cut into; the caller passes what the weight-streaming kernel uses for this N and K.
// tile_stats (grouped, optional): device int, from the grouping: the sum over groups of ceil(rows / 128), or (stats_choose) its choice
// of tiles for every class of K (tile_choice.h).
//
// Which form runs (every form gives an output element the same bits):
//   dense: up to 512 tiles of 64 rows (fewer where rows are few: deep_most) the 64-row form three tiles deep (two workgroups a
//     CU at most); else the wide form (8 waves, 128 x 256, three tiles deep) where it has at least 192 tiles for the 256 CUs, of
//     long K and many rows 150 (measured on 2,048 rows: 8,192 features 113 against 165 us, 3,072 features 100 against 108 us;
//     1,600 rows of 3,072 features of 6,144 values, 156 tiles: 86 against 92, but 192 rows of 20,480, 160 tiles: 98 against 91),
//     else 64-row
//     tiles (three workgroups a CU; more, smaller tiles fill the chip better when there are few, and up to 64 rows half
//     of a 128-row tile is padding: 200,064 features of 3,072, 48 rows 265 -> 257 us, 64 rows 276 -> 268).
//     With `runs_scratch` (llmx_gemm_tile_runs_scratch floats) a product of few tiles and several runs of K gives each
//     run a workgroup of its own and adds the runs' sums in a second kernel, in the order the one kernel adds them.
//   grouped with tile_stats: both a 128-row form (wide_routed: the wide one, or 4 waves for short K) and the 64-row form are
//     launched; on the device the one that fits the groups' rows works and the other leaves at once.
// Floats of scratch with which llmx_gemm_tile multiplies the runs of a dense product apart (0: it would not).
extern "C" long llmx_gemm_tile_runs_scratch(int M, int N, int K, int epi, int ks, int n_groups) {
    if (n_groups > 0 || epi == TL_SWIGLU || ks < 2 || K % TL_BK || M <= 0 || N <= 0) return 0;
    const int steps = (K + 31) / 32, per = (steps + ks - 1) / ks;
    if (per % 2) return 0;
    const long tiles = (long)((M + 63) / 64) * ((N + TL_BN - 1) / TL_BN);
    if (tiles >= runs_apart_below(M, K)) return 0;     // enough workgroups without
    const int runs = (K / TL_BK + per / 2 - 1) / (per / 2);
    return runs < 2 ? 0 : (long)runs * M * N;
}

static int gemm_tile(const void* A, const void* W, void* C, int c_dtype, int M, int N, int K, int lda, int ldc, int epi, int ks,
                                     int n_groups, int max_tiles, const int* group_offsets, const int* list, int a_div, long w_group_stride,
                                     int up_offset, const int* tile_stats, int stats_choose, float* runs_scratch, int act, const float* act_params, int glu_kind,
                                     float glu_limit, const float* glu_row_scale, const float* glu_row_gate, int glu_row_gate_ld, int* ticket, hipStream_t stream) {
    if (M <= 0 || N <= 0 || K <= 0) return 0;
    if (K % 8) return -2;
    const bool grouped = n_groups > 0;
    if (ks != 1 && ks != 2 && ks != 4 && ks != 8) return -2;
    const int steps = (K + 31) / 32, per = (steps + ks - 1) / ks;
    const bool lean = K % TL_BK == 0 && (ks == 1 || per % 2 == 0) && llmx_gemm_tile_offsets_fit(M, N, K, lda, epi, n_groups, a_div, up_offset);
    TileArgs g{(const bf16_t*)A, (const bf16_t*)W, C, M, N, K, lda, ldc, group_offsets, list, n_groups, a_div > 0 ? a_div : 1,
               w_group_stride, up_offset, 0, ks, 64, nullptr, -1, 0, 0, 0, 0, epi != TL_SWIGLU ? act : LLMX_ACT_NONE, act_params,
               GluArgs{epi == TL_SWIGLU ? glu_kind : LLMX_GLU_SILU, glu_limit, epi == TL_SWIGLU ? glu_row_scale : nullptr,
                       epi == TL_SWIGLU ? glu_row_gate : nullptr, glu_row_gate_ld},
               0, nullptr};
    g.stream_out = lean && epi == TL_STORE && c_dtype == LLMX_F32 && nothing_applied(g, epi) && llmx_gemm_tile_streams_out(C, M, N, K, ldc, n_groups);
    if (grouped && nothing_applied(g, epi) && tile_takes_tickets(K, (N + form_feats(FORM_WIDE, epi) - 1) / form_feats(FORM_WIDE, epi), M, n_groups)) g.ticket = ticket;
    if (!llmx_act_fits(act, act_params, epi == TL_STORE, epi == TL_ADD)) return -2;
    auto launch = [&](int form, int tiles_y, bool short_k = false) -> int {      // short_k: 128-row tiles of short K, whichever kernel has them
        g.bm = form_rows(form);
        g.m_tiles = (M + g.bm - 1) / g.bm;
        const int feats = form_feats(form, epi);
        dim3 grid((N + feats - 1) / feats, grouped ? tiles_y : g.m_tiles, 1);
        if (grid.y > 65535) return -2;
        g.strip_runs = grouped ? 0 : llmx_gemm_tile_strip_runs((int)grid.x, (int)grid.y, form == FORM_WIDE);
        if (form == FORM_64_DEEP) llmx_note_launch(LK_GEMM_TILE_64_DEEP);
        if (g.stream_out) llmx_note_launch(LK_GEMM_TILE_LINES);
        llmx_note_launch(short_k ? LK_GEMM_TILE_GROUPED_128
                         : form == FORM_WIDE ? (grouped ? LK_GEMM_TILE_GROUPED_WIDE : LK_GEMM_TILE_WIDE)
                         : form == FORM_128 ? LK_GEMM_TILE_GROUPED_128
                         : form == FORM_64 || form == FORM_64_DEEP ? (grouped ? LK_GEMM_TILE_GROUPED_64 : LK_GEMM_TILE_64)
                                           : (grouped ? LK_GEMM_TILE_GROUPED_BOUNDED : LK_GEMM_TILE_BOUNDED));
        return tile_launch_typed(g, form, grid, grouped, epi, c_dtype, stream);
    };
    int rc;
    if (!lean) {
        rc = launch(FORM_BOUNDED, max_tiles);
    } else if (!grouped && runs_scratch && llmx_gemm_tile_runs_scratch(M, N, K, epi, ks, 0) > 0) {
        // few tiles (a step of some tens of rows): a workgroup a run of K, then the runs' sums added in run order
        const int tiles_per_run = per / 2, runs = (K / TL_BK + tiles_per_run - 1) / tiles_per_run;
        TileArgs part = g;
        part.C = runs_scratch;
        part.ldc = N;
        part.ks = 1;
        part.bm = 64;
        part.m_tiles = (M + 63) / 64;
        part.run_tiles = tiles_per_run;
        part.strip_runs = llmx_gemm_tile_strip_runs((N + TL_BN - 1) / TL_BN, part.m_tiles, 0);
        part.stream_out = 0;
        part.act = LLMX_ACT_NONE;       // the runs' sums are stored bare; the kernel that adds them applies the activation
        llmx_note_launch(LK_GEMM_TILE_RUNS_APART);
        hipLaunchKernelGGL((gemm_tile_kernel<TL_STORE, float, false, false, true, 64>), dim3((N + TL_BN - 1) / TL_BN, part.m_tiles, runs), dim3(256), 0,
                           stream, part);
        const long quads = (long)M * ((N + 3) / 4);
        const dim3 sum_grid((unsigned)((quads + 255) / 256));
        if (epi == TL_ADD) {
            if (c_dtype != LLMX_F32) return -2;
            hipLaunchKernelGGL((gemm_runs_sum_kernel<true, float>), sum_grid, dim3(256), 0, stream, (const float*)runs_scratch, (float*)C, M, N, ldc, runs, g.act, g.act_params);
        } else if (c_dtype == LLMX_BF16) {
            hipLaunchKernelGGL((gemm_runs_sum_kernel<false, bf16_t>), sum_grid, dim3(256), 0, stream, (const float*)runs_scratch, (bf16_t*)C, M, N, ldc, runs, g.act, g.act_params);
        } else {
            hipLaunchKernelGGL((gemm_runs_sum_kernel<false, float>), sum_grid, dim3(256), 0, stream, (const float*)runs_scratch, (float*)C, M, N, ldc, runs, g.act, g.act_params);
        }
        rc = 0;
    } else if (!grouped) {
        const long wide_tiles = (long)((M + WD_BM - 1) / WD_BM) * ((N + form_feats(FORM_WIDE, epi) - 1) / form_feats(FORM_WIDE, epi));
        const long narrow_tiles = (long)((M + 63) / 64) * ((N + form_feats(FORM_64, epi) - 1) / form_feats(FORM_64, epi));
        rc = launch(narrow_tiles <= deep_most(M) ? FORM_64_DEEP : wide_tiles >= (K >= 4096 && M >= 512 ? 150 : 192) && M > 64 ? FORM_WIDE : FORM_64, 0);
    } else if (tile_stats && n_groups <= WD_MAX_GROUPS) {     // (more groups: 64-row tiles)
        // 128-row tiles: each group adds at most one partial tile
        const int big_tiles = (n_groups < M ? n_groups : M) + M / 128;
        g.tile_stats = tile_stats;
        g.choice_bit = stats_choose ? tile_k_class(K) : -1;
        g.choice_without = ticket && !g.ticket;
        g.run_if_big = 1;
        rc = launch(wide_routed(K, g.ticket) ? FORM_WIDE : FORM_128, big_tiles < max_tiles ? big_tiles : max_tiles, K < 2048);
        if (rc == 0) {
            g.run_if_big = 0;
            rc = launch(FORM_64, max_tiles);
        }
    } else {
        rc = launch(FORM_64, max_tiles);
    }
    if (rc) return rc;
    return LLMX_CHECK_LAUNCH();
}

// ticket (grouped, optional): device int that holds 0 and does again afterwards; with it the wide form's workgroups stay and take tiles by it.
extern "C" int llmx_gemm_tile_tickets(const void* A, const void* W, void* C, int c_dtype, int M, int N, int K, int lda, int ldc, int epi, int ks,
                                      int n_groups, int max_tiles, const int* group_offsets, const int* list, int a_div, long w_group_stride,
                                      int up_offset, const int* tile_stats, int stats_choose, int* ticket, float* runs_scratch, int act, const float* act_params,
                                      int glu_kind, float glu_limit, const float* glu_row_scale, const float* glu_row_gate, int glu_row_gate_ld,
                                      hipStream_t stream) {
    return gemm_tile(A, W, C, c_dtype, M, N, K, lda, ldc, epi, ks, n_groups, max_tiles, group_offsets, list, a_div, w_group_stride, up_offset, tile_stats,
                     stats_choose, runs_scratch, act, act_params, glu_kind, glu_limit, glu_row_scale, glu_row_gate, glu_row_gate_ld, ticket, stream);
}

// ... without one, and with the bare count in tile_stats, or none.
extern "C" int llmx_gemm_tile(const void* A, const void* W, void* C, int c_dtype, int M, int N, int K, int lda, int ldc, int epi, int ks,
                              int n_groups, int max_tiles, const int* group_offsets, const int* list, int a_div, long w_group_stride,
                              int up_offset, const int* tile_stats, float* runs_scratch, int act, const float* act_params, int glu_kind,
                              float glu_limit, const float* glu_row_scale, const float* glu_row_gate, int glu_row_gate_ld, hipStream_t stream) {
    return gemm_tile(A, W, C, c_dtype, M, N, K, lda, ldc, epi, ks, n_groups, max_tiles, group_offsets, list, a_div, w_group_stride, up_offset, tile_stats,
                     0, runs_scratch, act, act_params, glu_kind, glu_limit, glu_row_scale, glu_row_gate, glu_row_gate_ld, nullptr, stream);
}
