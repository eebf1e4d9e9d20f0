// The true 32-bit path's products on the matrix cores: C[M,N] (+)= A[M,K] * W[N,K]^T, all float32, dense or grouped, with the
// universal product's epilogues (v_mfma_f32_16x16x4_f32 multiplies and adds full float32 values; it has no reduced-precision mode).
//
// Two forms give an element the same bits.  K is cut into `ks` runs of whole steps of 16 (a function of N and K alone), a run is
// one accumulator walked over its steps in order, W as the instruction's A operand, and the runs' sums are added in order; so a
// row's bits depend on its own values and the weights only, not on the rows beside it or on the form.
//
//  * stream: few rows.  The weights' way from memory bounds it: a workgroup's `ks` waves share a strip of 16 features, one run of
//    K each, and ask for a round of steps while the round before is multiplied, as whole lines that are read once (weight_lines.h).
//    4 rows, 8 experts of 2 x 2,688 features of 2,048 values: 44.8 us, 60 with half lines that the caches keep; their 2,048 features of
//    2,688 values 27.5 (41.8), dense 3,072 of 2,048 9.4 (10.9); the universal product takes 0.2-0.5 ms for the smallest of these.
//  * tiles: many rows.  The instruction's rate bounds it (140 TFLOP/s measured alone): 64 rows x 128 (64) features a workgroup,
//    operands staged through LDS 32 values of k at a time, its runs folded in registers.  2,048 rows: 8,192 features
//    of 3,072 values 0.80 ms (130 TFLOP/s); 333 rows of 2,048 values: 32,768 features 0.44 ms (102 TFLOP/s), where the universal
//    product reaches 8 TFLOP/s.  Chunks asked for two ahead instead of one: 0.84 -> 0.78 ms and 0.47 -> 0.44 ms.
#include "gemm_args.h"
#include "weight_lines.h"
#include <type_traits>

typedef float f32x4_t __attribute__((ext_vector_type(4)));

// What an output element gets; `up` counts for the gated epilogue only.
template <int EPI>
__device__ __forceinline__ void f32_store_quad(const GemmArgs& g, const ActFn& act, int row, int n, f32x4_t v, f32x4_t up) {
    const GluRow glu(g.glu, EPI == EPI_SWIGLU ? row : 0);
    float* c = (float*)g.C + (size_t)row * g.ldc + n;
    const bool whole = n + 3 < g.N && g.ldc % 4 == 0 && ((uintptr_t)g.C & 15) == 0;
    f32x4_t old = {0.0f, 0.0f, 0.0f, 0.0f};
    if (EPI == EPI_ADD && whole) old = *reinterpret_cast<const f32x4_t*>(c);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        if (EPI == EPI_SWIGLU) {
            v[i] = glu(v[i], up[i]);
            continue;
        }
        v[i] = llmx_act_reads_vector(act.kind) ? biased_act(act.kind, v[i], act_feature(act.kind, g.act_params, n + i, g.N)) : act(v[i]);
        if (EPI == EPI_ADD) v[i] = (whole ? old[i] : n + i < g.N ? c[i] : 0.0f) + v[i];
    }
    if (whole) {
        *reinterpret_cast<f32x4_t*>(c) = v;
        return;
    }
#pragma unroll
    for (int i = 0; i < 4; ++i)
        if (n + i < g.N) c[i] = v[i];
}

// Grid: dense (strips, chunks of 16 MT rows); grouped (strips, groups, row chunks of a group).
template <int KS, int MT, int EPI>
__global__ void __launch_bounds__(64 * KS, MT == 1 ? 4 : 1) gemm_f32_stream_kernel(GemmArgs g) {
    constexpr int NS = EPI == EPI_SWIGLU ? 2 : 1;                  // weight strips: the features', and the up rows' of the same features
    constexpr int UN = NS * MT == 1 ? 4 : 2;    // steps of a round: its loads travel together (a wave has two rounds on their way, a SIMD four waves)
    __shared__ __attribute__((aligned(16))) float red[KS > 1 ? KS : 1][NS * MT][256];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;     // known to be one for the wave: else every load of weights is a loop over its lanes
    const int r = lane & 15, kg = lane >> 4;
    const int n0 = blockIdx.x * 16, K = g.K;
    const float* A = (const float*)g.A;
    const float* W = (const float*)g.W;
    int row_end = g.M, m0 = blockIdx.y * 16 * MT, m_step = gridDim.y * 16 * MT;
    if (g.group_offsets) {
        m0 = g.group_offsets[blockIdx.y] + blockIdx.z * 16 * MT;
        row_end = g.group_offsets[blockIdx.y + 1];
        m_step = gridDim.z * 16 * MT;
        W += (size_t)blockIdx.y * g.w_group_stride;
    }
    const int steps = (K + 15) >> 4, per = (steps + KS - 1) / KS, ranges = (steps + per - 1) / per;
    const int s_begin = min(steps, wave * per), s_end = min(steps, s_begin + per);
    const int whole_end = min(s_end, K >> 4);                      // steps before this one are whole
    // the strips' rows in memory, the lane's chunk of a line of two steps
    const uint32_t pitch = 4u * (uint32_t)g.ldw, w_at = (uint32_t)(r & 7) * pitch + line_chunk(r, kg);
    strip_t strip[NS];
#pragma unroll
    for (int ns = 0; ns < NS; ++ns)
        strip[ns] = strip_of(W + (size_t)(n0 + (ns ? g.up_offset : 0)) * g.ldw, (uint32_t)(min(16, g.N - n0) - 1) * pitch + 4u * (uint32_t)K);
    const bool lines = g.ldw % 32 == 0 && per % 2 == 0;       // a pair of steps is a line of each row
    const int n_steps = max(whole_end - s_begin, 0), rounds = (n_steps + UN - 1) / UN;
    const ActFn act(EPI != EPI_SWIGLU ? g.act : LLMX_ACT_NONE, g.act_params);

    auto all_rows = [&](auto as_lines) {
    for (; m0 < row_end; m0 += m_step) {
        // a row past the last reads the last one: what its column of the product gives is never stored
        const float* ap[MT];
        int row_c[MT];
#pragma unroll
        for (int t = 0; t < MT; ++t) {
            const int m = min(m0 + 16 * t + r, row_end - 1);
            row_c[t] = g.group_offsets ? g.list[m] : m;
            ap[t] = A + (size_t)(g.group_offsets ? row_c[t] / g.a_div : m) * g.lda + kg * 4;
        }
        f32x4_t acc[NS][MT];
#pragma unroll
        for (int ns = 0; ns < NS; ++ns)
#pragma unroll
            for (int t = 0; t < MT; ++t) acc[ns][t] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
        struct Round {
            WeightLines w[UN / 2][NS];
            f32x4_t a[UN][MT];
        };
        // of a last round that is not full the steps past the end are steps fetched before, and not multiplied
        auto fetch = [&](Round& f, int round) {
            const int s = s_begin + UN * round;
#pragma unroll
            for (int u = 0; u < UN; u += 2) {
                const int pair = min(s + u, whole_end - 1), back = s + u + 1 < whole_end ? 0 : 64 * (r >> 3);
#pragma unroll
                for (int ns = 0; ns < NS; ++ns) f.w[u / 2][ns] = two_lines<decltype(as_lines)::value>(strip[ns], w_at - back, 8 * pitch, 64u * (uint32_t)pair);
            }
#pragma unroll
            for (int u = 0; u < UN; ++u)
#pragma unroll
                for (int t = 0; t < MT; ++t) f.a[u][t] = *reinterpret_cast<const f32x4_t*>(ap[t] + (size_t)min(s + u, whole_end - 1) * 16);
        };
        auto multiply = [&](const f32x4_t (&w)[NS], const f32x4_t (&a)[MT]) {
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int ns = 0; ns < NS; ++ns)
#pragma unroll
                    for (int t = 0; t < MT; ++t) acc[ns][t] = __builtin_amdgcn_mfma_f32_16x16x4f32(w[ns][i], a[t][i], acc[ns][t], 0, 0, 0);
        };
        auto whole = [&](const Round& f, int n) {      // the round's first n steps
#pragma unroll
            for (int u = 0; u < UN; u += 2) {
                if (u >= n) break;
                f32x4_t first[NS], second[NS];
#pragma unroll
                for (int ns = 0; ns < NS; ++ns) two_steps(f.w[u / 2][ns], first[ns], second[ns]);
                multiply(first, f.a[u]);
                if (u + 1 < n) multiply(second, f.a[u + 1]);
            }
        };
        if (rounds > 0) {
            // rounds take turns in two sets of registers: the next is asked for before the present one is multiplied
            Round first, second;
            fetch(first, 0);
            int i = 0;
            for (; i + 2 < rounds; i += 2) {
                fetch(second, i + 1);
                __builtin_amdgcn_sched_barrier(0);
                whole(first, UN);
                __builtin_amdgcn_sched_barrier(0);
                fetch(first, i + 2);
                __builtin_amdgcn_sched_barrier(0);
                whole(second, UN);
                __builtin_amdgcn_sched_barrier(0);
            }
            if (i + 1 < rounds) {
                fetch(second, i + 1);
                __builtin_amdgcn_sched_barrier(0);
                whole(first, UN);
                __builtin_amdgcn_sched_barrier(0);
                whole(second, n_steps - UN * (i + 1));
            } else {
                whole(first, n_steps - UN * i);
            }
        }
        if (s_end > whole_end) {       // K's last step holds 4, 8 or 12 values
            const bool in = whole_end * 16 + 4 * kg < K;
            f32x4_t w[NS], a[MT];
#pragma unroll
            for (int ns = 0; ns < NS; ++ns) {
                const float* row = W + (size_t)(min(n0 + r, g.N - 1) + (ns ? g.up_offset : 0)) * g.ldw + kg * 4;
                w[ns] = in ? *reinterpret_cast<const f32x4_t*>(row + (size_t)whole_end * 16) : f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
            }
#pragma unroll
            for (int t = 0; t < MT; ++t) a[t] = in ? *reinterpret_cast<const f32x4_t*>(ap[t] + (size_t)whole_end * 16) : f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
            multiply(w, a);
        }
        if (KS > 1) {
#pragma unroll
            for (int ns = 0; ns < NS; ++ns)
#pragma unroll
                for (int t = 0; t < MT; ++t) *reinterpret_cast<f32x4_t*>(&red[wave][ns * MT + t][lane * 4]) = acc[ns][t];
            __syncthreads();
        }
#pragma unroll
        for (int t = 0; t < MT; ++t) {
            if (t % KS != wave) continue;
            f32x4_t v[NS];
#pragma unroll
            for (int ns = 0; ns < NS; ++ns) {
                v[ns] = acc[ns][t];
                if (KS > 1) {
                    v[ns] = *reinterpret_cast<f32x4_t*>(&red[0][ns * MT + t][lane * 4]);
                    for (int w = 1; w < ranges; ++w) {
                        const f32x4_t o = *reinterpret_cast<f32x4_t*>(&red[w][ns * MT + t][lane * 4]);
#pragma unroll
                        for (int i = 0; i < 4; ++i) v[ns][i] += o[i];
                    }
                }
            }
            if (m0 + 16 * t + r < row_end) f32_store_quad<EPI>(g, act, row_c[t], n0 + 4 * kg, v[0], v[NS - 1]);
        }
        if (KS > 1) __syncthreads();
    }
    };
    if constexpr (MT == 1) {
        if (lines) {
            all_rows(std::true_type{});
            return;
        }
    }
    all_rows(std::false_type{});
}

// K a multiple of 16.  A workgroup takes 64 rows and BN weight rows (gated: BN / 2 features' gate and up rows); grid (feature tiles,
// row tiles), grouped: the row tiles of the groups that have rows, in order.  A staged row takes 32 values of k and 4 of padding, so
// that 8 rows' 16-byte pieces fall into different banks; the next chunk travels while this one is multiplied.
#define FT_ROWS 64
#define FT_PITCH 36
#define FT_AHEAD 2      // (4: the same)
template <int EPI, int BN>
__global__ void __launch_bounds__(512) gemm_f32_tiles_kernel(GemmArgs g, int ks, int n_groups) {
    // eight waves of 32 weight rows by TT tiles of 16 rows: also a tile that has its CU to itself gives a SIMD two waves, so that one's
    // operand reads hide behind the other's multiplications (64 weight rows, 2,048 values, four waves of 32 x 32: 55 us a tile)
    constexpr int TT = BN / 64, THREADS = 512, WAVES = 8;
    constexpr int W_PIECES = BN * 8 / THREADS, ROWS_A_PASS = THREADS / 8;       // 16-byte pieces of a chunk a thread brings: these of W's, one of A's
    __shared__ __attribute__((aligned(16))) float Ws[2][BN * FT_PITCH];
    __shared__ __attribute__((aligned(16))) float As[2][FT_ROWS * FT_PITCH];
    __shared__ int rows_a[FT_ROWS], rows_c[FT_ROWS], tile_info[3], scan_waves[WAVES];
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    const int r = lane & 15, kg = lane >> 4;
    const int wn = wave % (BN / 32), wm = wave / (BN / 32);
    constexpr int FEATS = EPI == EPI_SWIGLU ? BN / 2 : BN;
    const int n0 = blockIdx.x * FEATS, K = g.K;
    const float* W = (const float*)g.W;
    int row_begin = blockIdx.y * FT_ROWS, row_end = g.M;
    if (g.group_offsets) {
        // which group's which tile: the groups' tile counts scanned by all threads together
        if (tid == 0) tile_info[0] = -1;
        int base = 0;
        for (int e0 = 0; e0 < n_groups; e0 += THREADS) {
            const int e = e0 + tid;
            const int begin = e < n_groups ? g.group_offsets[e] : 0, end = e < n_groups ? g.group_offsets[e + 1] : 0;
            const int tiles = (end - begin + FT_ROWS - 1) / FT_ROWS;
            int incl = tiles;
#pragma unroll
            for (int d = 1; d < 64; d <<= 1) {
                const int o = __shfl_up(incl, d, 64);
                if (lane >= d) incl += o;
            }
            if (lane == 63) scan_waves[wave] = incl;
            __syncthreads();
            int before = base;
            for (int w = 0; w < WAVES; ++w) {
                if (w < wave) before += scan_waves[w];
                base += scan_waves[w];
            }
            const int first = before + incl - tiles;
            if ((int)blockIdx.y >= first && (int)blockIdx.y < first + tiles) {
                tile_info[0] = e;
                tile_info[1] = begin + ((int)blockIdx.y - first) * FT_ROWS;
                tile_info[2] = end;
            }
            __syncthreads();
            if ((int)blockIdx.y < base) break;
        }
        if (tile_info[0] < 0) return;
        row_begin = tile_info[1];
        row_end = tile_info[2];
        W += (size_t)tile_info[0] * g.w_group_stride;
    }
    if (tid < FT_ROWS) {
        const int m = min(row_begin + tid, row_end - 1);
        const int p = g.group_offsets ? g.list[m] : m;
        rows_a[tid] = g.group_offsets ? p / g.a_div : m;      // a row past the last reads the last one and is not stored
        rows_c[tid] = row_begin + tid < row_end ? p : -1;
    }
    __syncthreads();
    const int piece = tid & 7, prow = tid >> 3;
    const float* w_src[W_PIECES];
#pragma unroll
    for (int j = 0; j < W_PIECES; ++j) {
        const int w = prow + ROWS_A_PASS * j;
        // gated: rows 32 q .. + 15 of the tile are features 16 q .. + 15's gate rows, the next 16 their up rows
        const int f = EPI == EPI_SWIGLU ? n0 + 16 * (w >> 5) + (w & 15) : n0 + w;
        w_src[j] = W + (size_t)(min(f, g.N - 1) + (EPI == EPI_SWIGLU && (w & 16) ? g.up_offset : 0)) * g.ldw + 4 * piece;
    }
    const float* a_src = (const float*)g.A + (size_t)rows_a[prow] * g.lda + 4 * piece;
    struct Fetched {
        f32x4_t w[W_PIECES], a;
    };
    auto fetch = [&](int c, Fetched& f) {
        const int kk = min(32 * c, K - 16 - 16 * (piece >> 2));      // K's last chunk may hold one step: the second is fetched from inside K and not multiplied
#pragma unroll
        for (int j = 0; j < W_PIECES; ++j) f.w[j] = *reinterpret_cast<const f32x4_t*>(w_src[j] + kk);
        f.a = *reinterpret_cast<const f32x4_t*>(a_src + kk);
    };
    auto stage = [&](const Fetched& f, int buf) {
#pragma unroll
        for (int j = 0; j < W_PIECES; ++j) *reinterpret_cast<f32x4_t*>(&Ws[buf][(prow + ROWS_A_PASS * j) * FT_PITCH + 4 * piece]) = f.w[j];
        *reinterpret_cast<f32x4_t*>(&As[buf][prow * FT_PITCH + 4 * piece]) = f.a;
    };
    const int steps = K >> 4, per = (steps + ks - 1) / ks, chunks = (steps + 1) / 2;
    f32x4_t total[2][TT], acc[2][TT];
#pragma unroll
    for (int ns = 0; ns < 2; ++ns)
#pragma unroll
        for (int t = 0; t < TT; ++t) acc[ns][t] = total[ns][t] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
    bool first_run = true;
    int in_run = 0;
    auto multiply = [&](auto live, int c, int buf) {
        constexpr int LIVE = decltype(live)::value;      // 16-row tiles of the wave that hold rows
        f32x4_t wf[2][2], af[2][TT];
        if constexpr (LIVE > 0) {
#pragma unroll
            for (int u = 0; u < 2; ++u) {
#pragma unroll
                for (int ns = 0; ns < 2; ++ns) wf[u][ns] = *reinterpret_cast<const f32x4_t*>(&Ws[buf][(32 * wn + 16 * ns + r) * FT_PITCH + 16 * u + 4 * kg]);
#pragma unroll
                for (int t = 0; t < LIVE; ++t) af[u][t] = *reinterpret_cast<const f32x4_t*>(&As[buf][(16 * (TT * wm + t) + r) * FT_PITCH + 16 * u + 4 * kg]);
            }
        }
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            const int s = 2 * c + u;
            if (s >= steps) break;
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int ns = 0; ns < 2; ++ns)
#pragma unroll
                    for (int t = 0; t < LIVE; ++t) acc[ns][t] = __builtin_amdgcn_mfma_f32_16x16x4f32(wf[u][ns][i], af[u][t][i], acc[ns][t], 0, 0, 0);
            if (++in_run == per || s + 1 == steps) {
#pragma unroll
                for (int ns = 0; ns < 2; ++ns)
#pragma unroll
                    for (int t = 0; t < LIVE; ++t) {
#pragma unroll
                        for (int i = 0; i < 4; ++i) total[ns][t][i] = first_run ? acc[ns][t][i] : total[ns][t][i] + acc[ns][t][i];
                        acc[ns][t] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
                    }
                first_run = false;
                in_run = 0;
            }
        }
    };
    const ActFn act(EPI != EPI_SWIGLU ? g.act : LLMX_ACT_NONE, g.act_params);
    // FT_AHEAD chunks are on their way, a register set each, while another is multiplied: a chunk's multiplications are far shorter than
    // the way to memory; past the end the last one again
    Fetched f[FT_AHEAD];
#pragma unroll
    for (int d = 0; d < FT_AHEAD; ++d) fetch(min(d, chunks - 1), f[d]);
    stage(f[0], 0);
    fetch(min(FT_AHEAD, chunks - 1), f[0]);
    __syncthreads();
    auto walk = [&](auto live) {
        for (int c = 0; c < chunks; c += FT_AHEAD)
#pragma unroll
            for (int d = 0; d < FT_AHEAD; ++d) {
                if (c + d >= chunks) break;
                multiply(live, c + d, d & 1);
                stage(f[(d + 1) % FT_AHEAD], (d & 1) ^ 1);
                fetch(min(c + d + 1 + FT_AHEAD, chunks - 1), f[(d + 1) % FT_AHEAD]);
                __syncthreads();
            }
    };
    // a wave whose rows are past the last ones (a group's last tile) leaves the matrix cores to the others; every wave meets every barrier
    const int held = min(row_end - row_begin, FT_ROWS) - 16 * TT * wm;
    if (TT > 1 && held > 16) walk(std::integral_constant<int, TT>());
    else if (held > 0) walk(std::integral_constant<int, 1>());
    else walk(std::integral_constant<int, 0>());
#pragma unroll
    for (int t = 0; t < TT; ++t) {
        const int row = rows_c[16 * (TT * wm + t) + r];
        if (row < 0) continue;
        if (EPI == EPI_SWIGLU) {
            const int n = n0 + 16 * wn + 4 * kg;
            if (n < g.N) f32_store_quad<EPI>(g, act, row, n, total[0][t], total[1][t]);
        } else {
#pragma unroll
            for (int ns = 0; ns < 2; ++ns) {
                const int n = n0 + 32 * wn + 16 * ns + 4 * kg;
                if (n < g.N) f32_store_quad<EPI>(g, act, row, n, total[ns][t], total[ns][t]);
            }
        }
    }
}

// Runs K is cut into: enough strips x runs to keep the chip's waves streaming, at least 12 steps of 16 a run.  N and K only.
static int f32_runs(int N, int K) {
    const int strips = (N + 15) / 16, steps = K >> 4;
    int ks = 1;
    while (ks < 8 && strips * ks < 2048 && steps / (ks * 2) >= 12) ks *= 2;
    return ks;
}

bool llmx_gemm_f32_cores_take(const GemmArgs& g, int n_groups) {
    return g.K % 4 == 0 && g.lda % 4 == 0 && g.ldw % 4 == 0 && ((uintptr_t)g.A & 15) == 0 && ((uintptr_t)g.W & 15) == 0 &&
           (n_groups == 0 || g.w_group_stride % 4 == 0);
}

template <int EPI>
static int launch_stream(const GemmArgs& g, int n_groups, int ks, int rows_a_group, hipStream_t stream) {
    const int mt = rows_a_group <= 16 ? 1 : rows_a_group <= 32 || EPI == EPI_SWIGLU ? 2 : 4;
    int chunks = (rows_a_group + 16 * mt - 1) / (16 * mt);
    const dim3 grid = n_groups ? dim3((g.N + 15) / 16, n_groups, chunks > 64 ? 64 : chunks) : dim3((g.N + 15) / 16, chunks > 4096 ? 4096 : chunks);
#define F32_STREAM(KS, MT) hipLaunchKernelGGL((gemm_f32_stream_kernel<KS, MT, EPI>), grid, dim3(64 * KS), 0, stream, g)
#define F32_STREAM_MT(KS)               \
    do {                                \
        if (mt == 1) F32_STREAM(KS, 1); \
        else if (mt == 2) F32_STREAM(KS, 2); \
        else if constexpr (EPI != EPI_SWIGLU) F32_STREAM(KS, 4); \
    } while (0)
    switch (ks) {
        case 1: F32_STREAM_MT(1); break;
        case 2: F32_STREAM_MT(2); break;
        case 4: F32_STREAM_MT(4); break;
        default: F32_STREAM_MT(8); break;
    }
#undef F32_STREAM_MT
#undef F32_STREAM
    return LLMX_CHECK_LAUNCH();
}

template <int EPI>
static int launch_tiles(const GemmArgs& g, int n_groups, int ks, int row_tiles, hipStream_t stream) {
    // 128 weight rows a workgroup read the activations half as often, 64 fill the chip with fewer rows.  Measured at K 2,048, 256
    // CUs: with n workgroups a CU the narrow form takes about 10 + 33 n us (1: 43, 2: 76, 3: 106), the wide one 12 + 61 n (1: 73,
    // 2: 136); rows count in sixteens, as the last tile's absent ones take no time (a group's last sixteen is half full on average).
    const int wide = EPI == EPI_SWIGLU ? 64 : 128, narrow = wide / 2;
    const long sixteens = n_groups ? (g.M + 8 * (n_groups < g.M ? n_groups : g.M) + 15) / 16 : (g.M + 15) / 16;
    const long n_wide = ((g.N + wide - 1) / wide * sixteens + 4 * 256 - 1) / (4 * 256), n_narrow = ((g.N + narrow - 1) / narrow * sixteens + 4 * 256 - 1) / (4 * 256);
    if (12 + 61 * n_wide <= 10 + 33 * n_narrow)
        hipLaunchKernelGGL((gemm_f32_tiles_kernel<EPI, 128>), dim3((g.N + wide - 1) / wide, row_tiles), dim3(512), 0, stream, g, ks, n_groups);
    else
        hipLaunchKernelGGL((gemm_f32_tiles_kernel<EPI, 64>), dim3((g.N + narrow - 1) / narrow, row_tiles), dim3(512), 0, stream, g, ks, n_groups);
    return LLMX_CHECK_LAUNCH();
}

// Which form: the stream form multiplies at about 45 TFLOP/s beyond 16 rows (every strip reads the rows again), the tiles at 100 to
// 130 but, at K 2,048, never in less than 43 us: they meet at rows x features of about 380,000 (3,072 features: 96 rows 40 against
// 43 us, 128 rows 47 against 44; 2,048: 128 rows 26 against 43, 192 rows 46 against 43; 8,192 of K 3,072: 48 rows 62 against 63).
// Groups of at most half a tile of rows on average stay with the stream form, the tiles being mostly padding.  The lines do not know K: both
// forms' times grow with it alike (2,048 features, 128 and 192 rows, across the line: K 2,048 23 and 42 us, 6,144 58 and 116, 8,192 75 and 153).
// K a multiple of 4 but not of 16 stays with the stream form at any number of rows, and there hardly gains on the universal product
// (2,048 rows, us, universal and this: 2,048 features of 2,052 values 360 and 325, 4,096 of 516 176 and 158; 128 rows 196 and 23, 52 and 14).
template <int EPI>
static int launch_f32(const GemmArgs& g, int n_groups, hipStream_t stream) {
    const int ks = f32_runs(g.N, g.K);
    const int rows = n_groups ? (g.M + n_groups - 1) / n_groups : g.M;      // grouped: a group's on average (the counts are on the device; both forms take any)
    const int row_tiles = n_groups ? (n_groups < g.M ? n_groups : g.M) + g.M / FT_ROWS : (g.M + FT_ROWS - 1) / FT_ROWS;
    const bool few = rows <= (n_groups ? FT_ROWS / 2 : 16) || (long)g.M * g.N <= 380000;
    if (!few && g.K % 16 == 0 && row_tiles <= 65535) {
        llmx_note_launch(LK_GEMM_GENERIC_TILES);
        return launch_tiles<EPI>(g, n_groups, ks, row_tiles, stream);
    }
    llmx_note_launch(LK_GEMM_GENERIC_STREAM);
    return launch_stream<EPI>(g, n_groups, ks, rows, stream);
}

int llmx_gemm_f32_cores(const GemmArgs& g, int epi, int n_groups, hipStream_t stream) {
    switch (epi) {
        case EPI_STORE: return launch_f32<EPI_STORE>(g, n_groups, stream);
        case EPI_ADD: return launch_f32<EPI_ADD>(g, n_groups, stream);
        case EPI_SWIGLU: return launch_f32<EPI_SWIGLU>(g, n_groups, stream);
        default: return -1;
    }
}
