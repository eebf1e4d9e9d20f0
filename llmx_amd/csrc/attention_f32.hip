// Float32 attention over pages on the float32 matrix instruction: what paged_attention_generic_kernel computes for plain causal
// (or windowed) attention, where the sizes allow 16-byte loads.
//
// The universal kernel gives a (row, head) one wave that reads its keys four bytes at a time: 421 us for four requests of 600 tokens,
// 448 us for a prompt of 333 (16 query heads over 4 of 128).  Here a workgroup takes up to 16 columns, the query heads of one KV head
// for one row or for neighbouring rows, and its waves share the context's segments of 32 keys out among them, a round of a segment
// a wave after the other; what bounds it is a segment's chain (keys, scores, softmax, values) a round, so a decoded row's rounds are
// kept few by eight waves: the prompt 37 us, the four requests 16 + 10 us with their contexts shared out.  Scores are K Q^T and results V^T P on 16x16x4: the scores' layout (a lane holds four neighbouring keys
// of its column) is the weights' operand layout as it stands, nothing is exchanged between lanes.
//
// A row's bits depend on its own query, its position and its request's cache only: segments are fixed runs of absolute positions,
// each with a softmax of its own (maximum, weights, their sum, the weighted values from zero), folded in key order with one formula,
// whichever wave made them; a segment none of whose keys a column sees leaves the column as it was.
#include "attention_args.h"

typedef float f32x4_t __attribute__((ext_vector_type(4)));

#define AF_SEG 32
#define AF_ONE_ROW_MAX 256   // up to this many rows a workgroup takes the columns of one row (decoded rows share no keys), beyond it neighbouring rows fill the 16 columns

// Where a split launch leaves its segments' results: [row][head][segment][v_dim], then a (maximum, sum) pair each.
struct SegmentParts {
    float* values;
    float* ml;
    int segments;       // a row's places
};

// DT: head_dim and v_dim are at most 16 DT.  NW waves; a round's partial results lie in LDS (NW x 16 columns x 16 DT floats, 64 KB).
// SPLIT: the row's rounds are dealt to gridDim.z workgroups, which leave every segment's result in memory for the merge kernel.
template <int DT, int NW, bool SPLIT>
__global__ void __launch_bounds__(64 * NW) paged_attention_f32_kernel(AttnArgs a, int rows, int rpt, SegmentParts out_parts) {
    constexpr int WIDTH = 16 * DT, THREADS = 64 * NW;
    constexpr int OWN = 16 * WIDTH / THREADS;          // neighbouring dims of one column that a thread folds
    static_assert(OWN % 4 == 0, "a thread folds whole quads");
    __shared__ __attribute__((aligned(16))) float part[SPLIT ? 1 : NW][16][WIDTH + 4];
    __shared__ __attribute__((aligned(16))) float queries[16][WIDTH + 4];
    __shared__ float part_m[NW][16], part_l[NW][16];
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    const int r = lane & 15, kg = lane >> 4;
    const int D = a.head_dim, VD = a.v_dim, dt = D >> 4, vt = VD >> 4, PT = a.page_tokens;
    const int ratio = a.n_heads / a.n_kv_heads, chunks = (ratio + 15) / 16;
    const int kvh = blockIdx.y / chunks, head0 = kvh * ratio + (blockIdx.y % chunks) * 16;
    const int hpt = min(16, (kvh + 1) * ratio - head0);                        // heads (columns of a row)
    const int t0 = ((int)gridDim.x - 1 - (int)blockIdx.x) * rpt;               // late rows, whose ranges are long, first
    const int n_rows = min(rpt, rows - t0);
    const int own_c = tid / (THREADS / 16), own_d = (tid % (THREADS / 16)) * OWN;
    // column c is head head0 + c % hpt of row t0 + c / hpt; a column past the last repeats the last row's
    const int my_at = min(r / hpt, n_rows - 1), my_row = t0 + my_at, my_pos = a.pos[my_row];
    const int own_at = min(own_c / hpt, n_rows - 1), own_row = t0 + own_at, own_pos = a.pos[own_row];
    const bool own_live = own_c < n_rows * hpt;
    const int my_lo = a.window > 0 ? max(0, my_pos - a.window + 1) : 0, own_lo = a.window > 0 ? max(0, own_pos - a.window + 1) : 0;

    {       // the columns' queries, in LDS: the registers are the keys' and values'
        const float* qp = (const float*)a.q + ((size_t)my_row * a.n_heads + head0 + r % hpt) * D + 4 * kg;
        for (int u = wave; u < dt; u += NW) *reinterpret_cast<f32x4_t*>(&queries[r][16 * u + 4 * kg]) = *reinterpret_cast<const f32x4_t*>(qp + 16 * u);
        __syncthreads();
    }
    float m = -INFINITY, l = 0.0f, own[OWN];
#pragma unroll
    for (int i = 0; i < OWN; ++i) own[i] = 0.0f;

    for (int j = 0; j < n_rows; ) {                   // the rows of one request after the other (nearly always a single pass)
        const int entry = a.row_entry[t0 + j];
        const int begin = j;
        int hi = 0, lo = 0x7fffffff;                  // the keys that some row of the pass sees lie in lo .. hi
        for (; j < n_rows && a.row_entry[t0 + j] == entry; ++j) {
            const int p = a.pos[t0 + j];
            hi = max(hi, p);
            lo = min(lo, a.window > 0 ? max(0, p - a.window + 1) : 0);
        }
        const int* table = a.tables + (size_t)entry * a.max_blocks;
        const bool mine = my_at >= begin && my_at < j;
        for (int first = lo / AF_SEG + (SPLIT ? (int)blockIdx.z * NW : 0); first <= hi / AF_SEG; first += SPLIT ? (int)gridDim.z * NW : NW) {
            const int seg = first + wave;
            if (seg <= hi / AF_SEG) {
                f32x4_t s[2], o[DT], v[2][DT];
                float top = -INFINITY;
                auto fetch_values = [&](int b) {
                    const int group = min(max(seg * AF_SEG + 16 * b + 4 * kg, lo & ~3), hi & ~3);       // four neighbouring tokens of a page
                    const float* vp = (const float*)a.v_cache + (((size_t)table[group / PT] * a.n_kv_heads + kvh) * VD + r) * PT + group % PT;
#pragma unroll
                    for (int u = 0; u < DT; ++u)
                        if (u < vt) v[b][u] = *reinterpret_cast<const f32x4_t*>(vp + (size_t)16 * u * PT);
                };
                if (DT <= 8) {       // on their way while the scores are formed; wider heads leave no registers for that
                    fetch_values(0);
                    fetch_values(1);
                }
#pragma unroll
                for (int b = 0; b < 2; ++b) {
                    // a key outside lo .. hi (its page may be gone) is read at the range's edge and masked below
                    const int base = seg * AF_SEG + 16 * b;
                    const int key = min(max(base + r, lo), hi);
                    const float* kp = (const float*)a.k_cache + (((size_t)table[key / PT] * a.n_kv_heads + kvh) * PT + key % PT) * D + 4 * kg;
                    f32x4_t k[DT];
#pragma unroll
                    for (int u = 0; u < DT; ++u)
                        if (u < dt) k[u] = *reinterpret_cast<const f32x4_t*>(kp + 16 * u);
                    f32x4_t even = {0.0f, 0.0f, 0.0f, 0.0f}, odd = even;             // two chains, so that the instruction's latency is covered
#pragma unroll
                    for (int u = 0; u < DT; ++u)
                        if (u < dt) {
                            const f32x4_t q = *reinterpret_cast<const f32x4_t*>(&queries[r][16 * u + 4 * kg]);
#pragma unroll
                            for (int i = 0; i < 4; ++i) {
                                if (i & 1) odd = __builtin_amdgcn_mfma_f32_16x16x4f32(k[u][i], q[i], odd, 0, 0, 0);
                                else even = __builtin_amdgcn_mfma_f32_16x16x4f32(k[u][i], q[i], even, 0, 0, 0);
                            }
                        }
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        const int at = base + 4 * kg + i;
                        s[b][i] = (at <= my_pos && at >= my_lo) ? (even[i] + odd[i]) * a.scale : -INFINITY;
                        top = fmaxf(top, s[b][i]);
                    }
                }
                top = rows_max4(top);
                float sum = 0.0f;
#pragma unroll
                for (int b = 0; b < 2; ++b)
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        const int at = seg * AF_SEG + 16 * b + 4 * kg + i;
                        s[b][i] = (at <= my_pos && at >= my_lo) ? expf(s[b][i] - top) : 0.0f;
                        sum += s[b][i];
                    }
                sum = rows_sum4(sum);
                // A value no column may see must not reach one as 0 x infinity: finite values go through the matrix cores, which
                // multiply every column's weight; a token outside the range counts as 0, and a value that is not finite is left
                // out there and added to the columns that see it.
#pragma unroll
                for (int u = 0; u < DT; ++u) o[u] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
                for (int b = 0; b < 2; ++b) {
                    if (DT > 8) fetch_values(b);
                    const int base = seg * AF_SEG + 16 * b;
                    bool odd_value = false;
#pragma unroll
                    for (int u = 0; u < DT; ++u)
                        if (u < vt) {
#pragma unroll
                            for (int i = 0; i < 4; ++i) {
                                if (base + 4 * kg + i < lo || base + 4 * kg + i > hi) v[b][u][i] = 0.0f;
                                odd_value |= !(fabsf(v[b][u][i]) <= 3.402823466e38f);
                            }
                        }
                    if (__any(odd_value)) {
                        for (int key = 0; key < 16; ++key) {
                            const bool sees = base + key <= my_pos && base + key >= my_lo;
                            const int i = key & 3;
                            const float w = __shfl(i == 0 ? s[b][0] : i == 1 ? s[b][1] : i == 2 ? s[b][2] : s[b][3], 4 * (key & 12) + r);      // its weight in the lane's column
#pragma unroll
                            for (int u = 0; u < DT; ++u) {
                                if (u >= vt) continue;
                                const float mine_v = i == 0 ? v[b][u][0] : i == 1 ? v[b][u][1] : i == 2 ? v[b][u][2] : v[b][u][3];
#pragma unroll
                                for (int d = 0; d < 4; ++d) {
                                    const float x = __shfl(mine_v, 4 * (key & 12) + 4 * kg + d);
                                    if (sees && !(fabsf(x) <= 3.402823466e38f)) o[u][d] += w * x;
                                }
                            }
                        }
#pragma unroll
                        for (int u = 0; u < DT; ++u)
#pragma unroll
                            for (int i = 0; i < 4; ++i)
                                if (u < vt && !(fabsf(v[b][u][i]) <= 3.402823466e38f)) v[b][u][i] = 0.0f;
                    }
#pragma unroll
                    for (int u = 0; u < DT; ++u)
                        if (u < vt) {
#pragma unroll
                            for (int i = 0; i < 4; ++i) o[u] = __builtin_amdgcn_mfma_f32_16x16x4f32(v[b][u][i], s[b][i], o[u], 0, 0, 0);
                        }
                }
                if (SPLIT) {
                    if (r < hpt) {
                        const size_t at = ((size_t)my_row * a.n_heads + head0 + r) * out_parts.segments + seg;
#pragma unroll
                        for (int u = 0; u < DT; ++u)
                            if (u < vt) *reinterpret_cast<f32x4_t*>(out_parts.values + at * VD + 16 * u + 4 * kg) = o[u];
                        if (kg == 0) {
                            out_parts.ml[2 * at] = top;
                            out_parts.ml[2 * at + 1] = sum;
                        }
                    }
                } else if (mine) {
#pragma unroll
                    for (int u = 0; u < DT; ++u)
                        if (u < vt) *reinterpret_cast<f32x4_t*>(&part[wave][r][16 * u + 4 * kg]) = o[u];
                    if (kg == 0) {
                        part_m[wave][r] = top;
                        part_l[wave][r] = sum;
                    }
                }
            }
            if (SPLIT) continue;
            __syncthreads();
            if (own_live && own_at >= begin && own_at < j && own_d < VD) {
#pragma unroll
                for (int w = 0; w < NW; ++w) {
                    const int from = (first + w) * AF_SEG;
                    if (from > own_pos || from + AF_SEG <= own_lo) continue;
                    const float ms = part_m[w][own_c], top = fmaxf(m, ms);
                    const float keep = expf(m - top), join = expf(ms - top);
                    l = fmaf(l, keep, part_l[w][own_c] * join);
#pragma unroll
                    for (int i = 0; i < OWN; i += 4) {
                        const f32x4_t p = *reinterpret_cast<const f32x4_t*>(&part[w][own_c][own_d + i]);
#pragma unroll
                        for (int d = 0; d < 4; ++d) own[i + d] = fmaf(own[i + d], keep, p[d] * join);
                    }
                    m = top;
                }
            }
            __syncthreads();
        }
    }
    if (SPLIT || !own_live || own_d >= VD) return;
    const int h = head0 + own_c % hpt;
    float* out = (float*)a.out + ((size_t)own_row * a.n_heads + h) * VD + own_d;
    const float factor = (a.gate && !a.gate_wide) ? sigmoid_f(a.gate[(size_t)own_row * a.gate_ld + h]) : 1.0f;
#pragma unroll
    for (int i = 0; i < OWN; ++i) {
        if (own_d + i >= VD) break;
        float y = own[i] / l;
        if (a.gate) y = y * (a.gate_wide ? sigmoid_f(a.gate[(size_t)own_row * a.gate_ld + (size_t)h * VD + own_d + i]) : factor);
        out[i] = y;
    }
}

// A split row's segments folded in key order: a thread holds 4 dims of one (row, head), grid (rows, heads).
__global__ void __launch_bounds__(64) attention_f32_merge_kernel(AttnArgs a, SegmentParts parts) {
    const int t = blockIdx.x, h = blockIdx.y, d = 4 * (int)threadIdx.x;
    if (d >= a.v_dim) return;
    const int p = a.pos[t], first = a.window > 0 ? max(0, p - a.window + 1) / AF_SEG : 0, last = p / AF_SEG;
    const size_t at = ((size_t)t * a.n_heads + h) * parts.segments;
    const float* ml = parts.ml + 2 * at;
    const float* values = parts.values + at * a.v_dim + d;
    float m = -INFINITY, l = 0.0f;
    f32x4_t o = {0.0f, 0.0f, 0.0f, 0.0f};
    constexpr int UN = 8;        // segments asked for together; past the last the last again, not folded
    for (int s0 = first; s0 <= last; s0 += UN) {
        f32x4_t v[UN];
        float ms[UN], ls[UN];
#pragma unroll
        for (int u = 0; u < UN; ++u) {
            const size_t s = min(s0 + u, last);
            v[u] = *reinterpret_cast<const f32x4_t*>(values + s * a.v_dim);
            ms[u] = ml[2 * s];
            ls[u] = ml[2 * s + 1];
        }
#pragma unroll
        for (int u = 0; u < UN; ++u) {
            if (s0 + u > last) break;
            const float top = fmaxf(m, ms[u]);
            const float keep = expf(m - top), join = expf(ms[u] - top);
            l = fmaf(l, keep, ls[u] * join);
#pragma unroll
            for (int i = 0; i < 4; ++i) o[i] = fmaf(o[i], keep, v[u][i] * join);
            m = top;
        }
    }
    float* out = (float*)a.out + ((size_t)t * a.n_heads + h) * a.v_dim + d;
    const float factor = (a.gate && !a.gate_wide) ? sigmoid_f(a.gate[(size_t)t * a.gate_ld + h]) : 1.0f;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        float y = o[i] / l;
        if (a.gate) y = y * (a.gate_wide ? sigmoid_f(a.gate[(size_t)t * a.gate_ld + (size_t)h * a.v_dim + d + i]) : factor);
        out[i] = y;
    }
}

bool llmx_attention_f32_takes(const AttnArgs& a) {
    return a.keep_first == 0 && a.chunk == 0 && a.maps == 1 && a.softcap == 0.0f && !a.slopes && !a.sink && a.head_dim % 16 == 0 && a.v_dim % 16 == 0 &&
           a.head_dim >= 16 && a.v_dim >= 16 && a.head_dim <= 256 && a.v_dim <= 256 && a.page_tokens % 4 == 0 &&
           (((uintptr_t)a.q | (uintptr_t)a.k_cache | (uintptr_t)a.v_cache) & 15) == 0;
}

// Floats of scratch with which a launch of `rows` rows over block tables this wide shares the rows' contexts out (0: it does not).
// A round of a workgroup of eight waves covers 256 keys and takes 8 to 13 us, so contexts of several rounds gain as long as the rows
// alone leave CUs idle (AF_SPLIT_BELOW workgroups; 4 rows of 600 tokens, 4 KV heads: 53 -> 16 + 10 us) and the segments' results
// stay small (64 MB).
#define AF_SPLIT_BELOW 512
#define AF_SPLIT_MAX_FLOATS (16L << 20)
static int af_segments(int max_blocks, int page_tokens) { return (int)(((long)max_blocks * page_tokens + AF_SEG - 1) / AF_SEG); }
extern "C" long llmx_attention_f32_scratch(int rows, int n_heads, int n_kv_heads, int v_dim, int page_tokens, int max_blocks) {
    if (rows < 1 || n_heads < 1 || n_kv_heads < 1 || n_heads % n_kv_heads || (long)max_blocks * page_tokens > (1L << 30)) return 0;
    const long groups = (long)rows * n_kv_heads * ((n_heads / n_kv_heads + 15) / 16), segments = af_segments(max_blocks, page_tokens);
    const long need = (long)rows * n_heads * segments * (v_dim + 2);
    return groups < AF_SPLIT_BELOW && segments > 8 && need <= AF_SPLIT_MAX_FLOATS ? need : 0;
}

int llmx_attention_f32(const AttnArgs& a, int rows, float* scratch, long scratch_floats, hipStream_t stream) {
    const int ratio = a.n_heads / a.n_kv_heads, hpt = ratio < 16 ? ratio : 16, groups = a.n_kv_heads * ((ratio + 15) / 16);
    const int widest = a.head_dim > a.v_dim ? a.head_dim : a.v_dim;
    llmx_note_launch(LK_ATTENTION_F32);
    const long need = scratch && ((uintptr_t)scratch & 15) == 0 ? llmx_attention_f32_scratch(rows, a.n_heads, a.n_kv_heads, a.v_dim, a.page_tokens, a.max_blocks) : 0;
    if (need > 0 && need <= scratch_floats) {
        const int segments = af_segments(a.max_blocks, a.page_tokens), nw = widest <= 128 && widest > 64 ? 8 : 4;
        const SegmentParts parts{scratch, scratch + (long)rows * a.n_heads * segments * a.v_dim, segments};
        int shares = (segments + nw - 1) / nw;
        const int wanted = (2 * AF_SPLIT_BELOW + rows * groups - 1) / (rows * groups);
        if (shares > wanted) shares = wanted;
        const dim3 grid(rows, groups, shares);
        if (widest <= 64) hipLaunchKernelGGL((paged_attention_f32_kernel<4, 4, true>), grid, dim3(256), 0, stream, a, rows, 1, parts);
        else if (widest <= 128) hipLaunchKernelGGL((paged_attention_f32_kernel<8, 8, true>), grid, dim3(512), 0, stream, a, rows, 1, parts);
        else hipLaunchKernelGGL((paged_attention_f32_kernel<16, 4, true>), grid, dim3(256), 0, stream, a, rows, 1, parts);
        llmx_note_launch(LK_ATTENTION_F32_MERGE);
        hipLaunchKernelGGL(attention_f32_merge_kernel, dim3(rows, a.n_heads), dim3(64), 0, stream, a, parts);
        return LLMX_CHECK_LAUNCH();
    }
    const int rpt = rows <= AF_ONE_ROW_MAX || ratio > 16 ? 1 : 16 / hpt;
    const dim3 grid((rows + rpt - 1) / rpt, groups);
    const SegmentParts none{nullptr, nullptr, 0};
    if (widest <= 64) hipLaunchKernelGGL((paged_attention_f32_kernel<4, 4, false>), grid, dim3(256), 0, stream, a, rows, rpt, none);
    else if (widest <= 128) hipLaunchKernelGGL((paged_attention_f32_kernel<8, 8, false>), grid, dim3(512), 0, stream, a, rows, rpt, none);
    else hipLaunchKernelGGL((paged_attention_f32_kernel<16, 4, false>), grid, dim3(256), 0, stream, a, rows, rpt, none);
    return LLMX_CHECK_LAUNCH();
}
