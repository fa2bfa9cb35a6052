// Softmax attention over the paged cache for the 32-bit path, on the float matrix instruction (v_mfma_f32_16x16x4_f32: whole
// floats in, float sums).  A block is one tile of up to 16 items (rows of one segment times the query heads that share a
// key head) and a split of its keys; its waves (eight, or two or four) take the 16-key steps in turn, each with a
// running maximum, sum and result of its own, which meet in LDS at the end.  Several splits leave partial results for the merge of
// csrc/attention_rowwise.hip.
//
// A step is S^T = K Q^T and O += P V.  With S^T a lane holds the scores of one item (column lane % 16) against the keys 4 g ..
// 4 g + 3, g = lane / 16, which is what the second product wants as its left operand: the weights go from one instruction to
// the other in the registers where they are.  Both products take their inner index as 4 g + e of a sixteen, so keys (a row of
// the page) and values (transposed in the page) are 16-byte loads; the next step's are in flight while this one is computed.
// An item does not see what it must not, whatever that holds: a wave whose result is not finite makes it again item by item.
// Bound by the two matrix products and a chain of one trip to memory a step and wave.
//
// Measured on an MI355X, 9 heads of 64 over 3: 130 rows at 128 to 350 keys beside two decoding rows 79 us with a wave a (row,
// head), lanes along the keys, each lane walking a key of its own -> 12.3; two rows at 350 keys 28 + 5 (two splits, merge) -> 13.0.
// Where many blocks have short contexts a block has two or four waves (kernels.attention.f32_waves).
#include "common.h"
#include <type_traits>

#define AF_WAVES 8                      // at most

typedef __attribute__((ext_vector_type(4))) float af_f32x4;

struct AttnF32Args {
    const float* q; int q_row_stride;
    const float* kcache; const float* vcache;
    const int* tables; const int* positions;
    const int* tasks;                 // [n][4]: segment (negative: none), first row, rows, unused
    float* out; float* part_o; float* part_ml;
    int heads, kv_heads, per_chunk, chunks;      // query heads of a tile; tiles of heads a key head
    int page_shift, width, window;
    float scale;
    int splits;
};

// What a wave wrote to LDS before is there for its own lanes after.
__device__ __forceinline__ void wave_order() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// DT sixteens of a head's coordinates, W waves
template <int DT, int W>
__global__ void __launch_bounds__(W * WAVE)
attn_f32_kernel(AttnF32Args p) {
    constexpr int D = 16 * DT;
    __shared__ float so[W][16][D + 4], sm[W][16], sl[W][16];
    const int seg = p.tasks[4 * blockIdx.x], row0 = p.tasks[4 * blockIdx.x + 1], n_rows = p.tasks[4 * blockIdx.x + 2];
    if (seg < 0 || n_rows <= 0) return;
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid / WAVE), lane = tid % WAVE, r = lane % 16, g = lane / 16;
    const int kvh = blockIdx.y / p.chunks, head0 = blockIdx.y % p.chunks * p.per_chunk, group = p.heads / p.kv_heads;
    // item i: row row0 + i / per_chunk, head kvh * group + head0 + i % per_chunk
    auto live = [&](int i) { return i / p.per_chunk < n_rows && head0 + i % p.per_chunk < group; };
    auto row_of = [&](int i) { return row0 + min(i / p.per_chunk, n_rows - 1); };
    auto head_of = [&](int i) { return kvh * group + min(head0 + i % p.per_chunk, group - 1); };
    const int pos = p.positions[row_of(r)];
    const int end = p.positions[row0 + n_rows - 1] + 1, low = p.positions[row0] + 1 - p.window;
    const int least = p.window > 0 && low > 0 ? low : 0;             // the first key that a row of the tile sees
    const int first = least / 16, steps = (end + 15) / 16 - first;
    const int share = (steps + p.splits - 1) / p.splits;
    const int begin = first + blockIdx.z * share, stop = min(begin + share, first + steps);
    const int P = 1 << p.page_shift;
    const int* table = p.tables + (size_t)seg * p.width;
    af_f32x4 fq[DT];                                                  // (a wave without a step does not wait for it)
    auto ask_q = [&]() __attribute__((always_inline)) {
        const float* qr = p.q + (size_t)row_of(r) * p.q_row_stride + (size_t)head_of(r) * D + 4 * g;
#pragma unroll
        for (int c = 0; c < DT; ++c) fq[c] = *(const af_f32x4*)(qr + 16 * c);
    };
    af_f32x4 o[DT];
#pragma unroll
    for (int c = 0; c < DT; ++c) o[c] = (af_f32x4){0.f, 0.f, 0.f, 0.f};
    float m = -INFINITY, l = 0.f;                                     // of item r (l: this lane's keys only)
    // a step's pages, keys and values: keys before the tile's first (whose pages may have gone back) and past its last are
    // that one again, their weights are zero
    auto key_of = [&](int t) { return min(max(t, least), end - 1); };
    auto ask_pages = [&](int s, int& pk, int& pv) {
        pk = table[key_of(s * 16 + r) >> p.page_shift];
        pv = table[key_of(s * 16 + 4 * g) >> p.page_shift];
    };
    auto ask = [&](int s, int pk, int pv, af_f32x4 (&fk)[DT], af_f32x4 (&fv)[DT]) __attribute__((always_inline)) {
        const int tk = key_of(s * 16 + r), tv = key_of(s * 16 + 4 * g) & ~3;      // (pages of whole fours)
        const float* kr = p.kcache + (((size_t)pk * p.kv_heads + kvh) * P + (tk & (P - 1))) * D + 4 * g;
        const float* vr = p.vcache + (((size_t)pv * p.kv_heads + kvh) * D + r) * P + (tv & (P - 1));
#pragma unroll
        for (int c = 0; c < DT; ++c) fk[c] = *(const af_f32x4*)(kr + 16 * c);
#pragma unroll
        for (int c = 0; c < DT; ++c) fv[c] = *(const af_f32x4*)(vr + (size_t)16 * c * P);
    };
    // careful: the second product item by item over the keys that it sees
    auto use = [&](int s, af_f32x4 (&fk)[DT], af_f32x4 (&fv)[DT], auto careful) __attribute__((always_inline)) {
        // (from 96 coordinates on a sum for every second sixteen of them: one chain of instructions is up to 1.08 times as far from 64
        // bits as the row-wise kernel there, two 0.46 to 0.72 times; up to 64 one chain is 0.72 to 0.98 times as far)
        constexpr int SUMS = DT >= 6 ? 2 : 1;
        af_f32x4 sums[SUMS];
#pragma unroll
        for (int i = 0; i < SUMS; ++i) sums[i] = (af_f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int c = 0; c < DT; c += SUMS)
#pragma unroll
            for (int e = 0; e < 4; ++e)
#pragma unroll
                for (int i = 0; i < SUMS; ++i) sums[i] = __builtin_amdgcn_mfma_f32_16x16x4f32(fk[c + i][e], fq[c + i][e], sums[i], 0, 0, 0);
        af_f32x4 sc = sums[0];
        if constexpr (SUMS == 2) sc += sums[1];
        // sc[e]: item r, key s * 16 + 4 g + e
        float best = -INFINITY;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int t = s * 16 + 4 * g + e;
            const bool sees = t <= pos && (p.window <= 0 || t > pos - p.window);
            sc[e] = sees ? sc[e] * p.scale : -INFINITY;
            best = fmaxf(best, sc[e]);
        }
        best = fmaxf(best, __shfl_xor(best, 16, WAVE));
        best = fmaxf(best, __shfl_xor(best, 32, WAVE));
        const float m_new = fmaxf(m, best);
        const float keep = m_new == -INFINITY ? 1.0f : expf(m - m_new);       // (nothing seen yet: nothing to keep)
        float sum = 0.f;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            sc[e] = sc[e] == -INFINITY ? 0.f : expf(sc[e] - m_new);
            sum += sc[e];
        }
        l = l * keep + sum;
        m = m_new;
        if (__any(keep != 1.0f)) {                                    // o[c][e]: item 4 g + e, coordinate 16 c + r
            float k[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) k[e] = __shfl(keep, 4 * g + e, WAVE);
#pragma unroll
            for (int c = 0; c < DT; ++c)
#pragma unroll
                for (int e = 0; e < 4; ++e) o[c][e] *= k[e];
        }
        if (s * 16 + 16 > end) {                                      // (uniform: values of keys that no row of the tile sees)
#pragma unroll
            for (int c = 0; c < DT; ++c)
#pragma unroll
                for (int e = 0; e < 4; ++e) fv[c][e] = s * 16 + 4 * g + e < end ? fv[c][e] : 0.f;
        }
        if constexpr (!decltype(careful)::value) {
#pragma unroll
            for (int e = 0; e < 4; ++e)
#pragma unroll
                for (int c = 0; c < DT; ++c) o[c] = __builtin_amdgcn_mfma_f32_16x16x4f32(sc[e], fv[c][e], o[c], 0, 0, 0);
        } else {
            // (through LDS, where the wave's result goes at the end: weights by item, -1 for none; values by key, a sixteen at a time)
            float* weights = &so[wave][0][0];
            float* values = weights + 256;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int t = s * 16 + 4 * g + e;
                weights[r * 16 + 4 * g + e] = t <= pos && (p.window <= 0 || t > pos - p.window) ? sc[e] : -1.f;
            }
#pragma unroll
            for (int c = 0; c < DT; ++c) {
#pragma unroll
                for (int e = 0; e < 4; ++e) values[(4 * g + e) * 16 + r] = fv[c][e];
                wave_order();
#pragma unroll 1
                for (int t = 0; t < 16; ++t)
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        const float weight = weights[(4 * g + e) * 16 + t];
                        if (!(weight < 0.f)) o[c][e] += weight * values[t * 16 + r];
                    }
                wave_order();
            }
        }
    };
    af_f32x4 ka[DT], va[DT], kb[DT], vb[DT];
    int s = begin + wave, pk = 0, pv = 0;
    if (s < stop) {
        ask_pages(s, pk, pv);
        ask_q();
        ask(s, pk, pv, ka, va);
        ask_pages(min(s + W, stop - 1), pk, pv);
    }
    for (; s < stop; s += 2 * W) {
        const bool more = s + W < stop;                        // (uniform over the wave)
        if (more) {
            ask(s + W, pk, pv, kb, vb);
            ask_pages(min(s + 2 * W, stop - 1), pk, pv);
        }
        use(s, ka, va, std::false_type{});
        if (!more) break;
        if (s + 2 * W < stop) {
            ask(s + 2 * W, pk, pv, ka, va);
            ask_pages(min(s + 3 * W, stop - 1), pk, pv);
        }
        use(s + W, kb, vb, std::false_type{});
    }
    // A value that is not finite, times the zero weight of an item that does not see its key, is no number: then once more, with care
    af_f32x4 finite = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int c = 0; c < DT; ++c) finite += o[c] * 0.f;
    if (__builtin_expect(__any((finite.x + finite.y) + (finite.z + finite.w) != 0.f), 0)) {
#pragma unroll
        for (int c = 0; c < DT; ++c) o[c] = (af_f32x4){0.f, 0.f, 0.f, 0.f};
        m = -INFINITY;
        l = 0.f;
        ask_q();
#pragma unroll 1
        for (int t = begin + wave; t < stop; t += W) {
            ask_pages(t, pk, pv);
            ask(t, pk, pv, ka, va);
            use(t, ka, va, std::true_type{});
        }
    }
    l += __shfl_xor(l, 16, WAVE);
    l += __shfl_xor(l, 32, WAVE);
    if (g == 0) { sm[wave][r] = m; sl[wave][r] = l; }
#pragma unroll
    for (int c = 0; c < DT; ++c)
#pragma unroll
        for (int e = 0; e < 4; ++e) so[wave][4 * g + e][16 * c + r] = o[c][e];
    __syncthreads();
    for (int idx = tid; idx < 16 * D; idx += W * WAVE) {
        const int i = idx / D, d = idx % D;
        if (!live(i)) continue;
        float best = -INFINITY, den = 0.f, num = 0.f;
#pragma unroll
        for (int w = 0; w < W; ++w) best = fmaxf(best, sm[w][i]);
#pragma unroll
        for (int w = 0; w < W; ++w) {                          // in the order of the waves
            const float f = sm[w][i] == -INFINITY ? 0.f : expf(sm[w][i] - best);
            den += f * sl[w][i];
            num += f * so[w][i][d];
        }
        const size_t at = (size_t)row_of(i) * p.heads + head_of(i);
        if (p.splits == 1) {                                          // (an item sees its own key: a sum of zero is of scores that are all -inf)
            p.out[at * D + d] = num / den;
        } else {                                                      // (a split may hold no key that the item sees)
            const size_t part = at * p.splits + blockIdx.z;
            p.part_o[part * D + d] = den > 0.f ? num / den : 0.f;
            if (d == 0) { p.part_ml[part * 2] = best; p.part_ml[part * 2 + 1] = den; }
        }
    }
}

// Whether cisr_attn_f32 takes heads of `dim` coordinates in pages of `page_size` keys.
extern "C" int cisr_attn_f32_ok(int dim, int page_size) {
    return (dim == 32 || dim == 64 || dim == 96 || dim == 128) && page_size >= 4 && (page_size & (page_size - 1)) == 0;
}

// q rows, keys and values 16-byte aligned; with several splits part_o [rows, heads, splits, dim] and part_ml [rows, heads,
// splits, 2] receive what attn_merge_kernel (natural logarithms) takes: rows that no task names are left alone.
extern "C" int cisr_attn_f32(const float* q, int q_row_stride, const float* kcache, const float* vcache, const int* tables,
                             const int* positions, const int* tasks, int n_tasks, float* out, float* part_o, float* part_ml, int heads,
                             int kv_heads, int dim, int page_size, int width, int window, float scale, int splits, int waves,
                             hipStream_t stream) {
    if (n_tasks <= 0) return 0;
    if (!cisr_attn_f32_ok(dim, page_size) || kv_heads <= 0 || heads % kv_heads || splits < 1 || splits > 65535 || q_row_stride % 4 || (waves != 2 && waves != 4 && waves != AF_WAVES) ||
        ((uintptr_t)q) % 16 || ((uintptr_t)kcache) % 16 || ((uintptr_t)vcache) % 16 || (splits > 1 && (!part_o || !part_ml)))
        return (int)hipErrorInvalidValue;
    const int group = heads / kv_heads, per_chunk = group < 16 ? group : 16, chunks = (group + per_chunk - 1) / per_chunk;
    if ((long long)kv_heads * chunks > 65535) return (int)hipErrorInvalidValue;
    int shift = 0;
    while ((1 << shift) < page_size) ++shift;
    const AttnF32Args p{q, q_row_stride, kcache, vcache, tables, positions, tasks, out, part_o, part_ml, heads, kv_heads, per_chunk, chunks,
                        shift, width, window, scale, splits};
    const dim3 grid(n_tasks, kv_heads * chunks, splits);
#define AF_OF(DT) do { \
        if (waves == 2) attn_f32_kernel<DT, 2><<<grid, 2 * WAVE, 0, stream>>>(p); \
        else if (waves == 4) attn_f32_kernel<DT, 4><<<grid, 4 * WAVE, 0, stream>>>(p); \
        else attn_f32_kernel<DT, AF_WAVES><<<grid, AF_WAVES * WAVE, 0, stream>>>(p); \
    } while (0)
    if (dim == 32) AF_OF(2);
    else if (dim == 64) AF_OF(4);
    else if (dim == 96) AF_OF(6);
    else AF_OF(8);
#undef AF_OF
    return CISR_LAUNCH_CHECK();
}
