// Row-wise kernels of layers that norm after the sum, of an embedding with a hashed table of token pairs, and of
// attention that norms queries and keys over the whole projection:
//   x[r] = table[token_r] * scale + pairs[hash(previous token, token_r)]          (the last row of `pairs` at position 0)
//   x <- rmsnorm(alpha x + y * sigmoid(g + b)) * w     (y a row, or the weighted sum of `top` rows; the gate optional)
//   q, k normed over all heads at once, neighbouring coordinates turned by the position, q into a buffer of padded
//   heads, k and v into the pages of the cache
// Statistics and the residual stream are float; `T` is the storage type of activations (float or bf16).
#include "common.h"

// ------------------------------------------------------------------ embedding with a table of hashed token pairs
// One block a row.  The token before a segment's first row is the request's last token of the step before, kept in
// `last_token[state slot]`.  SINGLE: every segment has one row, and the thread that reads the kept token then stores
// the row's own; otherwise store_last_token_kernel runs afterwards.
// Bound by the chain to the pair's row (segment, slot, kept token, hash): a thread has a word of V elements (four, or one where the rows are
// not aligned for that), and the table's is on its way meanwhile.  24 rows of 2,048 bf16 in a captured step 9.4 -> 6.2 us (256 threads
// a row that went round after the chain).
template <typename TE, typename TH, bool SINGLE, int V>
__global__ void __launch_bounds__(1024)
embedding_pairs_kernel(const int* __restrict__ tokens, const int* __restrict__ positions, const int* __restrict__ seg_of_row,
                       const int* __restrict__ seg_start, const int* __restrict__ state_slots, int* last_token,
                       const TE* __restrict__ table, const TE* __restrict__ pairs, float* __restrict__ out, TH* __restrict__ cast,
                       int dim, int vocab, float scale, int buckets, unsigned long long mul_prev, unsigned long long mul_cur) {
    __shared__ int pair_row;
    const int row = blockIdx.x;
    int tok = tokens[row];
    tok = tok < 0 ? 0 : tok >= vocab ? vocab - 1 : tok;
    const TE* e = table + (size_t)tok * dim;
    const int first = threadIdx.x * V, step = blockDim.x * V;
    float v[V];
    load_run<V>(e + min(first, dim - V), v);
    if (pairs != nullptr) {
        if (threadIdx.x == 0) {
            const int seg = seg_of_row[row];
            int at = buckets;                                   // a sequence's first token (and rows of no segment)
            if (seg >= 0) {
                const int slot = state_slots[seg];
                if (positions[row] > 0) {
                    const int prev = row > seg_start[seg] ? tokens[row - 1] : last_token[slot];
                    at = (int)(((unsigned long long)(prev < 0 ? 0 : prev) * mul_prev + (unsigned long long)tok * mul_cur) % (unsigned long long)buckets);
                }
                if (SINGLE) last_token[slot] = tok;
            }
            pair_row = at;
        }
        __syncthreads();
    }
    const TE* p = pairs ? pairs + (size_t)pair_row * dim : nullptr;
    for (int d = first; d < dim; d += step) {
        if (d != first) load_run<V>(e + d, v);
#pragma unroll
        for (int i = 0; i < V; ++i) v[i] *= scale;
        if (p) {
            float q[V];
            load_run<V>(p + d, q);
#pragma unroll
            for (int i = 0; i < V; ++i) v[i] += q[i];
        }
        store_run<V>(out + (size_t)row * dim + d, v);
        if (cast) store_run<V>(cast + (size_t)row * dim + d, v);
    }
}

__global__ void store_last_token_kernel(const int* __restrict__ tokens, const int* __restrict__ seg_start,
                                        const int* __restrict__ state_slots, int* __restrict__ last_token, int segments, int vocab) {
    const int seg = blockIdx.x * blockDim.x + threadIdx.x;
    if (seg >= segments) return;
    const int first = seg_start[seg], end = seg_start[seg + 1];
    if (end <= first) return;                                  // (padding of a captured step)
    int tok = tokens[end - 1];
    last_token[state_slots[seg]] = tok < 0 ? 0 : tok >= vocab ? vocab - 1 : tok;
}

extern "C" int cisr_embedding_pairs(const int* tokens, const int* positions, const int* seg_of_row, const int* seg_start,
                                    const int* state_slots, int* last_token, const void* table, const void* pairs, float* out,
                                    void* cast, int rows, int segments, int dim, int vocab, float scale, int buckets,
                                    long long mul_prev, long long mul_cur, int single_rows, int table_dtype, int cast_dtype,
                                    hipStream_t stream) {
    if (rows <= 0) return 0;
    if (dim <= 0 || vocab <= 0 || (pairs && (buckets <= 0 || mul_prev < 0 || mul_cur < 0 || !last_token))) return (int)hipErrorInvalidValue;
    const size_t run = table_dtype == DT_F32 ? 16 : 8, cast_run = cast_dtype == DT_F32 ? 16 : 8;
    const bool wide = dim % 4 == 0 && (uintptr_t)table % run == 0 && (uintptr_t)pairs % run == 0 && (uintptr_t)out % 16 == 0 && (uintptr_t)cast % cast_run == 0;
    // Rows that are not aligned for words: a thread an element as long as all blocks of 1,024 threads are resident, beyond that 256 threads that go
    // round (8,192 rows of 1,023 bf16 28.2 us with a thread an element, 17.9 so; 300 rows 3.2, going round 3.5).  Of words likewise: 2,048 rows of 8,192 floats
    // in portions 42.2 / 41.4, 64 rows 5.8, 11.5 going round.
    const int words = wide ? dim / 4 : dim, most = rows <= 512 ? 1024 : wide ? 512 : 256, threads = words >= most ? most : (words + 63) / 64 * 64;
#define EMB_V(TE, TH, S, V) embedding_pairs_kernel<TE, TH, S, V><<<rows, threads, 0, stream>>>(tokens, positions, seg_of_row, seg_start, state_slots, \
        last_token, (const TE*)table, (const TE*)pairs, out, (TH*)cast, dim, vocab, scale, buckets, (unsigned long long)mul_prev, (unsigned long long)mul_cur)
#define EMB(TE, TH, S) do { if (wide) EMB_V(TE, TH, S, 4); else EMB_V(TE, TH, S, 1); } while (0)
    if (table_dtype == DT_F32) { if (single_rows) EMB(float, float, true); else EMB(float, float, false); }
    else if (cast_dtype == DT_F32) { if (single_rows) EMB(bf16_t, float, true); else EMB(bf16_t, float, false); }
    else { if (single_rows) EMB(bf16_t, bf16_t, true); else EMB(bf16_t, bf16_t, false); }
#undef EMB_V
#undef EMB
    int err = CISR_LAUNCH_CHECK();
    if (err || !pairs || single_rows || segments <= 0) return err;
    store_last_token_kernel<<<(segments + 63) / 64, 64, 0, stream>>>(tokens, seg_start, state_slots, last_token, segments, vocab);
    return CISR_LAUNCH_CHECK();
}

// ------------------------------------------------------------------ the norm after the sum, with a gated sublayer
// One block a row: x <- rmsnorm(alpha x + y' gate) w, y' = y[row] or sum_k yw[row, k] y[row * top + k], gate =
// sigmoid(g[row] + gb) or 1.  The sum waits in x between the two passes (a thread reads back what it wrote itself).
// `cast`: a copy of the new row in the activations' type, what the sublayers read next.
template <typename TH>
__global__ void __launch_bounds__(256)
gate_post_norm_kernel(float* __restrict__ x, const float* __restrict__ y, int top, const float* __restrict__ yw,
                      const float* __restrict__ g, int ldg, const float* __restrict__ gb, const float* __restrict__ w,
                      TH* __restrict__ cast, int dim, float eps, float alpha) {
    __shared__ float red[4];
    const size_t row = blockIdx.x;
    float* xr = x + row * dim;
    float ss = 0.f;
    for (int d = threadIdx.x; d < dim; d += 256) {
        float v;
        if (yw) {
            v = 0.f;
            for (int k = 0; k < top; ++k) v += yw[row * top + k] * y[(row * top + k) * dim + d];
        } else {
            v = y[row * dim + d];
        }
        if (g) v *= 1.0f / (1.0f + expf(-(g[row * ldg + d] + (gb ? gb[d] : 0.f))));
        v += alpha * xr[d];
        xr[d] = v;
        ss += v * v;
    }
    const float rs = 1.0f / sqrtf(block_sum<256>(ss, red) / (float)dim + eps);
    for (int d = threadIdx.x; d < dim; d += 256) {
        const float v = xr[d] * rs * w[d];
        xr[d] = v;
        if (cast) store_f32(cast + row * dim + d, v);
    }
}

// The same with the row in registers (rows of up to 256 E floats, up to two choices a sum): everything a thread needs of the
// row is asked for before any of it is used, and the sum does not go through memory.  32 rows of 2,048, two choices: 13.8 us
// as above (eight trips to memory one after the other) -> 4.8.  The same bits: the same sums in the same order.
template <int E, typename TH>
__global__ void __launch_bounds__(256)
gate_post_norm_short_kernel(float* __restrict__ x, const float* __restrict__ y, int top, const float* __restrict__ yw,
                            const float* __restrict__ g, int ldg, const float* __restrict__ gb, const float* __restrict__ w,
                            TH* __restrict__ cast, int dim, float eps, float alpha) {
    __shared__ float red[4];
    const size_t row = blockIdx.x;
    const int second = top - 1;                       // (top 1: the one row again, left out of the sum)
    float vx[E], y0[E], y1[E], vg[E], vb[E], vw[E];
#pragma unroll
    for (int e = 0; e < E; ++e) {
        const int d = min((int)threadIdx.x + 256 * e, dim - 1);
        y0[e] = y[(yw ? row * top : row) * dim + d];
        y1[e] = yw ? y[(row * top + second) * dim + d] : 0.f;
        vg[e] = g ? g[row * ldg + d] : 0.f;
        vb[e] = gb ? gb[d] : 0.f;
        vx[e] = x[row * dim + d];
        vw[e] = w[d];
    }
    float ss = 0.f;
#pragma unroll
    for (int e = 0; e < E; ++e) {
        if (threadIdx.x + 256 * e >= dim) continue;
        float v;
        if (yw) {
            v = 0.f;
            v += yw[row * top] * y0[e];
            if (top > 1) v += yw[row * top + 1] * y1[e];
        } else {
            v = y0[e];
        }
        if (g) v *= 1.0f / (1.0f + expf(-(vg[e] + vb[e])));
        v += alpha * vx[e];
        vx[e] = v;
        ss += v * v;
    }
    const float rs = 1.0f / sqrtf(block_sum<256>(ss, red) / (float)dim + eps);
#pragma unroll
    for (int e = 0; e < E; ++e) {
        const int d = threadIdx.x + 256 * e;
        if (d >= dim) continue;
        const float v = vx[e] * rs * vw[e];
        x[row * dim + d] = v;
        if (cast) store_f32(cast + row * dim + d, v);
    }
}

template <typename TH>
static void launch_gate_post_norm(float* x, const float* y, int top, const float* yw, const float* g, int ldg, const float* gb,
                                  const float* w, TH* cast, int rows, int dim, float eps, float alpha, hipStream_t stream) {
#define GPN_SHORT(E) gate_post_norm_short_kernel<E, TH><<<rows, 256, 0, stream>>>(x, y, top, yw, g, ldg, gb, w, cast, dim, eps, alpha)
    if (top <= 2 && dim <= 1024) GPN_SHORT(4);
    else if (top <= 2 && dim <= 2048) GPN_SHORT(8);
    else if (top <= 2 && dim <= 4096) GPN_SHORT(16);
    else gate_post_norm_kernel<TH><<<rows, 256, 0, stream>>>(x, y, top, yw, g, ldg, gb, w, cast, dim, eps, alpha);
#undef GPN_SHORT
}

extern "C" int cisr_gate_post_norm(float* x, const float* y, int top, const float* yw, const float* g, int ldg, const float* gb,
                                   const float* w, void* cast, int rows, int dim, float eps, float alpha, int cast_dtype,
                                   hipStream_t stream) {
    if (rows <= 0) return 0;
    if (dim <= 0 || top < 1) return (int)hipErrorInvalidValue;
    if (cast_dtype == DT_F32) launch_gate_post_norm(x, y, top, yw, g, ldg, gb, w, (float*)cast, rows, dim, eps, alpha, stream);
    else launch_gate_post_norm(x, y, top, yw, g, ldg, gb, w, (bf16_t*)cast, rows, dim, eps, alpha, stream);
    return CISR_LAUNCH_CHECK();
}

// ------------------------------------------------------------------ queries and keys normed over the whole projection
// One block a row of a projection with float results [q: heads x dim | k: kv_heads x dim | v: kv_heads x vdim | ...]
// (`bias`: float over these columns, added first, or null): q and k are RMS-normed over all their heads at once (a
// weight an element), the first 2 `half` coordinates of every head turn by the position's angles (cos / sin float
// [max_pos, half]) in neighbouring pairs (2i, 2i + 1), or with `split_half` in pairs (i, i + half); q goes to q_out
// [T, heads * pad], k and v into the pages at `slots` as heads of `pad` coordinates, the rest zero (keys [pages,
// kv_heads, page_size, pad], values transposed in a page).  `value_norm`: each head's value is divided by its root mean
// square over vdim first (no weight).  has_kv 0: the row has queries only.
#define WN_MAX_KV_HEADS 256
template <typename T>
__global__ void __launch_bounds__(256)
whole_norm_rope_scatter_kernel(const float* __restrict__ proj, int ld, const float* __restrict__ bias, const float* __restrict__ qw,
                               const float* __restrict__ kw, const int* __restrict__ positions, const int* __restrict__ slots,
                               const float* __restrict__ cosines, const float* __restrict__ sines, int half, int max_pos,
                               T* __restrict__ q_out, T* __restrict__ kcache, T* __restrict__ vcache, int heads, int kv_heads, int dim,
                               int vdim, int pad, int page_size, float eps, int has_kv, int split_half, int value_norm) {
    __shared__ float red[4];
    __shared__ float rv[WN_MAX_KV_HEADS];
    const size_t row = blockIdx.x;
    const float* pr = proj + row * ld;
    const int nq = heads * dim, nk = kv_heads * dim;
    auto val = [&](int i) { return bias ? pr[i] + bias[i] : pr[i]; };
    float sq = 0.f, sk = 0.f;
    for (int i = threadIdx.x; i < nq; i += 256) { const float v = val(i); sq += v * v; }
    const float rq = 1.0f / sqrtf(block_sum<256>(sq, red) / (float)nq + eps);
    float rk = 0.f;
    if (has_kv) {
        for (int i = threadIdx.x; i < nk; i += 256) { const float v = val(nq + i); sk += v * v; }
        rk = 1.0f / sqrtf(block_sum<256>(sk, red) / (float)nk + eps);
        if (value_norm) {
            const int wave = threadIdx.x / WAVE, lane = threadIdx.x % WAVE;
            for (int h = wave; h < kv_heads; h += 4) {
                float sv = 0.f;
                for (int c = lane; c < vdim; c += WAVE) { const float v = val(nq + nk + h * vdim + c); sv += v * v; }
                sv = wave_sum(sv);
                if (lane == 0) rv[h] = 1.0f / sqrtf(sv / (float)vdim + eps);
            }
            __syncthreads();
        }
    }
    int p = positions[row];
    p = p < 0 ? 0 : p >= max_pos ? max_pos - 1 : p;
    const float* cr = cosines + (size_t)p * half;
    const float* sr = sines + (size_t)p * half;
    // coordinate c of a head of the normed vector that starts at column `first` (weights wt), turned if it lies among
    // the turning ones
    auto turned = [&](int first, const float* wt, int base, int c, float r) {
        const float own = val(first + base + c) * r * wt[base + c];
        if (c >= 2 * half) return own;
        const int mate = split_half ? (c < half ? c + half : c - half) : c ^ 1;
        const bool second = split_half ? c >= half : (c & 1);
        const int pair = split_half ? (c < half ? c : c - half) : c >> 1;
        const float other = val(first + base + mate) * r * wt[base + mate];
        const float co = cr[pair], si = sr[pair];
        return second ? own * co + other * si : own * co - other * si;
    };
    // (blockIdx.y: with few rows several blocks share a row's outputs; each makes the row's statistics for itself)
    const int first = threadIdx.x + 256 * blockIdx.y, stride = 256 * gridDim.y;
    for (int i = first; i < heads * pad; i += stride) {
        const int h = i / pad, c = i % pad;
        store_f32(q_out + row * (size_t)(heads * pad) + i, c < dim ? turned(0, qw, h * dim, c, rq) : 0.f);
    }
    if (!has_kv) return;
    const int slot = slots[row];
    if (slot < 0) return;
    const size_t page = slot / page_size, off = slot % page_size;
    for (int i = first; i < kv_heads * pad; i += stride) {
        const int h = i / pad, c = i % pad;
        const float kv = c < dim ? turned(nq, kw, h * dim, c, rk) : 0.f;
        const float vv = c < vdim ? val(nq + nk + h * vdim + c) * (value_norm ? rv[h] : 1.0f) : 0.f;
        store_f32(kcache + ((page * kv_heads + h) * page_size + off) * pad + c, kv);
        store_f32(vcache + ((page * kv_heads + h) * pad + c) * page_size + off, vv);
    }
}

extern "C" int cisr_whole_norm_rope_scatter(const float* proj, int ld, const float* bias, const float* qw, const float* kw,
                                            const int* positions, const int* slots, const float* cosines, const float* sines, int half,
                                            int max_pos, void* q_out, void* kcache, void* vcache, int rows, int heads, int kv_heads,
                                            int dim, int vdim, int pad, int page_size, float eps, int has_kv, int split_half,
                                            int value_norm, int dtype, hipStream_t stream) {
    if (rows <= 0) return 0;
    if (dim <= 0 || dim > pad || vdim > pad || 2 * half > dim || half < 0 || heads <= 0 || (has_kv && (kv_heads <= 0 || page_size <= 0)) ||
        (value_norm && kv_heads > WN_MAX_KV_HEADS))
        return (int)hipErrorInvalidValue;
    const dim3 grid(rows, rows <= 128 ? 4 : 1);
    if (dtype == DT_F32)
        whole_norm_rope_scatter_kernel<float><<<grid, 256, 0, stream>>>(proj, ld, bias, qw, kw, positions, slots, cosines, sines, half, max_pos,
            (float*)q_out, (float*)kcache, (float*)vcache, heads, kv_heads, dim, vdim, pad, page_size, eps, has_kv, split_half, value_norm);
    else
        whole_norm_rope_scatter_kernel<bf16_t><<<grid, 256, 0, stream>>>(proj, ld, bias, qw, kw, positions, slots, cosines, sines, half, max_pos,
            (bf16_t*)q_out, (bf16_t*)kcache, (bf16_t*)vcache, heads, kv_heads, dim, vdim, pad, page_size, eps, has_kv, split_half, value_norm);
    return CISR_LAUNCH_CHECK();
}
