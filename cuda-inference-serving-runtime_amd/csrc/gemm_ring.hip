// Which tile and how many slices a ring product (gemm_ring.inc) takes, and its entry points.
#include "gemm_ring.h"
#include <algorithm>
#include <cmath>

namespace {

// What a round of blocks takes (one a compute unit, 256 of them), us on an MI355X: `start` and `step` for every 64 of the inner size
// with all units busy, `half` with half of them (less contention and a higher clock).  Measured with bf16 results, 16 x 16 and
// 8 x 16 tiles, inner sizes of 576, 2,048 and 8,192; `start` has the launch, the first copies and the stores.  (Taken
// again with the kernels as they are, `step` is 13 % lower at 64 x 128, 7 % at 128 x 64 and 256 x 128, 5 to 12 % at 256 columns and within 6 % else; `half` is
// 11 % lower at 64 x 128 and 14 to 34 % at 256 columns, within 7 % else.  The choice stands on the figures below, with which the cases were timed.)
struct Tile { int rows, cols; float start, step, half; };
constexpr Tile TILES[] = {
    {64, 32, 3.3f, 0.190f, 0.170f},    {64, 64, 3.4f, 0.230f, 0.180f},    {64, 128, 4.2f, 0.350f, 0.275f},   {128, 64, 3.9f, 0.344f, 0.264f},
    {96, 128, 4.9f, 0.415f, 0.325f},   {128, 128, 5.6f, 0.496f, 0.377f},  {160, 128, 6.1f, 0.589f, 0.437f},  {192, 128, 6.7f, 0.671f, 0.507f},
    {224, 128, 7.6f, 0.776f, 0.588f},  {256, 128, 8.1f, 0.894f, 0.671f},  {64, 256, 5.2f, 0.590f, 0.590f},   {96, 256, 6.2f, 0.739f, 0.700f},
    {128, 256, 7.9f, 0.859f, 0.780f},  {160, 256, 8.6f, 1.029f, 0.855f},  {192, 256, 9.1f, 1.228f, 1.228f},  {224, 256, 10.2f, 1.389f, 1.308f},
    {256, 256, 11.4f, 1.505f, 1.347f}, {288, 256, 12.3f, 1.665f, 1.395f},
};
constexpr int UNITS = 256, MOST_SLICES = 8, LEAST_STEPS = 4, NORMED_COLS = 1024;

struct Plan { int tile, slices; float us; };

// With one tile of rows every block streams its rows of W from memory alone: a step then is no shorter than the way there (measured
// 0.29, 0.48 and 0.77 us with 64, 128 and 256 columns); and the rows of W that a round reads come at 5.6 TB/s at best.
float round_us(const Tile& t, int blocks, int tiles_m, int steps) {
    float step = t.half + (t.step - t.half) * std::max(0.f, 2.f * blocks / UNITS - 1.f);
    if (tiles_m == 1) step = std::max(step, 0.13f + 0.0025f * t.cols);
    return t.start + steps * std::max(step, (float)blocks / tiles_m * t.cols * 128 / 5.6e6f);
}

float rounds_us(const Tile& t, long long blocks, int tiles_m, int steps) {
    const long long full = blocks / UNITS;
    const int rest = (int)(blocks % UNITS);
    return (full ? full * round_us(t, UNITS, tiles_m, steps) : 0.f) + (rest ? round_us(t, rest, std::min(tiles_m, rest), steps) : 0.f);
}

// The least of the model's times.  `slices` 0: any number of them, whose float sums are written and read once more (at 5 TB/s) by a
// kernel that mostly runs anyway (the norm that follows).
Plan plan_of(int M, int N, int K, bool gated, int slices) {
    Plan best{0, 1, INFINITY};
    const int steps = K / 64, cols = gated ? 2 * N : N;
    for (const Tile& t : TILES) {
        const int tiles_m = (M + t.rows - 1) / t.rows;
        const long long tiles = (long long)tiles_m * ((cols + t.cols - 1) / t.cols);
        for (int s = slices ? slices : 1; s <= (slices ? slices : MOST_SLICES); ++s) {
            if (s > 1 && steps / s < LEAST_STEPS) break;
            float us = rounds_us(t, tiles * s, tiles_m, (steps + s - 1) / s);
            if (s > 1) us += (float)s * M * N * 8 / 5e6f + 0.5f;
            if (us < best.us) best = {t.rows * 1000 + t.cols, s, us};
        }
    }
    return best;
}

bool fits(const RingArgs& a, int out_bytes) {
    const long long reach = ((long long)std::max(a.dual_off, 0) + 512) * a.ldw * 2;
    return a.M > 0 && a.N > 0 && a.N % 4 == 0 && a.K > 0 && a.K % 64 == 0 && a.lda >= a.K && a.ldw >= a.K && a.lda % 8 == 0 && a.ldw % 8 == 0 &&
           (uintptr_t)a.A % 16 == 0 && (uintptr_t)a.W % 16 == 0 && a.ldc >= a.N && a.ldc % 4 == 0 && (uintptr_t)a.C % (4 * out_bytes) == 0 &&
           (!a.R || (a.ldr % 4 == 0 && (uintptr_t)a.R % 16 == 0)) && (long long)a.lda * 2 * 512 < 0x7fffffffll && reach < 0x7fffffffll;
}

// The rows A are what cisr_gemm_ring_normed leaves (sums null: they are normed).
void finish_norm(RingArgs& a, const float* sums, int parts, float eps) {
    a.sums = const_cast<float*>(sums); a.parts = parts; a.inv_k = 1.f / a.K; a.eps = eps;
}

int launch(const RingArgs& a, int tile, int mode, hipStream_t stream) {
    const int rows = tile / 1000, cols = tile % 1000;
    if (a.sums && mode == RING_GATED) mode = RING_GATED_NORMED;
    if (a.sums && mode == RING_ROPE) mode = RING_ROPE_NORMED;
    if (a.sums && mode == RING_FLOAT) mode = RING_FLOAT_NORMED;
    if (a.sums && (mode == RING_FLOAT_NORMED ? a.parts != (a.N + cols - 1) / cols : a.parts <= 0)) return (int)hipErrorInvalidValue;
    if (cols == 256 && rows >= 224) return cisr_ring_launch_a(a, tile, mode, stream);
    if (cols == 256 && rows >= 96) return cisr_ring_launch_b(a, tile, mode, stream);
    if (cols == 256 || (cols == 128 && rows >= 192)) return cisr_ring_launch_c(a, tile, mode, stream);
    return cisr_ring_launch_d(a, tile, mode, stream);
}

}  // namespace

// How many slices a product whose inner size may be cut is best cut into.  0: not a shape of these kernels.
extern "C" int cisr_gemm_ring_slices(int M, int N, int K) {
    if (M <= 0 || N <= 0 || K <= 0 || K % 64 || N % 4) return 0;
    return plan_of(M, N, K, false, 0).slices;
}

// Sums a row that cisr_gemm_ring_normed leaves, or 0 where the product is better followed by the norm as a kernel of its own: where it is
// best cut along its inner size, as the kernel that adds the slices makes the norm on the way, and in rows of more than NORMED_COLS.  The norm
// of 1,000 to 2,000 rows is 5 us at any width below 2,048; without it the product before takes 1.3 us more at a width of 576 and
// 2.7 at 2,048 (it stores the rows a second time), the one behind 1.1 and 4.5 (at 2,048 columns 288 x 256 tiles have 16 sums a row).
extern "C" int cisr_gemm_ring_normed_parts(int M, int N, int K) {
    if (M <= 0 || N <= 0 || N > NORMED_COLS || K <= 0 || K % 64 || N % 4) return 0;
    const Plan plan = plan_of(M, N, K, false, 0);
    return plan.slices > 1 ? 0 : (N + plan.tile % 1000 - 1) / (plan.tile % 1000);
}

// C += A . W^T (float), and what a product that finishes the RMSNorm of C's rows reads: `scaled` = bf16(C norm_w) and the sums of squares.
extern "C" int cisr_gemm_ring_normed(const void* A, int lda, const void* W, int ldw, float* C, int ldc, const float* norm_w, void* scaled, int ldy,
                                     float* sums, int parts, int M, int N, int K, hipStream_t stream) {
    if (M <= 0 || N <= 0) return 0;
    RingArgs a{(const bf16_t*)A, lda, (const bf16_t*)W, ldw, C, ldc, C, ldc, M, N, K, 0, GateLaw{}, 0, 1};
    if (!fits(a, 4) || !norm_w || (uintptr_t)norm_w % 16 || !scaled || (uintptr_t)scaled % 8 || ldy < N || ldy % 4 || !sums)
        return (int)hipErrorInvalidValue;
    a.scaled = (bf16_t*)scaled; a.ldy = ldy; a.norm_w = norm_w; a.sums = sums; a.parts = parts;
    return launch(a, plan_of(M, N, K, false, 1).tile, RING_FLOAT, stream);
}

// C = A . W^T, bf16 or float; R (float C only) is added, and may be C; `act` (bf16 C only): an ungated activation.  `tile` 0: the model's.
extern "C" int cisr_gemm_ring_bf16(const void* A, int lda, const void* W, int ldw, void* C, int ldc, const float* R, int ldr, int M, int N,
                                   int K, int out_dtype, int act, int tile, hipStream_t stream) {
    if (M <= 0 || N <= 0) return 0;
    const bool wide = out_dtype == DT_F32;
    const RingArgs a{(const bf16_t*)A, lda, (const bf16_t*)W, ldw, C, ldc, R, ldr, M, N, K, 0, GateLaw{}, act, 1};
    if (!fits(a, wide ? 4 : 2) || (R && !wide) || (act && wide) || act < ACT_NONE || act > ACT_RELU2) return (int)hipErrorInvalidValue;
    return launch(a, tile ? tile : plan_of(M, N, K, false, 1).tile, wide ? RING_FLOAT : RING_STORE, stream);
}

// C = act(A . Wg^T, A . Wu^T), W = [Wg; Wu] with `dual_off` rows between the blocks; the law as GateLaw.  `sums` (else null): A's rows are
// those of cisr_gemm_ring_normed, `parts` sums each, here and below.
extern "C" int cisr_gemm_ring_bf16_gated(const void* A, int lda, const void* W, int ldw, void* C, int ldc, int M, int N, int K, int dual_off,
                                         float limit, float slope, float shift, const float* sums, int parts, float eps, int tile, hipStream_t stream) {
    if (M <= 0 || N <= 0) return 0;
    RingArgs a{(const bf16_t*)A, lda, (const bf16_t*)W, ldw, C, ldc, nullptr, 0, M, N, K, dual_off, GateLaw{limit, slope, shift}, 0, 1};
    if (!fits(a, 2) || dual_off < N) return (int)hipErrorInvalidValue;
    finish_norm(a, sums, parts, eps);
    return launch(a, tile ? tile : plan_of(M, N, K, true, 1).tile, RING_GATED, stream);
}

// The product's partial sums, parts[slices][M][N] (float): to be added in slice order by the kernel that reads them next.
extern "C" int cisr_gemm_ring_partials_bf16(const void* A, int lda, const void* W, int ldw, float* parts, int M, int N, int K, int slices,
                                            int tile, hipStream_t stream) {
    if (M <= 0 || N <= 0) return 0;
    const RingArgs a{(const bf16_t*)A, lda, (const bf16_t*)W, ldw, parts, N, nullptr, 0, M, N, K, 0, GateLaw{}, 0, slices};
    if (!fits(a, 4) || slices < 1 || slices > K / 64) return (int)hipErrorInvalidValue;
    return launch(a, tile ? tile : plan_of(M, N, K, false, slices).tile, RING_FLOAT, stream);
}

// The projection W = [Wq; Wk; Wv] of bf16 rows with the rotary embedding (pairs (i, i + dim / 2) of whole heads) and the cache write:
// q into q_out (rows of ldq), k and v into the pages at `slots` (a negative one: nowhere); kv_heads 0: W = Wq only.
extern "C" int cisr_gemm_ring_rope(const void* A, int lda, const void* W, int ldw, void* q_out, int ldq, int M, int K, const int* positions,
                                   const int* slots, const float* cos_tab, const float* sin_tab, void* kcache, void* vcache, int heads,
                                   int kv_heads, int dim, int page_size, int max_pos, const float* sums, int parts, float eps, int tile,
                                   hipStream_t stream) {
    if (M <= 0 || heads <= 0) return 0;
    if (dim <= 0 || dim % 32 || kv_heads < 0 || max_pos <= 0 || !positions || !cos_tab || !sin_tab || (uintptr_t)cos_tab % 16 || (uintptr_t)sin_tab % 16 ||
        (kv_heads && (!slots || !kcache || !vcache || page_size <= 0 || (uintptr_t)kcache % 8)) || ldq < heads * dim)
        return (int)hipErrorInvalidValue;
    RingArgs a{(const bf16_t*)A, lda, (const bf16_t*)W, ldw, q_out, ldq, nullptr, 0, M, heads * dim, K, 0, GateLaw{}, 0, 1,
               positions, slots, cos_tab, sin_tab, (bf16_t*)kcache, (bf16_t*)vcache, heads, kv_heads, dim, std::max(page_size, 1), max_pos};
    if (!fits(a, 2)) return (int)hipErrorInvalidValue;
    finish_norm(a, sums, parts, eps);
    a.N = (heads + 2 * kv_heads) * dim;
    if (((long long)a.N + 512) * ldw * 2 >= 0x7fffffffll) return (int)hipErrorInvalidValue;
    return launch(a, tile ? tile : plan_of(M, a.N, K, false, 1).tile, RING_ROPE, stream);
}
