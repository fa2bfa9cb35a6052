// The 32-bit product  C[M,N] = A[M,K] . W[N,K]^T (+ R): float operands, float multiply-adds on the matrix cores
// (v_mfma_f32_16x16x4_f32, whose inputs and sums are whole floats: no reduced-precision mode).
//
// With few rows the product is a stream of W, with many it is bound by the matrix instruction; in between (the layer
// products of small models) it is a chain of trips to memory.  All three want K cut over the waves of a block: a tile of
// TM x TN sixteens of C is made by WK waves, each with a contiguous run of K's sixteens, DEPTH of them in flight; a wave
// hands its operands through LDS to the lanes that want them (loaded in the instruction's own layout, sixteen rows side by
// side in neighbouring lanes, a load costs the cache four times the lines: 2 rows 4.5 -> 3.9 us, 16 rows 5.9 -> 4.6 at
// 576 x 576), without a barrier; the waves' tiles meet in LDS once.
//
// The order of the sum of an element of C is fixed by K alone (WK by K, runs by WK, four interleaved chains a sixteen, a
// tree over the waves), whatever M, N and the tile are: a row's result does not depend on the other rows of a step.
//
// Measured on an MI355X beside what stood here before (vector multiply-adds in tiles of 64 x 64 x 16 staged through LDS: 9
// to 48 blocks at these sizes, one trip to memory a sixteen of K), 2 / 16 / 130 rows: 576 x 576 61 / 58 / 65 us -> 3.9 /
// 4.6 / 7.8, 3072 x 576 60 / 58 / 61 -> 4.2 / 5.1 / 13.4, 576 x 1536 158 / 152 / 170 -> 5.7 / 7.1 / 14.7; the head of two
// rows, 49152 x 576, 94 -> 28 (4.0 TB/s); 2,048 rows against 8192 x 2048 1,797 -> 786 (87 of 157 TFLOP/s).  Relative error
// against 64 bits 4.3e-7 -> 1.6e-7 (K = 576), 8.1e-7 -> 2.1e-7 (K = 2,048): K's runs are sums of their own.
//
// GATED and ROTARY products make two rows of W a column, the gate's and the up's or a rotary pair's two halves: half of a tile's sixteens
// (in tiles of one sixteen, half of its rows) are the first rows, the others the second, and the wave that finishes a sixteen
// holds both sums.  The activation, or the rotation
// with the keys' and values' way into their pages, is then no kernel of its own (2 rows at 576 x 3072 / 960: 2.1 and 3.2 us a layer and
// two gaps between kernels of about 1.5; 130 rows 4.7 and 4.9).
#include "common.h"

typedef __attribute__((ext_vector_type(4))) float gf_f32x4;

struct GemmF32Args {
    const float* A; int lda;
    const float* W; int ldw;
    float* C; int ldc;
    const float* R; int ldr;         // residual added at the end, or null; may be C
    int M, N, K;                     // N: columns of the product, or of the first rows (GATED), or pairs (ROTARY)
    int m_tiles;
    // ROTARY: W = [Wq; Wk; Wv], C the queries; pair i of a head is coordinates (i, i + dim / 2)
    const int* positions; const int* slots; const float* cos_tab; const float* sin_tab;
    float* kcache; float* vcache;
    int heads, kv_heads, dim, page_size, max_pos;
    // NORM
    const float* norm_w; float eps, inv_k;
    const int* rows;                 // row m of A is row rows[m] of x; null: row m
};
enum { F32_PLAIN = 0, F32_GATED = 1, F32_ROTARY = 2 };

// Four floats of row `row` at k; VEC: one 16-byte load, rows 16-byte aligned and K a multiple of 4.  Addresses are
// clamped, never branched around; what lies past K is cleared by `clear_tail`.
template <bool VEC>
__device__ __forceinline__ gf_f32x4 gf_load(const float* row, int k, int K) {
    if (VEC) return *(const gf_f32x4*)(row + min(k, K - 4));
    gf_f32x4 v;
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = row[min(k + e, K - 1)];
    return v;
}

__device__ __forceinline__ gf_f32x4 gf_clear_tail(gf_f32x4 v, int k, int K) {
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = k + e < K ? v[e] : 0.f;
    return v;
}

// What a wave wrote to LDS before is there for its own lanes after (a wave's LDS accesses are served in order: only the
// compiler must not move them).
__device__ __forceinline__ void wave_order() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// The pair (a, b) of row m, pair n (of all heads' pairs), turned by the angle (c, s): queries to C, keys and values to `slot`.
__device__ __forceinline__ void finish_pair(const GemmF32Args& p, int m, int n, float a, float b, float c, float s, int slot) {
    const int half = p.dim / 2, head = n / half, i = n % half;
    if (head < p.heads + p.kv_heads) {
        const float x = fmaf(a, c, -(b * s));         // (as the rotary kernel's sums are contracted: the same bits)
        b = fmaf(b, c, a * s);
        a = x;
    }
    if (head < p.heads) {
        float* q = p.C + (size_t)m * p.ldc + head * p.dim + i;
        q[0] = a;
        q[half] = b;
        return;
    }
    if (slot < 0) return;
    const int page = slot / p.page_size, off = slot % p.page_size;
    if (head < p.heads + p.kv_heads) {
        float* k = p.kcache + (((size_t)page * p.kv_heads + head - p.heads) * p.page_size + off) * p.dim + i;
        k[0] = a;
        k[half] = b;
    } else {
        float* v = p.vcache + (((size_t)page * p.kv_heads + head - p.heads - p.kv_heads) * p.dim + i) * p.page_size + off;
        v[0] = a;
        v[(size_t)half * p.page_size] = b;
    }
}

#define GF_RUN 256                       // NORM: floats of LDS for a wave's run of the norm's weights (a word a lane stores them; it reads at most 144)

// 16-byte words of LDS: the waves' operands on their way, and then their tiles
constexpr int gf_lds_items(int tm, int tn, int wk) { return wk * (tm * tn > tm + tn ? tm * tn : tm + tn) * WAVE; }

template <int TM, int TN, int WK, int DEPTH, bool VEC, int FORM, bool NORM>
__global__ void __launch_bounds__(WK * WAVE) gemm_f32_kernel(GemmF32Args p) {
    extern __shared__ __attribute__((aligned(16))) char gf_lds[];
    constexpr bool HALVES = FORM != F32_PLAIN && TN == 1;            // the sixteen's first eight rows of W and its last
    constexpr int OT = FORM == F32_PLAIN || HALVES ? TN : TN / 2;    // sixteens of columns (eights with HALVES)
    constexpr int OC = HALVES ? 8 : 16;
    gf_f32x4* meet = (gf_f32x4*)gf_lds;                              // [WK][TM * TN][64], after the waves are through
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid / WAVE), lane = tid % WAVE, r = lane % 16, g = lane / 16;
    const int m0 = (blockIdx.x % p.m_tiles) * TM * 16, n0 = (blockIdx.x / p.m_tiles) * OT * OC;   // (neighbours share rows of W)
    const int K = p.K, sixteens = (K + 15) / 16;
    const int first = (int)((long long)sixteens * wave / WK), last = (int)((long long)sixteens * (wave + 1) / WK);
    // Neighbouring lanes load neighbouring words of a row (lane: row lane / 4, four k from 4 (lane % 4)); the instruction wants
    // row lane % 16, four k from 4 (lane / 16).  They change places in LDS, in slots of the wave's own: 16 bytes at row * 4 +
    // (fourth ^ row / 2), so that neither way has two lanes on a bank.
    const int lrow = lane / 4, lk = 4 * (lane % 4);
    gf_f32x4* put = (gf_f32x4*)gf_lds + wave * (TM + TN) * WAVE + lrow * 4 + ((lane % 4) ^ (lrow / 2 % 4));
    const gf_f32x4* get = (const gf_f32x4*)gf_lds + wave * (TM + TN) * WAVE + r * 4 + (g ^ (r / 2 % 4));
    const float* a_row[TM];
    const float* w_row[TN];
#pragma unroll
    for (int i = 0; i < TM; ++i) {
        const int m = min(m0 + i * 16 + lrow, p.M - 1);
        a_row[i] = p.A + (size_t)(NORM && FORM == F32_PLAIN && p.rows ? p.rows[m] : m) * p.lda;
    }
#pragma unroll
    for (int j = 0; j < TN; ++j) {
        const int n = min(n0 + j % OT * OC + lrow % OC, p.N - 1), half = p.dim / 2;
        const bool second = HALVES ? lrow >= 8 : j >= OT;
        const int row = FORM == F32_PLAIN ? n : FORM == F32_GATED ? n + (second ? p.N : 0) : n / half * p.dim + n % half + (second ? half : 0);
        w_row[j] = p.W + (size_t)row * p.ldw;
    }
    gf_f32x4 acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) acc[i][j] = (gf_f32x4){0.f, 0.f, 0.f, 0.f};
    gf_f32x4 fa[DEPTH][TM], fw[DEPTH][TN];
    float squares[TM];                                               // NORM: of the lane's words of its rows
#pragma unroll
    for (int i = 0; i < TM; ++i) squares[i] = 0.f;
    auto ask = [&](int d, int s) {
        const int k = min(s, sixteens - 1) * 16 + lk;
#pragma unroll
        for (int j = 0; j < TN; ++j) fw[d][j] = gf_load<VEC>(w_row[j], k, K);
#pragma unroll
        for (int i = 0; i < TM; ++i) fa[d][i] = gf_load<VEC>(a_row[i], k, K);
    };
    // NORM: the wave's run of the norm's weights waits in LDS and is read a sixteen ahead of its use, beside operands that take the registers
    float* const ssq = (float*)((gf_f32x4*)gf_lds + gf_lds_items(TM, TN, WK));      // [WK][TM * 16] sums of squares
    float* const run = ssq + WK * TM * 16 + wave * GF_RUN - first * 16;              // [WK][GF_RUN], from its first sixteen on
    gf_f32x4 next = {0.f, 0.f, 0.f, 0.f};
    auto use = [&](int d, int s) {
        const gf_f32x4 norm = next;
        if constexpr (NORM) next = *(const gf_f32x4*)(run + min(s + 1, last - 1) * 16 + lk);
        if (s * 16 + 16 > K) {                                       // (uniform: K's last, partly filled sixteen)
            const int k = s * 16 + lk;
#pragma unroll
            for (int j = 0; j < TN; ++j) fw[d][j] = gf_clear_tail(fw[d][j], k, K);
#pragma unroll
            for (int i = 0; i < TM; ++i) fa[d][i] = gf_clear_tail(fa[d][i], k, K);
        }
        if constexpr (NORM)
#pragma unroll
            for (int i = 0; i < TM; ++i) {
                const gf_f32x4 x = fa[d][i];
                squares[i] += (x[0] * x[0] + x[1] * x[1]) + (x[2] * x[2] + x[3] * x[3]);
                fa[d][i] = x * norm;
            }
#pragma unroll
        for (int j = 0; j < TN; ++j) put[j * WAVE] = fw[d][j];
#pragma unroll
        for (int i = 0; i < TM; ++i) put[(TN + i) * WAVE] = fa[d][i];
        wave_order();
        gf_f32x4 xa[TM], xw[TN];
#pragma unroll
        for (int j = 0; j < TN; ++j) xw[j] = get[j * WAVE];
#pragma unroll
        for (int i = 0; i < TM; ++i) xa[i] = get[(TN + i) * WAVE];
        wave_order();
#pragma unroll
        for (int e = 0; e < 4; ++e)
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int j = 0; j < TN; ++j)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(xa[i][e], xw[j][e], acc[i][j], 0, 0, 0);
    };
    const int t = tid / WAVE, i = t / OT, j = t % OT;                // (the first TM OT waves finish a sixteen by sixteen each)
    static_assert(TM * OT <= WK, "a wave finishes at most one sixteen by sixteen");
    const bool finishes = t < TM * OT;
    const int n = n0 + j * OC + r % OC, m = m0 + i * 16 + 4 * g;
    // (the rows' positions are asked for before the operands and the angles behind the first of them, not at the end)
    int pos[4] = {0, 0, 0, 0}, slot[4] = {-1, -1, -1, -1};
    float turn_c[4] = {1.f, 1.f, 1.f, 1.f}, turn_s[4] = {0.f, 0.f, 0.f, 0.f};
    if (FORM == F32_ROTARY && finishes)
#pragma unroll
        for (int e = 0; e < 4; ++e) pos[e] = p.positions[min(m + e, p.M - 1)];
    gf_f32x4 mine;
    if constexpr (NORM) mine = gf_load<VEC>(p.norm_w, first * 16 + 4 * lane, K);
#pragma unroll
    for (int d = 0; d < DEPTH; ++d) {
        ask(d, first + d);
        __builtin_amdgcn_sched_barrier(0);
    }
    if constexpr (NORM) {
        *(gf_f32x4*)(run + first * 16 + 4 * lane) = mine;
        wave_order();
        next = *(const gf_f32x4*)(run + first * 16 + lk);
    }
    if (FORM == F32_ROTARY && finishes) {
        const int half = p.dim / 2, angle = min(n, p.N - 1) % half;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const size_t at = (size_t)min(max(pos[e], 0), p.max_pos - 1) * half + angle;
            turn_c[e] = p.cos_tab[at];
            turn_s[e] = p.sin_tab[at];
            if (p.kv_heads > 0) slot[e] = p.slots[min(m + e, p.M - 1)];
        }
    }
    // whole turns ask for the turn behind them (past the last sixteen: that one again, so that every wait counts the same
    // loads); the last turn asks for nothing: a wave with up to DEPTH sixteens is one trip to memory
    int turn = first;
    for (; turn + DEPTH < last; turn += DEPTH)
#pragma unroll
        for (int d = 0; d < DEPTH; ++d) {
            use(d, turn + d);
            __builtin_amdgcn_sched_barrier(0);
            ask(d, turn + d + DEPTH);
            __builtin_amdgcn_sched_barrier(0);
        }
#pragma unroll
    for (int d = 0; d < DEPTH; ++d)
        if (turn + d < last) use(d, turn + d);                       // (uniform over the wave)
    // element 4 g + e of a lane's four is row 4 g + e, column r of its sixteen by sixteen
    constexpr int ITEMS = TM * TN * WAVE;
    if constexpr (NORM)
#pragma unroll
        for (int ii = 0; ii < TM; ++ii) {                            // (a row's words of a sixteen are its quad's)
            float x = squares[ii];
            x += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), 0xb1, 0xf, 0xf, false));     // quad_perm 1, 0, 3, 2
            x += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), 0x4e, 0xf, 0xf, false));     // quad_perm 2, 3, 0, 1
            if (lane % 4 == 0) ssq[(wave * TM + ii) * 16 + lrow] = x;
        }
    float resid[4] = {0.f, 0.f, 0.f, 0.f};
    if (finishes && p.R && n < p.N)
#pragma unroll
        for (int e = 0; e < 4; ++e) resid[e] = p.R[(size_t)min(m + e, p.M - 1) * p.ldr + n];
    __syncthreads();                                                 // (the slots above are free)
#pragma unroll
    for (int ii = 0; ii < TM; ++ii)
#pragma unroll
        for (int jj = 0; jj < TN; ++jj) meet[(wave * TM * TN + ii * TN + jj) * WAVE + lane] = acc[ii][jj];
    __syncthreads();
    if (!finishes) return;
    gf_f32x4 factor = {1.f, 1.f, 1.f, 1.f};
    if constexpr (NORM) {
        // (a row a lane, and all lanes change them, those past the last column too: four rows a lane, with the library's root and quotients, are 0.7 us)
        float all = 0.f;
#pragma unroll
        for (int w = 0; w < WK; ++w) all += ssq[(w * TM + i) * 16 + r];
        const float f = row_factor(all, p.inv_k, p.eps);
#pragma unroll
        for (int e = 0; e < 4; ++e) factor[e] = __shfl(f, 4 * g + e, WAVE);
    }
    if (!HALVES && n >= p.N) return;
    auto total = [&](int tile) {
        gf_f32x4 part[WK];
#pragma unroll
        for (int w = 0; w < WK; ++w) part[w] = meet[w * ITEMS + tile * WAVE + lane];
#pragma unroll
        for (int half = WK / 2; half > 0; half /= 2)
#pragma unroll
            for (int w = 0; w < half; ++w) part[w] += part[w + half];
        return part[0];
    };
    gf_f32x4 sum = total(i * TN + j);
    if constexpr (NORM) sum *= factor;
    if constexpr (FORM == F32_PLAIN) {
#pragma unroll
        for (int e = 0; e < 4; ++e)
            if (m + e < p.M) p.C[(size_t)(m + e) * p.ldc + n] = sum[e] + resid[e];
    } else {
        gf_f32x4 second;
        if constexpr (HALVES) {
#pragma unroll
            for (int e = 0; e < 4; ++e) second[e] = __shfl_xor(sum[e], 8, WAVE);
        } else {
            second = total(i * TN + OT + j) * factor;
        }
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            if (m + e >= p.M || (HALVES && (r >= 8 || n >= p.N))) continue;
            if constexpr (FORM == F32_GATED) p.C[(size_t)(m + e) * p.ldc + n] = sum[e] / (1.0f + expf(-sum[e])) * second[e];
            else finish_pair(p, m + e, n, sum[e], second[e], turn_c[e], turn_s[e], slot[e]);
        }
    }
}

template <int TM, int TN, int WK, int DEPTH, bool VEC, int FORM, bool NORM>
static int launch_f32(GemmF32Args p, hipStream_t stream) {
    constexpr int COLUMNS = FORM == F32_PLAIN ? 16 * TN : 8 * TN;
    p.m_tiles = (p.M + 16 * TM - 1) / (16 * TM);
    const long long blocks = (long long)p.m_tiles * ((p.N + COLUMNS - 1) / COLUMNS);
    if (blocks > 0x7fffffff) return (int)hipErrorInvalidValue;
    constexpr int lds = gf_lds_items(TM, TN, WK) * (int)sizeof(gf_f32x4) + (NORM ? WK * (TM * 16 + GF_RUN) * (int)sizeof(float) : 0);
    if (lds > 65536) {
        const hipError_t e = hipFuncSetAttribute((const void*)gemm_f32_kernel<TM, TN, WK, DEPTH, VEC, FORM, NORM>, hipFuncAttributeMaxDynamicSharedMemorySize, lds);
        if (e != hipSuccess) return (int)e;
    }
    gemm_f32_kernel<TM, TN, WK, DEPTH, VEC, FORM, NORM><<<(unsigned)blocks, WK * WAVE, lds, stream>>>(p);
    return CISR_LAUNCH_CHECK();
}

// The tile (sixteens of rows x sixteens of W's rows): the smallest that needs no more blocks than there are compute units, as a block alone
// on its unit takes the longer the larger its tile, and a second round costs more.  192 rows, us of the tile before / now: 576 x 576 2 x 2
// (108 blocks) 8.2 / 1 x 2 (216) 6.4, 576 x 1,536 15.2 / 1 x 2 11.3, 960 x 576 8.7 / 2 x 2 with two sixteens in flight instead of four 7.9,
// 3,072 x 576 gated 2 x 2 (576) 18.1 / 3 x 4 (192) 15.8; 2,048 x 2,048 33 / 3 x 2 24; 512 x 576, K 1,536 26.6 / 3 x 2 18.9.  (3 x 4 only where
// 2 x 2 would be more than 512, 4 x 4 where it would be more than 800: 90 x 4,608 x 768 gated, 432 of them, 18.2 / 17.0; 256 x 3,072 x 576, 768,
// 20.2 / 18.0; 1,024 x 960, 960, 19.6 / 20.8.)
// Beyond one round, K below 1,024: 2 x 4 has two blocks a unit and is ahead where these are many (1,024 x 3,072 x 576, 1,536 of them, 49.5, with 2 x 2
// 52.5; 2,048 x 2,048 x 1,000 105 / 110) or fill their last round of 512 well (4,096 x 512 x 512, 1,024, 31.2 / 33.3; 1,800 x 1,000 x 1,000, 912, 56.4 / 60.7;
// 1,300 rows, 656, 43.8 / 46.3), 2 x 2 else (384 x 3,072 x 576, 576, 28.3 / 25.0; 700 rows, 1,056, 40.6 / 39.7; K 512 to 960 up to half a round:
// 1,024 x 1,536 x 576, 768, 31.5 / 29.1).  K from 1,024 on: 4 x 2 for up to 256 rows that fill it (192 x 8,192 x 2,048 84.5, 2 x 4 90; 130 x 6,144 x 1,024
// 43.8, 2 x 2 37.8); else 2 x 2 with four sixteens in flight up to 400 blocks of 2 x 4 (300 x 2,048 x 2,048 48.6, 2 x 4 55.2, K 8,192
// 148 / 195), then 2 x 4 (1,500 x 576 x 1,536, 423 blocks, 44.2, 2 x 2 55.2; 512 x 8,192 x 2,048 207, 4 x 2 210).
// Rows that are not aligned load word by word: three tiles, 2 x 4 from 512 of them on (512 x 3,072 x 577 58.4, 2 x 2 69.9; 1,024 x 8,192 x 1,030 572 / 658).
// Up to 16 rows the tile has 16 of them.  A tile never changes a sum: its order is K's.
template <int WK, bool VEC, int FORM, bool NORM>
static int launch_f32_tile(const GemmF32Args& p, hipStream_t stream) {
    const int cols = FORM == F32_PLAIN ? p.N : 2 * p.N;
    auto blocks = [&](int tm, int tn) { return (long long)((p.M + 16 * tm - 1) / (16 * tm)) * ((cols + 16 * tn - 1) / (16 * tn)); };
    auto one_round = [&](int tm, int tn) { return blocks(tm, tn) <= 256; };
    constexpr int DEEP = WK == 16 ? 8 : 4;               // sixteens in flight where a wave has few operands each
    const long long wide = blocks(2, 4);
    if (p.M <= 16 || one_round(1, 1)) return launch_f32<1, 1, WK, DEEP, VEC, FORM, NORM>(p, stream);
    if constexpr (!VEC) {
        if (wide >= 512) return launch_f32<2, 4, WK, 2, VEC, FORM, NORM>(p, stream);
        if constexpr (WK == 16)                           // (192 x 2,048 x 4,099 152 us with two sixteens in flight, 146 with four)
            if (p.K >= 2048 && blocks(2, 2) >= 128) return launch_f32<2, 2, WK, 4, VEC, FORM, NORM>(p, stream);
    } else {
        if (one_round(1, 2)) return launch_f32<1, 2, WK, 4, VEC, FORM, NORM>(p, stream);
        if (one_round(2, 2)) return launch_f32<2, 2, WK, 2, VEC, FORM, NORM>(p, stream);
        if (one_round(3, 2)) return launch_f32<3, 2, WK, 2, VEC, FORM, NORM>(p, stream);
        if (one_round(4, 2)) return launch_f32<4, 2, WK, 2, VEC, FORM, NORM>(p, stream);
        if constexpr (WK == 8 && FORM != F32_PLAIN) {    // (a wave finishes at most one sixteen by sixteen of columns)
            if (one_round(3, 4) && blocks(2, 2) > 512) return launch_f32<3, 4, WK, 2, VEC, FORM, NORM>(p, stream);
            if (one_round(4, 4) && blocks(2, 2) > 800) return launch_f32<4, 4, WK, 2, VEC, FORM, NORM>(p, stream);
        }
        if constexpr (WK == 16) {
            if (p.M <= 256 && wide > 400 && blocks(4, 2) <= wide) return launch_f32<4, 2, WK, 2, VEC, FORM, NORM>(p, stream);
            return wide <= 400 ? launch_f32<2, 2, WK, 4, VEC, FORM, NORM>(p, stream) : launch_f32<2, 4, WK, 2, VEC, FORM, NORM>(p, stream);
        }
        const int over = (int)(wide % 512), most = p.K >= 512 && p.K <= 960 ? 256 : 128;
        if (wide >= 1200 || (wide >= 512 && (over == 0 || over > most))) return launch_f32<2, 4, WK, 2, VEC, FORM, NORM>(p, stream);
    }
    return launch_f32<2, 2, WK, 2, VEC, FORM, NORM>(p, stream);
}

// Waves a tile: sixteen from an inner size of 1,024 on, else eight (so that a wave has at least two sixteens at the small
// models' 576).  A fused norm takes eight waves and rows in 16-byte words only; up to how many results it is the faster, with both sides'
// times, stands at f32_norm_ahead (kernels/ops.py).
#define GF_SIXTEEN_WAVES 1024
static_assert(GF_SIXTEEN_WAVES / 8 + 16 <= GF_RUN, "a wave's run of the norm's weights");
template <int FORM>
static int launch_f32_form(const GemmF32Args& p, hipStream_t stream) {
    const bool vec = p.K % 4 == 0 && p.lda % 4 == 0 && p.ldw % 4 == 0 && (uintptr_t)p.A % 16 == 0 && (uintptr_t)p.W % 16 == 0;
    if (p.norm_w) {
        if (!vec || (uintptr_t)p.norm_w % 16 || p.K >= GF_SIXTEEN_WAVES) return (int)hipErrorInvalidValue;
        return launch_f32_tile<8, true, FORM, true>(p, stream);
    }
    if (p.K >= GF_SIXTEEN_WAVES) return vec ? launch_f32_tile<16, true, FORM, false>(p, stream) : launch_f32_tile<16, false, FORM, false>(p, stream);
    return vec ? launch_f32_tile<8, true, FORM, false>(p, stream) : launch_f32_tile<8, false, FORM, false>(p, stream);
}

// The entry points with `norm_w`: A is float rows x, and the product's rows are RMSNorm(x[rows]) (rows null: of x's rows in order).

// C[M, N] = silu(A . Wg^T) * (A . Wu^T) with W = [Wg; Wu], 2 N rows
extern "C" int cisr_gemm_f32_swiglu(const float* A, int lda, const float* W, int ldw, float* C, int ldc, int M, int N, int K,
                                    const float* norm_w, float eps, hipStream_t stream) {
    if (M <= 0 || N <= 0) return 0;
    if (K <= 0) return (int)hipErrorInvalidValue;
    GemmF32Args p{A, lda, W, ldw, C, ldc, nullptr, 0, M, N, K, 0};
    p.norm_w = norm_w;
    p.eps = eps;
    p.inv_k = 1.0f / (float)K;
    return launch_f32_form<F32_GATED>(p, stream);
}

// W = [Wq; Wk; Wv] (kv_heads 0: Wq alone): queries and keys turned over the whole head by the rows' positions, queries to C, keys
// and values to the pages at `slots`
extern "C" int cisr_gemm_f32_rope(const float* A, int lda, const float* W, int ldw, float* q_out, int ldq, int M, int K, const int* positions,
                                  const int* slots, const float* cos_tab, const float* sin_tab, float* kcache, float* vcache, int heads,
                                  int kv_heads, int dim, int page_size, int max_pos, const float* norm_w, float eps, hipStream_t stream) {
    if (M <= 0 || heads <= 0) return 0;
    if (K <= 0 || dim <= 0 || dim % 2 || kv_heads < 0 || page_size <= 0 || max_pos <= 0 || !positions || (kv_heads && (!slots || !kcache || !vcache)))
        return (int)hipErrorInvalidValue;
    GemmF32Args p{A, lda, W, ldw, q_out, ldq, nullptr, 0, M, (heads + 2 * kv_heads) * dim / 2, K, 0,
                  positions, slots, cos_tab, sin_tab, kcache, vcache, heads, kv_heads, dim, page_size, max_pos, norm_w, eps, 1.0f / (float)K};
    return launch_f32_form<F32_ROTARY>(p, stream);
}

extern "C" int cisr_gemm_f32(const float* A, int lda, const float* W, int ldw, float* C, int ldc, const float* R, int ldr, int M, int N, int K,
                             const float* norm_w, float eps, const int* rows, hipStream_t stream) {
    if (M <= 0 || N <= 0) return 0;
    if (K <= 0 || (rows && !norm_w)) return (int)hipErrorInvalidValue;
    GemmF32Args p{A, lda, W, ldw, C, ldc, R, ldr, M, N, K, 0};
    p.norm_w = norm_w;
    p.eps = eps;
    p.inv_k = 1.0f / (float)K;
    p.rows = rows;
    return launch_f32_form<F32_PLAIN>(p, stream);
}
