// Matrix products  C[M,N] = A[M,K] . W[N,K]^T (+ R)  for linear layers whose
// weights are stored [out, in] (reference: runtime/blas.py:41-56 does the same
// product through a vendor library).
//
//  * gemm_bf16: bf16 operands on the matrix cores (v_mfma_f32_16x16x32_bf16),
//    float accumulation; output float or bf16.  (Float operands: gemm_f32.hip.)
// Any M, N, K >= 1.  R (float, may be null, may alias a float C) is a
// residual added in the epilogue from the float accumulator.
#include "common.h"

// ------------------------------------------------------------------- bf16
typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(4))) float f32x4;
typedef __attribute__((ext_vector_type(4))) uint32_t u32x4;

// 16 bytes = 8 bf16 from row-major global memory, zero-filled outside the matrix.
// VEC: rows are 16-byte aligned and K % 8 == 0, so a chunk lies wholly inside or outside; the load
// is unconditional from a clamped address (no branch between the loads of a tile, so they are all
// in flight together) and the result is zeroed by a select.  Otherwise element by element.
template <bool VEC>
__device__ __forceinline__ u32x4 load_chunk(const bf16_t* base, int ld, int row, int nrows, int k, int K) {
    if (VEC) {
        // no branch and nothing that touches the loaded value (it would wait for the load): rows
        // past the end read the last row (their products land in output rows or columns that are
        // never stored); a chunk past K reads the last chunk and is zeroed by a mask when the tile
        // is written to LDS, so that nothing is added to valid outputs
        const int rr = row < nrows ? row : nrows - 1;
        const int kk = k < K ? k : K - 8;
        return *(const u32x4*)(base + (size_t)rr * ld + kk);   // the caller masks chunks past K when it uses them
    }
    u32x4 v = {0u, 0u, 0u, 0u};
    if (row >= nrows || k >= K) return v;
    const bf16_t* p = base + (size_t)row * ld + k;
    uint32_t w[4] = {0u, 0u, 0u, 0u};
#pragma unroll
    for (int e = 0; e < 8; ++e)
        if (k + e < K) w[e / 2] |= ((uint32_t)p[e]) << (16 * (e % 2));
    v.x = w[0]; v.y = w[1]; v.z = w[2]; v.w = w[3];
    return v;
}

// Side of the patches in which tiles are numbered: `tiles` cut into the fewest parts of at most 8, evenly.
__host__ __device__ inline int patch_side(int tiles) {
    const int parts = (tiles + 7) / 8;
    return (tiles + parts - 1) / parts;
}

// Block tile (16 WM TM) x (32 TN), BK deep; WM x 2 waves (WM = 2 or 4), each wave TM x TN tiles of 16 x 16.
// Operands go global memory -> registers -> LDS -> matrix-core operands: PF tiles of global loads are in flight in a ring of
// registers, and two LDS buffers let the next tile be written while the current one is multiplied, with one barrier per tile.
// The products that come here leave a compute unit one or two blocks, so the time is the chain of a block's turns (copy, barrier,
// LDS reads, products) and not the matrix cores.  What shortens it: eight waves a block, so that a SIMD has a second wave to run
// in the waits of the first; 128 of the inner size a turn in the small tiles, half as many barriers; exact waits (below).
// Measured on an MI355X, rows x columns x inner size, four waves and 64 a turn before: 1,741 x 576 x 1,536 16.3 -> 8.8 us, 1,741 x
// 960 x 576 8.8 -> 7.4, 100 x 2,048 x 2,048 12.6 -> 8.0, 300 x 2,048 x 2,048 16.1 -> 11.0, 4,000 x 4,096 x 2,048 144 -> 94 (0.71
// PFLOP/s), 1,741 x 1,536 x 576 with SwiGLU 17.8 -> 16.1, 100 x 4,096 x 2,048 with it 17.3 -> 10.8.  Reading a turn's operands
// ahead of the next tile's copies (two tiles deep in LDS) was 5-25 % slower: the copies' waits then stand before the products.
// SWIGLU: W holds two blocks of N rows, `dual_off` rows apart (gate, then up).  A wave's first TN/2
// column tiles take gate rows and its last TN/2 the up rows of the same output columns, so a lane ends
// with gate and up of one output element in its registers and writes silu(gate) * up (both rounded to
// bf16 first, as the two-kernel path does); a block then covers BN/2 output columns.
// A batch of products in one launch (grid.y of them): product h reads A + h a, W + h w and writes C + h c (elements);
// with `gate`, row m of product h is multiplied by sigmoid(gate[m * ldg + h]); with `act` (ACT_*, no residual) an ungated
// activation is applied before the store.  Zeros: one product, no gate, no activation.
struct HeadBatch { long long a, w, c; const float* gate; int ldg; int act; };

template <int TM, int TN, int BK, typename TC, bool VEC, bool TAIL, bool SWIGLU = false, int WM = 2, int PF = 3>
__global__ void __launch_bounds__(WM * 128)
gemm_bf16_kernel(const bf16_t* __restrict__ A, int lda, const bf16_t* __restrict__ W, int ldw,
                 TC* C, int ldc, const float* R, int ldr, int M, int N, int K, int dual_off = 0, GateLaw law = {},
                 HeadBatch heads = {}) {
    static_assert(!SWIGLU || (TN % 2 == 0 && VEC), "the activation pairs column tiles");
    // blockIdx.y: which of a batch of products with a matrix of its own each (one launch for all heads)
    A += (size_t)blockIdx.y * heads.a;
    W += (size_t)blockIdx.y * heads.w;
    C += (size_t)blockIdx.y * heads.c;
    constexpr int BM = WM * TM * 16, BN = 2 * TN * 16, NT = WM * 128;   // WM x 2 waves
    constexpr int BN_OUT = SWIGLU ? BN / 2 : BN;           // output columns a block covers
    constexpr int CPR = BK / 8;                            // 16-byte chunks per tile row
    // LDS rows are not padded; the 16-byte chunks of a row are permuted by a function of the row instead,
    // so that neither the copies into LDS (consecutive chunks of a few rows) nor the operand reads (one
    // chunk of 16 consecutive rows) meet in a bank
    auto lds_at = [](int row, int chunk) {
        const int turn = BK == 32 ? ((row >> 1) ^ (row >> 3)) : (row ^ (row >> 3));
        return row * BK + ((chunk ^ turn) & (CPR - 1)) * 8;
    };
    static_assert((BM * CPR) % NT == 0 && (BN * CPR) % NT == 0, "a tile is a whole number of 16-byte chunks per thread");
    constexpr int A_PER_THREAD = BM * CPR / NT;
    constexpr int W_PER_THREAD = BN * CPR / NT;
    __shared__ __attribute__((aligned(16))) bf16_t As[2][BM * BK];
    __shared__ __attribute__((aligned(16))) bf16_t Ws[2][BN * BK];

    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid / WAVE), lane = tid % WAVE;   // (uniform: scalar loop control)
    const int wm = wave / 2, wn = wave % 2;
    const int r = lane % 16, g = lane / 16;
    // The hardware deals consecutive workgroups round-robin to the 8 XCDs, each with an L2 of its own.
    // Renumber so that an XCD gets a contiguous run of tiles, and order the tiles in patches of up to
    // 8 x 8 (sides as even as the tile counts allow, so that few slots fall outside the matrix): the sixty-odd blocks that run on an XCD at one time then share 8 row bands of A and 8 of W
    // (16 bands from memory for 64 tiles) instead of one band of A and 64 of W.
    const int tiles_m = (M + BM - 1) / BM, tiles_n = (N + BN_OUT - 1) / BN_OUT;
    const int tiles = tiles_m * tiles_n, per_xcd = (tiles + 7) / 8;
    const int slot = (blockIdx.x % 8) * per_xcd + blockIdx.x / 8;
    if (slot >= tiles) return;                             // the grid is rounded up to a multiple of 8
    // (the last patches of a row or column are cut to the matrix: a slot outside it would leave its compute unit idle
    // while another takes two tiles)
    const int gm = patch_side(tiles_m), gn = patch_side(tiles_n);
    const int band = slot / (gm * tiles_n), rows = min(gm, tiles_m - band * gm);
    const int in_band = slot - band * gm * tiles_n, patch = in_band / (rows * gn), in_patch = in_band - patch * rows * gn;
    const int tile_m = band * gm + in_patch % rows, tile_n = patch * gn + in_patch / rows;
    const int m0 = tile_m * BM, n0 = tile_n * BN_OUT;

    f32x4 acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) acc[i][j] = (f32x4){0.f, 0.f, 0.f, 0.f};

    u32x4 ra[PF][A_PER_THREAD], rw[PF][W_PER_THREAD];
    auto fetch = [&](int k0, u32x4 (&fa)[A_PER_THREAD], u32x4 (&fw)[W_PER_THREAD]) {
#pragma unroll
        for (int i = 0; i < A_PER_THREAD; ++i) {
            const int c = tid + i * NT;
            fa[i] = load_chunk<VEC>(A, lda, m0 + c / CPR, M, k0 + (c % CPR) * 8, K);
        }
#pragma unroll
        for (int i = 0; i < W_PER_THREAD; ++i) {
            const int c = tid + i * NT;
            if (SWIGLU) {
                // local column -> (wave, column tile, column): the W row of its output column, gate or up
                const int lc = c / CPR, jj = (lc % (TN * 16)) / 16;
                const int oc = min(n0 + (lc / (TN * 16)) * (TN / 2) * 16 + (jj % (TN / 2)) * 16 + lc % 16, N - 1);
                fw[i] = load_chunk<VEC>(W, ldw, oc + (jj >= TN / 2 ? dual_off : 0), dual_off + N, k0 + (c % CPR) * 8, K);
            } else {
                fw[i] = load_chunk<VEC>(W, ldw, n0 + c / CPR, N, k0 + (c % CPR) * 8, K);
            }
        }
    };
#pragma unroll
    for (int s = 0; s < PF; ++s) fetch(s * BK, ra[s], rw[s]);   // beyond K: the last chunk again (VEC) or zeros, never used

    auto turn = [&](int t, u32x4 (&ta)[A_PER_THREAD], u32x4 (&tw)[W_PER_THREAD], bool ask) {
        const int kk0 = t * BK, buf = t & 1;
        // TAIL (K is no multiple of BK): chunks beyond K, which only the last tile has and the loop's turns (ask) never see, are
        // cleared on both sides: zero times an infinite weight of the row's last chunk, which they repeat, is no number.
        auto put = [&](bf16_t* to, int c, const u32x4& chunk) {
            *(u32x4*)(to + lds_at(c / CPR, c % CPR)) = chunk & (TAIL && !ask && kk0 + c % CPR * 8 >= K ? 0u : 0xffffffffu);
        };
#pragma unroll
        for (int i = 0; i < A_PER_THREAD; ++i) put(As[buf], tid + i * NT, ta[i]);
#pragma unroll
        for (int i = 0; i < W_PER_THREAD; ++i) put(Ws[buf], tid + i * NT, tw[i]);
        // one barrier a tile: whoever writes this buffer again (two tiles on) has passed
        // the next tile's barrier, which every wave reaches only after reading this one
        __syncthreads();
        if (ask) fetch(kk0 + PF * BK, ta, tw);
#pragma unroll
        for (int kk = 0; kk < BK; kk += 32) {
            bf16x8 fa[TM], fw[TN];
#pragma unroll
            for (int i = 0; i < TM; ++i)
                fa[i] = *(const bf16x8*)(&As[buf][lds_at(wm * TM * 16 + i * 16 + r, kk / 8 + g)]);
#pragma unroll
            for (int j = 0; j < TN; ++j)
                fw[j] = *(const bf16x8*)(&Ws[buf][lds_at(wn * TN * 16 + j * 16 + r, kk / 8 + g)]);
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int j = 0; j < TN; ++j)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fa[i], fw[j], acc[i][j], 0, 0, 0);
        }
    };
    // Every turn of the loop asks for PF tiles and uses PF, with no branch between: only then are the waits counted exactly
    // (a load asked for under a condition makes the next wait one for all that is in flight).  The last turn asks for nothing.
    const int k_tiles = (K + BK - 1) / BK;
    int t = 0;
    for (; t + PF < k_tiles; t += PF)
#pragma unroll
        for (int s = 0; s < PF; ++s) turn(t + s, ra[s], rw[s], true);
#pragma unroll
    for (int s = 0; s < PF; ++s)
        if (t + s < k_tiles) turn(t + s, ra[s], rw[s], false);
    if (SWIGLU) {
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN / 2; ++j) {
                const int n = n0 + wn * (TN / 2) * 16 + j * 16 + r;
                if (n >= N) continue;
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const int m = m0 + wm * TM * 16 + i * 16 + g * 4 + e;
                    const float gq = bf16_to_f32(f32_to_bf16(acc[i][j][e])), uq = bf16_to_f32(f32_to_bf16(acc[i][j + TN / 2][e]));
                    if (m < M) store_f32(C + (size_t)m * ldc + n, gated_activation<TC>(gq, uq, law));
                }
            }
        return;
    }
    // lane holds rows 4g..4g+3 of column r in every 16 x 16 tile.  The residual is read with
    // unconditional loads from clamped addresses, all issued before the first is used.
    if (R) {
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j) {
                const int n = min(n0 + wn * TN * 16 + j * 16 + r, N - 1);
                float rv[4];
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const int m = min(m0 + wm * TM * 16 + i * 16 + g * 4 + e, M - 1);
                    rv[e] = R[(size_t)m * ldr + n];
                }
#pragma unroll
                for (int e = 0; e < 4; ++e) acc[i][j][e] += rv[e];
            }
    }
    if (heads.gate) {
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int m = min(m0 + wm * TM * 16 + i * 16 + g * 4 + e, M - 1);
                const float s = 1.0f / (1.0f + expf(-heads.gate[(size_t)m * heads.ldg + blockIdx.y]));
#pragma unroll
                for (int j = 0; j < TN; ++j) acc[i][j][e] *= s;
            }
    }
#pragma unroll
    for (int i = 0; i < TM; ++i) {
#pragma unroll
        for (int j = 0; j < TN; ++j) {
            const int n = n0 + wn * TN * 16 + j * 16 + r;
            if (n >= N) continue;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int m = m0 + wm * TM * 16 + i * 16 + g * 4 + e;
                if (m < M) store_f32(C + (size_t)m * ldc + n, heads.act ? activated<TC>(acc[i][j][e], heads.act) : acc[i][j][e]);
            }
        }
    }
}

template <int TM, int TN, int BK, int WM = 2, int PF = 3>
static int launch_bf16(const bf16_t* A, int lda, const bf16_t* W, int ldw, void* C, int ldc, const float* R,
                       int ldr, int M, int N, int K, int out_dtype, hipStream_t stream, HeadBatch heads = {}, int n_heads = 1) {
    constexpr int BM = WM * TM * 16, BN = 2 * TN * 16, NT = WM * 128;
    const long long tiles = (long long)((M + BM - 1) / BM) * ((N + BN - 1) / BN);
    if (tiles > (1ll << 30) || n_heads < 1 || n_heads > 65535) return (int)hipErrorInvalidValue;
    dim3 grid((unsigned)((tiles + 7) / 8 * 8), n_heads);
    const bool vec = lda % 8 == 0 && ldw % 8 == 0 && K % 8 == 0 && ((uintptr_t)A) % 16 == 0 && ((uintptr_t)W) % 16 == 0 &&
                     heads.a % 8 == 0 && heads.w % 8 == 0;
    const GateLaw law{};
#define GEMM_OF(TC, VEC, TAIL) gemm_bf16_kernel<TM, TN, BK, TC, VEC, TAIL, false, WM, PF><<<grid, NT, 0, stream>>>( \
        A, lda, W, ldw, (TC*)C, ldc, R, ldr, M, N, K, 0, law, heads)
#define GEMM_TO(TC) do { if (!vec) GEMM_OF(TC, false, false); else if (K % BK) GEMM_OF(TC, true, true); else GEMM_OF(TC, true, false); } while (0)
    if (out_dtype == DT_F32) GEMM_TO(float);
    else GEMM_TO(bf16_t);
#undef GEMM_TO
#undef GEMM_OF
    return CISR_LAUNCH_CHECK();
}

// C[M, N] = silu(A . Wg^T) * (A . Wu^T), W = [Wg; Wu] with `dual_off` rows between the blocks; bf16 in and out,
// 16-byte aligned rows with K % 8 == 0.
template <int TM, int TN, int BK, int WM = 2, int PF = 3>
static int launch_bf16_swiglu(const bf16_t* A, int lda, const bf16_t* W, int ldw, bf16_t* C, int ldc, int M, int N, int K,
                              int dual_off, GateLaw law, hipStream_t stream) {
    constexpr int BM = WM * TM * 16, BN_OUT = TN * 16;
    const long long tiles = (long long)((M + BM - 1) / BM) * ((N + BN_OUT - 1) / BN_OUT);
    if (tiles > (1ll << 30)) return (int)hipErrorInvalidValue;
    dim3 grid((unsigned)((tiles + 7) / 8 * 8));
    if (K % BK) gemm_bf16_kernel<TM, TN, BK, bf16_t, true, true, true, WM, PF><<<grid, WM * 128, 0, stream>>>(A, lda, W, ldw, C, ldc, nullptr, 0, M, N, K, dual_off, law);
    else gemm_bf16_kernel<TM, TN, BK, bf16_t, true, false, true, WM, PF><<<grid, WM * 128, 0, stream>>>(A, lda, W, ldw, C, ldc, nullptr, 0, M, N, K, dual_off, law);
    return CISR_LAUNCH_CHECK();
}

// `tile`: 0 picks by the rule below; otherwise a block tile by its code (a tile that is not built: an error).
static int swiglu_tile_entry(const void* A, int lda, const void* W, int ldw, void* C, int ldc, int M, int N, int K,
                             int dual_off, int tile, GateLaw law, hipStream_t stream);

extern "C" int cisr_gemm_bf16_swiglu_tile(const void* A, int lda, const void* W, int ldw, void* C, int ldc, int M, int N, int K,
                                          int dual_off, int tile, hipStream_t stream) {
    return swiglu_tile_entry(A, lda, W, ldw, C, ldc, M, N, K, dual_off, tile, GateLaw{}, stream);
}

// The same with the gated activation's law given: see GateLaw.
extern "C" int cisr_gemm_bf16_gated(const void* A, int lda, const void* W, int ldw, void* C, int ldc, int M, int N, int K,
                                    int dual_off, float limit, float slope, float shift, hipStream_t stream) {
    return swiglu_tile_entry(A, lda, W, ldw, C, ldc, M, N, K, dual_off, 0, GateLaw{limit, slope, shift}, stream);
}

static int swiglu_tile_entry(const void* A, int lda, const void* W, int ldw, void* C, int ldc, int M, int N, int K,
                             int dual_off, int tile, GateLaw law, hipStream_t stream) {
    if (M <= 0 || N <= 0) return 0;
    if (K <= 0 || K % 8 || lda % 8 || ldw % 8 || ((uintptr_t)A) % 16 || ((uintptr_t)W) % 16 || dual_off < N)
        return (int)hipErrorInvalidValue;
    const bf16_t* a = (const bf16_t*)A; const bf16_t* w = (const bf16_t*)W;
    auto blocks = [&](int bm, int bn) { return (long long)((M + bm - 1) / bm) * ((2 * N + bn - 1) / bn); };
    if (tile == 0) {
        // As below, over the columns of both halves: 300 rows, 1,536 outputs, K 576: 32 x 64 (480 blocks) 6.8 us, 64 x 64 (240) 6.1,
        // 128 x 64 7.8; 300 rows, 3,072 outputs: 64 x 64 (480 blocks, two a unit) 9.5, 128 x 64 (288) 12.4, 128 x 128 12.8.  With one
        // round of 128 x 128, 128 x 64 up to K 576 (1,000 rows, 1,536 outputs: 12.0 against 12.4), 128 x 128 from there (1,000 rows,
        // 2,048 outputs, K 1,024: 17.5 against 17.1; 500 rows, 4,096 outputs, K 2,048: 32.8 against 29.5).  With a second round that
        // is mostly idle 128 x 64 (1,500 rows, 2,048 outputs, K 1,024, 384 blocks: 24.1 against 25.6), from 400 blocks on 128 x 128
        // (1,777 rows, 448 blocks: 29.8 against 26.0; 4,000 rows of 1,536 outputs, K 576: 29.0 against 26.3).
        if (blocks(32, 64) <= 256) tile = 122;
        else if (blocks(64, 64) <= 256) tile = 222;
        else if (blocks(128, 64) <= 256) tile = 422;
        else if (blocks(64, 64) <= 512) tile = 222;
        else if (blocks(128, 128) <= 256) tile = K <= 576 ? 422 : 442;
        else tile = blocks(128, 128) < 400 ? 422 : 442;
    }
#define SWIGLU_TILE(CODE, TM, TN, BK, WM, PF) \
    case CODE: return launch_bf16_swiglu<TM, TN, BK, WM, PF>(a, lda, w, ldw, (bf16_t*)C, ldc, M, N, K, dual_off, law, stream);
    // (128 x 128: 32 of the inner size a turn keeps two blocks on a unit; 2,000 rows, 4,096 outputs, K 2,048: 64 deep 94 us, 32 deep 87)
    switch (tile) {
        SWIGLU_TILE(122, 1, 2, 64, 2, 3) SWIGLU_TILE(222, 1, 2, 128, 4, 2) SWIGLU_TILE(422, 2, 2, 64, 4, 2) SWIGLU_TILE(442, 2, 4, 32, 4, 4)
    }
#undef SWIGLU_TILE
    return (int)hipErrorInvalidValue;
}

extern "C" int cisr_gemm_bf16_swiglu(const void* A, int lda, const void* W, int ldw, void* C, int ldc, int M, int N, int K,
                                     int dual_off, hipStream_t stream) {
    return cisr_gemm_bf16_swiglu_tile(A, lda, W, ldw, C, ldc, M, N, K, dual_off, 0, stream);
}

// The codes name a block tile: rows / 32, columns / 32, and a 2 (112: 32 x 32, 422: 128 x 64).
// Tile choice: the smallest that needs no more blocks than there are compute units: a block alone on its unit takes the longer the
// larger its tile, and a second round costs more than a larger tile does.  1,741 rows, us: 576 columns (K 1,536) 32 x 32 12.4, 64 x
// 32 10.4, 64 x 64 (252 blocks) 8.8, 128 x 64 12.8; 960 columns (K 576) 64 x 64 (420 blocks) 9.8, 128 x 64 (210) 7.4, 128 x 128 10.3.
// 300 rows x 960: 32 x 32 (300 blocks) 5.1, 64 x 32 (150) 4.6, 64 x 64 5.4.  Up to 32 rows a tile has 32 of them (32 x 12,000, K
// 1,024: 32 x 64 6.6, 64 x 64 6.8).
// Where 128 x 64 needs more than one round, us of 64 x 64 / 128 x 64 / 128 x 128:
//   64 x 64 twice a unit at once (its LDS leaves room for two): 1,300 x 1,536 (504, 264 and 132 blocks), K 576 11.9 / 12.5 / 12.3, K
//   1,536 18.7 / 24.3 / 21.5; 1,500 rows (576 of 64 x 64) are too many for that: 25.8 / 24.0 / 21.6;
//   one round of 128 x 128: the same up to K 576 (2,000 x 2,048, 512 and 256 blocks, K 512: 18.3 / 12.7 / 13.1; 1,777 x 1,536, 336
//   and 168, K 576: 16.1 / 12.9 / 12.8), above it the larger tile's fewer bytes (2,000 x 2,048, K 1,024 27.0 / 20.5 / 19.8, K 2,048
//   41.0 / 31.8 / 29.0; 1,777 x 1,536, K 1,536 25.9 / 24.0 / 22.3);
//   more than one: 128 x 64 up to K 1,536 (4,000 x 2,048, 1,024 and 512 blocks, K 512: 24.2 / 26.0; 6,000 x 1,536, 1,128 and 564, K
//   1,536: 54.1 / 61.2; 8,000 x 1,536: 66.1 / 64.3) and where the second round of 128 x 128 is mostly idle (7,936 x 576, K 1,536,
//   558 and 310 blocks: 32.2 / 36.5), else 128 x 128 (8,000 x 1,024, K 2,048, 1,008 and 504: 56.4 / 54.1).
static int pick_tile(int M, int N, int K, int heads) {
    auto blocks = [&](int bm, int bn) { return (long long)((M + bm - 1) / bm) * ((N + bn - 1) / bn) * heads; };
    if (blocks(32, 32) <= 256) return 112;
    if (M <= 32) return 122;
    if (blocks(64, 32) <= 256) return 212;
    if (blocks(64, 64) <= 256) return 222;
    if (blocks(128, 64) <= 256) return 422;
    if (blocks(64, 64) <= 512) return 222;
    if (blocks(128, 128) <= 256) return K <= 576 ? 422 : 442;
    return K <= 1536 || blocks(128, 128) < 400 ? 422 : 442;
}

static int launch_tile(int tile, const void* A, int lda, const void* W, int ldw, void* C, int ldc, const float* R, int ldr, int M, int N,
                       int K, int out_dtype, hipStream_t stream, HeadBatch batch = {}, int heads = 1) {
    const bf16_t* a = (const bf16_t*)A; const bf16_t* w = (const bf16_t*)W;
#define GEMM_TILE(CODE, TM, TN, BK, WM, PF) \
    case CODE: return launch_bf16<TM, TN, BK, WM, PF>(a, lda, w, ldw, C, ldc, R, ldr, M, N, K, out_dtype, stream, batch, heads);
    switch (tile) {
        GEMM_TILE(112, 1, 1, 128, 2, 3) GEMM_TILE(122, 1, 2, 64, 2, 3) GEMM_TILE(212, 1, 1, 128, 4, 2) GEMM_TILE(222, 1, 2, 128, 4, 2)
        GEMM_TILE(422, 2, 2, 64, 4, 2) GEMM_TILE(442, 2, 4, 64, 4, 2)
    }
#undef GEMM_TILE
    return (int)hipErrorInvalidValue;
}

// `tile`: 0 picks by the rule above; otherwise a block tile by its code (a tile that is not built: an error).
extern "C" int cisr_gemm_bf16_tile(const void* A, int lda, const void* W, int ldw, void* C, int ldc, const float* R,
                                   int ldr, int M, int N, int K, int out_dtype, int tile, hipStream_t stream) {
    if (M <= 0 || N <= 0) return 0;
    if (K <= 0 || (R && out_dtype != DT_F32)) return (int)hipErrorInvalidValue;
    return launch_tile(tile ? tile : pick_tile(M, N, K, 1), A, lda, W, ldw, C, ldc, R, ldr, M, N, K, out_dtype, stream);
}

// A product a head in one launch: C[m, h * c_head + n] = sum_k A[m, h * a_head + k] W[h][n][k] (W [heads, N, K] contiguous),
// times sigmoid(gate[m * ldg + h]) where `gate` is given.  bf16 operands, bf16 or float results.
extern "C" int cisr_gemm_bf16_heads(const void* A, int lda, int a_head, const void* W, void* C, int ldc, int c_head,
                                    const float* gate, int ldg, int M, int N, int K, int heads, int out_dtype, hipStream_t stream) {
    if (M <= 0 || N <= 0 || heads <= 0) return 0;
    if (K <= 0) return (int)hipErrorInvalidValue;
    const HeadBatch batch{a_head, (long long)N * K, c_head, gate, ldg, ACT_NONE};
    return launch_tile(pick_tile(M, N, K, heads), A, lda, W, K, C, ldc, nullptr, 0, M, N, K, out_dtype, stream, batch, heads);
}

// C = act(A . W^T) with an ungated activation (ACT_GELU, ACT_GELU_TANH, ACT_RELU2) as the epilogue; the tile is picked as for the
// plain product.
extern "C" int cisr_gemm_bf16_act(const void* A, int lda, const void* W, int ldw, void* C, int ldc, int M, int N, int K,
                                  int out_dtype, int act, hipStream_t stream) {
    if (M <= 0 || N <= 0) return 0;
    if (K <= 0 || act < ACT_GELU || act > ACT_RELU2) return (int)hipErrorInvalidValue;
    const HeadBatch batch{0, 0, 0, nullptr, 0, act};
    return launch_tile(pick_tile(M, N, K, 1), A, lda, W, ldw, C, ldc, nullptr, 0, M, N, K, out_dtype, stream, batch);
}

extern "C" int cisr_gemm_bf16(const void* A, int lda, const void* W, int ldw, void* C, int ldc, const float* R,
                              int ldr, int M, int N, int K, int out_dtype, hipStream_t stream) {
    return cisr_gemm_bf16_tile(A, lda, W, ldw, C, ldc, R, ldr, M, N, K, out_dtype, 0, stream);
}
