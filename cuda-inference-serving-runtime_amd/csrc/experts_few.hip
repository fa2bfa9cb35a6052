// The experts' products of steps that bring an expert few rows (decoding tens of requests): the same tiles of places as
// csrc/experts.hip, bound by the bytes of the experts' matrices.
//
// A wave makes 16 columns of one expert (GATED: the gates and the ups of 16 outputs) for all rows of its tile, alone: DEPTH
// 64-deep units of the matrix are in flight, nothing waits for another wave.  Loads are whole 128-byte lines (a load: eight
// rows of the matrix, eight neighbouring lanes a row); the lanes that the matrix instruction wants them in get them through
// LDS, in slots of the wave's own.  (Loaded in the instruction's layout, sixteen rows in neighbouring lanes, the cache serves
// a load at a quarter of its rate.)  Rows past the tile's last pair are not loaded: 16, 32 or 64 rows are multiplied as the
// tile needs.  A sum is one chain of matrix instructions over K from `first_unit` on, as in the other kernel: the same bits.
//
// Measured on an MI355X, 16 experts, 48 pairs: matrices of 4096 x 2048 in 42 us (6.0 TB/s; 54 when every sum began at the first
// unit, 52 in tiles of 64 x 128), of 2048 x 4096 in 42 (67 and 68).
#include "common.h"

#define EXF_TILE 64
#define EXF_WAVES 1                     // (blocks of four waves leave some compute units with half as many again as others: 58 us instead of 50)

typedef __attribute__((ext_vector_type(8))) __bf16 exf_bf16x8;
typedef __attribute__((ext_vector_type(4))) float exf_f32x4;
typedef __attribute__((ext_vector_type(4))) uint32_t exf_u32x4;

struct FewArgs {
    const bf16_t* A; int lda;
    const bf16_t* W;                    // [experts][N or 2 N][K]
    const int* tile_expert; const int* pair_of_pos;
    int gather_div, scatter;            // as in cisr_experts_gemm
    void* C; int ldc;
    int N, K;                           // columns of C, inner size
    GateLaw law;
};

enum { FEW_PLAIN = 0, FEW_RELU2 = 1, FEW_GATED = 2 };

__device__ __forceinline__ void exf_wave_order() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// MT sixteens of rows.  Element (row, 16-byte chunk c) of a 16 x 64 piece waits in slot row * 8 + (c ^ row % 8).
template <int MT, int DEPTH, typename TC, int ACT>
__device__ __forceinline__ void few_tile(const FewArgs& p, int e, int tile, int places, exf_u32x4* lds) {
    constexpr int NT = ACT == FEW_GATED ? 2 : 1, PIECE = 128;         // 16-byte words of a 16 x 64 piece
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE), lane = threadIdx.x % WAVE, r = lane % 16, g = lane / 16;
    const int K = p.K, units = (K + 63) / 64;
    const int lrow = lane / 8, chunk = lane % 8;
    const int n0 = (blockIdx.y * EXF_WAVES + wave) * 16;
    if (n0 >= p.N) return;
    const int begin = first_unit(e, n0 / (ACT == FEW_GATED ? 64 : 128), units);
    auto place_of = [&](int u) { const int at = u + begin; return at < units ? at : at - units; };
    const bf16_t* We = p.W + (size_t)e * NT * p.N * K;
    const bf16_t* w_row[NT][2];
#pragma unroll
    for (int j = 0; j < NT; ++j)
#pragma unroll
        for (int h = 0; h < 2; ++h) w_row[j][h] = We + (size_t)(j * p.N + min(n0 + 8 * h + lrow, p.N - 1)) * K;
    const bf16_t* a_row[MT][2];
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const int pos = tile * EXF_TILE + min(16 * i + 8 * h + lrow, places - 1);
            const int pair = max(p.pair_of_pos[pos], 0);
            a_row[i][h] = p.A + (size_t)(p.gather_div > 0 ? pair / p.gather_div : pos) * p.lda;
        }
    exf_u32x4* mine = lds + wave * (MT + NT) * PIECE;
    exf_u32x4* put = mine + lrow * 8 + (chunk ^ lrow);
    exf_f32x4 acc[MT][NT];
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j) acc[i][j] = (exf_f32x4){0.f, 0.f, 0.f, 0.f};
    exf_u32x4 fw[DEPTH][NT][2], fa[DEPTH][MT][2];
    auto ask = [&](int d, int u) {
        const int k = min(place_of(min(u, units - 1)) * 64 + 8 * chunk, K - 8);
#pragma unroll
        for (int j = 0; j < NT; ++j)
#pragma unroll
            for (int h = 0; h < 2; ++h) fw[d][j][h] = __builtin_nontemporal_load((const exf_u32x4*)(w_row[j][h] + k));
#pragma unroll
        for (int i = 0; i < MT; ++i)
#pragma unroll
            for (int h = 0; h < 2; ++h) fa[d][i][h] = *(const exf_u32x4*)(a_row[i][h] + k);
    };
    auto use = [&](int d, int u) {
        const int k0 = place_of(u) * 64;
        const bool tail = k0 + 64 > K;                                // (uniform: K's last, partly filled unit)
        const uint32_t keep = !tail || k0 + 8 * chunk < K ? 0xffffffffu : 0u;
#pragma unroll
        for (int j = 0; j < NT; ++j)
#pragma unroll
            for (int h = 0; h < 2; ++h) put[j * PIECE + 64 * h] = fw[d][j][h] & keep;
#pragma unroll
        for (int i = 0; i < MT; ++i)
#pragma unroll
            for (int h = 0; h < 2; ++h) put[(NT + i) * PIECE + 64 * h] = fa[d][i][h] & keep;
        exf_wave_order();
#pragma unroll
        for (int ks = 0; ks < 2; ++ks) {
            const int slot = r * 8 + ((4 * ks + g) ^ (r % 8));
            exf_bf16x8 xw[NT], xa[MT];
#pragma unroll
            for (int j = 0; j < NT; ++j) xw[j] = __builtin_bit_cast(exf_bf16x8, mine[j * PIECE + slot]);
#pragma unroll
            for (int i = 0; i < MT; ++i) xa[i] = __builtin_bit_cast(exf_bf16x8, mine[(NT + i) * PIECE + slot]);
#pragma unroll
            for (int i = 0; i < MT; ++i)
#pragma unroll
                for (int j = 0; j < NT; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(xa[i], xw[j], acc[i][j], 0, 0, 0);
        }
        exf_wave_order();
    };
#pragma unroll
    for (int d = 0; d < DEPTH; ++d) {
        ask(d, d);
        __builtin_amdgcn_sched_barrier(0);
    }
    int turn = 0;
    for (; turn + DEPTH < units; turn += DEPTH)
#pragma unroll
        for (int d = 0; d < DEPTH; ++d) {
            use(d, turn + d);
            __builtin_amdgcn_sched_barrier(0);
            ask(d, turn + d + DEPTH);
            __builtin_amdgcn_sched_barrier(0);
        }
#pragma unroll
    for (int d = 0; d < DEPTH; ++d)
        if (turn + d < units) use(d, turn + d);                       // (uniform)
    const int n = n0 + r;
    if (n >= p.N) return;
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int x = 0; x < 4; ++x) {
            const int place = 16 * i + 4 * g + x;
            if (place >= places) continue;
            const int pos = tile * EXF_TILE + place;
            float v = acc[i][0][x];
            if (ACT == FEW_RELU2) { v = fmaxf(v, 0.f); v *= v; }
            if (ACT == FEW_GATED) v = gated_activation<TC>(v, acc[i][NT - 1][x], p.law);
            store_f32((TC*)p.C + (size_t)(p.scatter ? p.pair_of_pos[pos] : pos) * p.ldc + n, v);
        }
}

template <typename TC, int ACT>
__global__ void __launch_bounds__(EXF_WAVES * WAVE)
experts_few_kernel(FewArgs p) {
    __shared__ exf_u32x4 lds[EXF_WAVES * (ACT == FEW_GATED ? 6 : 5) * 128];   // (at most so many pieces a wave: 12 or 10 KB, sixteen blocks a compute unit)
    const int tile = blockIdx.x, e = p.tile_expert[tile];
    if (e < 0) return;
    // a tile's pairs come first, padding behind them
    const int places = __popcll(__ballot(p.pair_of_pos[tile * EXF_TILE + threadIdx.x % WAVE] >= 0));
    if (places <= 0) return;
    if (places <= 16) few_tile<1, 4, TC, ACT>(p, e, tile, places, lds);
    else if (places <= 32) few_tile<2, ACT == FEW_GATED ? 3 : 4, TC, ACT>(p, e, tile, places, lds);
    else few_tile<4, 2, TC, ACT>(p, e, tile, places, lds);
}

// The product of cisr_experts_gemm (act 0 or 1: relu(z)^2) and cisr_experts_gemm_gated (act 2: W [experts, 2 N, K], C by
// place, bf16) for bf16 operands with K % 8 == 0 and 16-byte aligned rows.
extern "C" int cisr_experts_few(const void* A, int lda, const void* W, const int* tile_expert, const int* pair_of_pos, int gather_div,
                                int scatter, void* C, int ldc, int max_tiles, int N, int K, int act, int out_dtype, float limit,
                                float slope, float shift, hipStream_t stream) {
    if (max_tiles <= 0 || N <= 0) return 0;
    constexpr int columns = 16 * EXF_WAVES;
    if (K < 8 || K % 8 || lda % 8 || ((uintptr_t)A) % 16 || ((uintptr_t)W) % 16 || act < 0 || act > 2 || (N + columns - 1) / columns > 65535 ||
        (act == FEW_GATED && (out_dtype != DT_BF16 || scatter)))
        return (int)hipErrorInvalidValue;
    const FewArgs p{(const bf16_t*)A, lda, (const bf16_t*)W, tile_expert, pair_of_pos, gather_div, scatter, C, ldc, N, K, GateLaw{limit, slope, shift}};
    const dim3 grid(max_tiles, (N + columns - 1) / columns);
#define FEW(TC, ACT) experts_few_kernel<TC, ACT><<<grid, EXF_WAVES * WAVE, 0, stream>>>(p)
    if (act == FEW_GATED) FEW(bf16_t, FEW_GATED);
    else if (out_dtype == DT_F32) { if (act) FEW(float, FEW_RELU2); else FEW(float, FEW_PLAIN); }
    else { if (act) FEW(bf16_t, FEW_RELU2); else FEW(bf16_t, FEW_PLAIN); }
#undef FEW
    return CISR_LAUNCH_CHECK();
}
