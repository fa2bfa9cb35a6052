// Arguments of the ring products (gemm_ring.inc) and the entry points of the units that hold their tiles (so that the tiles
// compile in parallel).
#pragma once
#include "common.h"

enum { RING_STORE = 0, RING_GATED = 1, RING_FLOAT = 2, RING_ROPE = 3, RING_GATED_NORMED = 4, RING_ROPE_NORMED = 5, RING_FLOAT_NORMED = 6 };

struct RingArgs {
    const bf16_t* A; int lda;
    const bf16_t* W; int ldw;
    void* C; int ldc;                  // bf16 (RING_STORE, RING_GATED) or float (RING_FLOAT)
    const float* R; int ldr;           // RING_FLOAT with one slice: a residual, which may be C itself; else null
    int M, N, K;
    int dual_off; GateLaw law;         // RING_GATED: W = [gate; up], `dual_off` rows apart; the activation's law
    int act;                           // RING_STORE: an ungated activation (ACT_*) before the store
    int slices;                        // RING_FLOAT: parts of the inner size; slice s writes C + s M ldc
    // RING_ROPE: W = [Wq; Wk; Wv] (or Wq alone, kv_heads 0); C: q, rows of ldc; k and v go into the pages at `slots`
    const int* positions; const int* slots; const float* cos_tab; const float* sin_tab;
    bf16_t* kcache; bf16_t* vcache; int heads, kv_heads, dim, page_size, max_pos;
    // An RMSNorm between two ring products, of which no kernel is made.  RING_FLOAT_NORMED (R given, one slice): rows `scaled` (of ldy) = bf16(C norm_w),
    // sums[i * M + m] = the squares of C's row m summed over the columns of the i-th tile (`parts` of them).  RING_GATED_NORMED and
    // RING_ROPE_NORMED: as the modes without, A is such rows and the factor that the sums give finishes the results
    bf16_t* scaled; int ldy; const float* norm_w; float* sums; int parts; float inv_k, eps;
};

// one function per unit: 0 or a HIP error; hipErrorInvalidValue: the unit does not hold this tile (nothing is launched)
int cisr_ring_launch_a(const RingArgs& a, int tile, int mode, hipStream_t stream);
int cisr_ring_launch_b(const RingArgs& a, int tile, int mode, hipStream_t stream);
int cisr_ring_launch_c(const RingArgs& a, int tile, int mode, hipStream_t stream);
int cisr_ring_launch_d(const RingArgs& a, int tile, int mode, hipStream_t stream);
