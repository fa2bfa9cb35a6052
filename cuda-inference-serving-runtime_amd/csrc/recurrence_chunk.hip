// Recurrences over prompt portions, chunk by chunk on the matrix cores (float operands, v_mfma_f32_16x16x4_f32): the gated
// delta rule (DELTA) and the linear scan S <- diag(g) S + k v^T, o = S^T q, each with a decay a key channel (VEC) or one a
// head.  A segment's rows in chunks of 16; with D(t, i) the product of a chunk's decays g_(i+1) .. g_t, channel by channel,
// D(t) that of g_0 .. g_t, and S0 the state at the chunk's start:
//
//   DELTA:  A[t, i] = beta_t sum_r k_t k_i D(t, i), i < t,  M = (I + A)^-1 diag(beta),  Kg_t = D(t) k_t
//           U = M (V - Kg S0)                                 (the rows' writes u_t)
//   else:   U = V, times the rows' step sizes if there are any
//   P[t, i] = sum_r q_t k_i D(t, i), i <= t
//   o_t = (D(t) q_t)^T S0 + sum_i P[t, i] u_i
//   S  <- D(15) S0 + sum_i (D(15, i) k_i) u_i^T
//
// Every product of decays is made by multiplying decays along the rows: no quotients and no differences of logarithms, so a
// channel whose decays vanish within a chunk costs neither range nor precision.  A first kernel makes, chunk by chunk and
// all side by side, what does not need the state: M V, M Kg, D q, P, D(15, i) k and D(15); a second walks a segment's chunks
// in order, a block a (head, 16 columns of S): its waves own the rows of S in turn, two products with S0 (one without DELTA),
// one meeting through LDS, one product into S.  Rows behind a segment's end count as k = q = v = 0 with decays of one.  A row
// does not see the rows behind it, whatever they hold: where a write is not finite, scores and writes are summed row by row.
// The operands lie in memory as the walk's lanes want them, 16 bytes a lane side by side: read in rows of the chunk instead,
// each load of the walk touches four times the lines.
// Measured on an MI355X, us of both kernels (in brackets the scans that walk row by row): 2,048 rows of one request, the delta
// rule with 32 heads of 128 x 128 and a decay a channel 207, with a decay a head 176 (840); gated linear attention, 8 heads
// of 128 x 256, 111 (290), three requests of 782 rows 99 (361); state-space duality, 64 heads of 128 x 64, 170 (495) and
// 224 (477).  The walk's bound is its chain a chunk (0.7 to 1 us), with many heads what the two kernels write and read in
// between (30 KB a chunk and head at 128 x 64).
//
// Sums: the scans round the state once a row, the walk twice a chunk (what its rows write is summed apart from it); products with
// the state are a sum a tile of sixteen rows; scores and products of decays are made in double where that is cheap.  Relative
// error of 1,500 rows' results against 64 bits, row by row / so: delta rule, 8 heads of 128 x 128, decays from 0.999 to 1
// 3.2e-7 / 1.9e-7, from 0.8 to 1 1.13e-7 / 1.02e-7; gated linear attention, 4 heads of 128 x 256, 5.1e-7 / 2.3e-7 and 9.7e-8 /
// 8.6e-8; state-space duality, 16 heads of 128 x 64, 5.1e-7 / 2.2e-7 and 1.00e-7 / 8.2e-8.
#include "common.h"
#include <type_traits>

#define CHUNK 16

typedef __attribute__((ext_vector_type(4))) float f32x4_t;
typedef __attribute__((ext_vector_type(4))) double f64x4_t;

struct ChunkArgs {
    const float* q; int ldq;          // q[t * ldq + (head / share) * R + r]
    const float* k; int ldk;
    const float* v; int ldv;          // v[t * ldv + head * C + c]
    const float* g; int ldg;          // VEC: g[t * ldg + head * R + r]; else g[t * ldg + head]
    const float* b; int ldb;          // DELTA: b[t * ldb + head], beta = sigmoid(b); else null or the step size b[t * ldb + head] that multiplies v
    float* out; int ldo;
    float* state; long long slot_stride;
    const int* seg_start; const int* state_slots;
    int R, C, share, heads, segments;
    float q_scale;
    int Rp, Cp;                       // R and C rounded up to 16
    int slot0, slots;                 // this launch's chunk slots (a chunk's slot: seg_start / 16 + segment + its number)
    float* work;                      // [slots][heads][chunk_floats]
};

// A (chunk, head) in `work`, in floats: M Kg (DELTA only) and D q as [Rp / 16] tiles of 16 rows x 16 channels, D(15, i) k as
// tiles of 16 channels x 16 rows, M V as [Cp / 16] tiles of 16 columns x 16 rows, P as one tile, D(15) [Rp].  In a tile, float
// ((b / 4) * 16 + a) * 4 + b % 4 is element (a, b): what lane 16 (b / 4) + a of the walk takes as its 16 bytes.
template <bool DELTA>
struct ChunkLayout {
    int q, kd, u, pr, g, floats;
    __host__ __device__ __forceinline__ ChunkLayout(int Rp, int Cp) {
        q = DELTA ? CHUNK * Rp : 0;
        kd = q + CHUNK * Rp;
        u = kd + CHUNK * Rp;
        pr = u + CHUNK * Cp;
        g = pr + CHUNK * CHUNK;
        floats = g + Rp;
    }
};

// The segment whose chunk slots hold `slot` (segments without rows own a slot without a chunk).
__device__ __forceinline__ int segment_of_slot(const int* seg_start, int segments, int slot) {
    int lo = 0, hi = segments - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) / 2;
        if (seg_start[mid] / CHUNK + mid <= slot) lo = mid; else hi = mid - 1;
    }
    return lo;
}

template <int CTRL>
__device__ __forceinline__ float lanes_moved(float x) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), CTRL, 0xF, 0xF, false));
}

template <int CTRL>
__device__ __forceinline__ double lanes_moved(double x) {
    const uint64_t b = __builtin_bit_cast(uint64_t, x);
    const uint32_t lo = __builtin_amdgcn_update_dpp(0, (int)(uint32_t)b, CTRL, 0xF, 0xF, false);
    const uint32_t hi = __builtin_amdgcn_update_dpp(0, (int)(uint32_t)(b >> 32), CTRL, 0xF, 0xF, false);
    return __builtin_bit_cast(double, (uint64_t)hi << 32 | lo);
}

// the sum over the 16 lanes of an aligned row, in each of them
template <typename T>
__device__ __forceinline__ T row_sum(T x) {
    x += lanes_moved<0xB1>(x);                   // quad_perm [1, 0, 3, 2]
    x += lanes_moved<0x4E>(x);                   // quad_perm [2, 3, 0, 1]
    x += lanes_moved<0x141>(x);                  // row_half_mirror
    x += lanes_moved<0x140>(x);                  // row_mirror
    return x;
}

// The row of its chunk that stands in slot s of the walk's operands.  A matrix instruction of the walk takes slots i, 4 + i, 8 + i
// and 12 + i (float i of the four that a lane holds of its result), which are rows 4 i .. 4 i + 3: sums over a chunk's
// rows run in the order of time, so that under strong decays the large terms come last and are rounded few times.
__host__ __device__ constexpr int row_of_slot(int s) { return 4 * (s % 4) + s / 4; }

// Scores, products of decays and the inverse of I + A are double and rounded once (with a decay a head the scores are Gram matrices,
// on v_mfma_f64_16x16x4_f64): what is rounded here is an error that all columns of a chunk share, which row by row no two of
// them do.  (The delta rule with a decay a channel makes them in float: two scores a pair of rows, each with products of
// decays of its own, are most of its work.)
template <bool DELTA, bool VEC>
__global__ void __launch_bounds__(256, 4) channel_chunk_kernel(ChunkArgs p) {
    extern __shared__ __attribute__((aligned(16))) float lds[];
    using Wide = std::conditional_t<VEC && DELTA, float, double>;
    __shared__ Wide sA[DELTA ? CHUNK : 1][CHUNK + 1];
    __shared__ double sD[CHUNK], sE[CHUNK], sG[VEC ? 1 : CHUNK];
    __shared__ double gram[VEC ? 1 : 4][VEC ? 1 : CHUNK * CHUNK];
    __shared__ __attribute__((aligned(16))) float sM[DELTA ? CHUNK : 1][CHUNK];
    __shared__ float sBeta[CHUNK];
    const int slot = p.slot0 + blockIdx.y, head = blockIdx.x, tid = threadIdx.x;
    const int seg = segment_of_slot(p.seg_start, p.segments, slot);
    const int t0 = p.seg_start[seg] + (slot - p.seg_start[seg] / CHUNK - seg) * CHUNK, t1 = p.seg_start[seg + 1];
    if (t0 >= t1 || t0 < p.seg_start[seg]) return;
    const int n = min(CHUNK, t1 - t0), R = p.R, C = p.C, Rp = p.Rp, RS = Rp + 4;
    float* sk = lds;
    float* sq = sk + CHUNK * RS;
    float* sg = sq + CHUNK * RS;
    const float* kh = p.k + (size_t)t0 * p.ldk + (size_t)(head / p.share) * R;
    const float* qh = p.q + (size_t)t0 * p.ldq + (size_t)(head / p.share) * R;
    const float* gh = p.g + (size_t)t0 * p.ldg + (VEC ? (size_t)head * R : (size_t)head);
    for (int idx = tid; idx < CHUNK * Rp; idx += 256) {
        const int i = idx / Rp, r = idx % Rp, tt = min(i, n - 1), rr = min(r, R - 1);
        const bool in = r < R && i < n;
        const float k = kh[tt * p.ldk + rr], q = qh[tt * p.ldq + rr];
        sk[i * RS + r] = in ? k : 0.f;
        sq[i * RS + r] = in ? q * p.q_scale : 0.f;
        if (VEC) {
            const float g = gh[tt * p.ldg + rr];
            sg[i * RS + r] = in ? g : 1.f;
        }
    }
    if (DELTA && tid < CHUNK) sBeta[tid] = tid < n ? 1.0f / (1.0f + expf(-p.b[(size_t)(t0 + tid) * p.ldb + head])) : 0.f;
    if (!DELTA && tid < CHUNK) sBeta[tid] = tid < n && p.b ? p.b[(size_t)(t0 + tid) * p.ldb + head] : 1.f;     // (the step sizes)
    if (!VEC && tid < CHUNK) sG[tid] = tid < n ? (double)gh[tid * p.ldg] : 1.0;
    __syncthreads();
    const ChunkLayout<DELTA> at(Rp, p.Cp);
    float* work = p.work + ((size_t)blockIdx.y * p.heads + head) * at.floats;
    float* wP = work + at.pr;
    if constexpr (VEC) {
        // column i of A and P: sixteen neighbouring threads, each with every sixteenth run of four channels, carry k_i down the
        // rows behind i (times their decays) and meet
        const int i = tid / 16, part = tid % 16;
        f32x4_t x[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) x[j] = 64 * j + 4 * part < Rp ? *(const f32x4_t*)(sk + i * RS + 64 * j + 4 * part) : (f32x4_t){0.f, 0.f, 0.f, 0.f};
        for (int t = 0; t < CHUNK; ++t) {
            Wide a = 0, b = 0;
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const int r = 64 * j + 4 * part;
                if (64 * j >= Rp) break;                           // (uniform)
                if (r >= Rp || t < i) continue;
                const f32x4_t k = *(const f32x4_t*)(sk + t * RS + r), q = *(const f32x4_t*)(sq + t * RS + r);
                if (t > i) x[j] *= *(const f32x4_t*)(sg + t * RS + r);
                if constexpr (DELTA) {
                    a += (x[j][0] * k[0] + x[j][1] * k[1]) + (x[j][2] * k[2] + x[j][3] * k[3]);
                    b += (x[j][0] * q[0] + x[j][1] * q[1]) + (x[j][2] * q[2] + x[j][3] * q[3]);
                } else {
#pragma unroll
                    for (int e = 0; e < 4; ++e) b += (double)x[j][e] * q[e];
                }
            }
            if (DELTA) a = row_sum(a);
            b = row_sum(b);
            if (part == t) {
                if (DELTA) sA[t][i] = sBeta[t] * a;                // (only i < t is read)
                const int row = row_of_slot(t), col = row_of_slot(i);          // (its own inverse)
                wP[(col / 4 * 16 + row) * 4 + col % 4] = (float)b; // (0 for i > t)
            }
        }
    } else {
        // q k^T and, for A, k k^T, a part of the channels a wave
        const int wave = __builtin_amdgcn_readfirstlane(tid / WAVE), lane = tid % WAVE;
        const bool score = !DELTA || wave < 2;
        const int parts = DELTA ? 2 : 4, part = wave % parts;
        const float* left = (score ? sq : sk) + lane % 16 * RS + lane / 16;
        const float* right = sk + lane % 16 * RS + lane / 16;
        f64x4_t acc = {0.0, 0.0, 0.0, 0.0};
#pragma unroll 4
        for (int r = part * (Rp / parts); r < (part + 1) * (Rp / parts); r += 4)
            acc = __builtin_amdgcn_mfma_f64_16x16x4f64((double)left[r], (double)right[r], acc, 0, 0, 0);
#pragma unroll
        for (int e = 0; e < 4; ++e) gram[wave][(4 * e + lane / 16) * CHUNK + lane % 16] = acc[e];      // (element e: row 4 e + lane / 16)
        __syncthreads();
        const int t = tid / CHUNK, i = tid % CHUNK;
        double d = 1.0, ahead = 1.0, so_far = 1.0;
#pragma unroll
        for (int u = 0; u < CHUNK; ++u) {
            const double g = sG[u];
            d *= u > i && u <= t ? g : 1.0;
            so_far *= u <= i ? g : 1.0;
            ahead *= u > i ? g : 1.0;
        }
        if (t == 0) { sD[i] = so_far; sE[i] = ahead; }
        const double b = DELTA ? gram[0][tid] + gram[1][tid] : (gram[0][tid] + gram[1][tid]) + (gram[2][tid] + gram[3][tid]);
        if (DELTA) sA[t][i] = sBeta[t] * (d * (gram[2][tid] + gram[3][tid]));              // (only i < t is read)
        const int row = row_of_slot(t), col = row_of_slot(i);                                      // (its own inverse)
        wP[(col / 4 * 16 + row) * 4 + col % 4] = i <= t ? (float)(b * d) : 0.f;
    }
    __syncthreads();
    // column j of the inverse of the unit triangle I + A by forward substitution, times beta_j
    if (DELTA && tid < CHUNK) {
        Wide x[CHUNK];
#pragma unroll
        for (int t = 0; t < CHUNK; ++t) x[t] = t == tid ? 1 : 0;
#pragma unroll
        for (int i = 0; i < CHUNK; ++i) {
#pragma unroll
            for (int t = i + 1; t < CHUNK; ++t) x[t] -= sA[t][i] * x[i];
            __builtin_amdgcn_sched_barrier(0);                     // (the columns' operands are not asked for all at once: registers)
        }
#pragma unroll
        for (int t = 0; t < CHUNK; ++t) sM[t][tid] = (float)(x[t] * sBeta[tid]);
    }
    if (DELTA) __syncthreads();
    // a thread a channel (M Kg and the other operands over the state's rows, which take the place of k, q and the decays) or a
    // column of v (M V)
    for (int idx = tid; idx < Rp + p.Cp; idx += 256) {
        const bool key = idx < Rp;
        const int c = key ? idx : idx - Rp;
        float x[CHUNK];
        if (key) {
            float kd[CHUNK];
            Wide d = 1;
#pragma unroll
            for (int i = CHUNK - 1; i >= 0; --i) {
                if (!VEC) d = sE[i];
                kd[i] = (float)(sk[i * RS + c] * d);
                if (VEC) d *= sg[i * RS + c];
            }
            d = 1;
#pragma unroll
            for (int i = 0; i < CHUNK; ++i) {
                if (VEC) d *= sg[i * RS + c];
                else d = sD[i];
                if (DELTA) x[i] = (float)(sk[i * RS + c] * d);
                sq[i * RS + c] = (float)(sq[i * RS + c] * d);
            }
            work[at.g + c] = (float)d;
#pragma unroll
            for (int i = 0; i < CHUNK; ++i) sg[i * RS + c] = kd[i];
        } else {
#pragma unroll
            for (int i = 0; i < CHUNK; ++i) x[i] = i < n && c < C ? p.v[(size_t)(t0 + min(i, n - 1)) * p.ldv + (size_t)head * C + min(c, C - 1)] : 0.f;
        }
        if (!DELTA && key) continue;
        float y[CHUNK];
#pragma unroll
        for (int t = 0; t < CHUNK; ++t) {
            if (DELTA) {
                float s = 0.f;
#pragma unroll
                for (int i = 0; i <= t; ++i) s += sM[t][i] * x[i];
                y[t] = s;
                __builtin_amdgcn_sched_barrier(0);
            } else {
                y[t] = x[t] * sBeta[t];
            }
        }
        if (key) {
#pragma unroll
            for (int t = 0; t < CHUNK; ++t) sk[t * RS + c] = y[t];
        } else {
            f32x4_t* wv = (f32x4_t*)(work + at.u) + c / 16 * WAVE + c % 16;
#pragma unroll
            for (int s = 0; s < CHUNK; s += 4) wv[s * 4] = (f32x4_t){y[row_of_slot(s)], y[row_of_slot(s + 1)], y[row_of_slot(s + 2)], y[row_of_slot(s + 3)]};
        }
    }
    __syncthreads();
    for (int unit = tid; unit < Rp * 4; unit += 256) {             // (CHUNK * Rp floats in 16 bytes each)
        const int tile = unit / WAVE, a = unit % 16, b = unit % WAVE / 16 * 4;
        const int row = row_of_slot(a);
        ((f32x4_t*)(work + at.q))[unit] = *(const f32x4_t*)(sq + row * RS + tile * 16 + b);
        if (DELTA) ((f32x4_t*)work)[unit] = *(const f32x4_t*)(sk + row * RS + tile * 16 + b);
        const float* kd = sg + b / 4 * RS + tile * 16 + a;         // (slots b .. b + 3: rows b / 4, 4 + b / 4, ..)
        ((f32x4_t*)(work + at.kd))[unit] = (f32x4_t){kd[0], kd[4 * RS], kd[8 * RS], kd[12 * RS]};
    }
}

// A block a (head, segment, 16 columns), five waves.  The state's rows in tiles of 16: wave w < 4 owns the tiles w NT ..
// w NT + NT - 1, in the matrix instruction's result layout (lane l: rows 4 (l / 16) + i of the tile, column l % 16), which
// serves as its right operand as it is when the left operand's inner index runs alike: every operand is a 16-byte load.
// A chunk is M Kg S0 (each wave its rows' share), the meeting of the four shares through LDS, (D q) S0 while they travel,
// and the new S; the fifth wave adds the shares of (D q) S0 and P U, one chunk behind, and writes the results.
// AHEAD chunks' operands are in flight (an even number).  The loads of a chunk are kept together in program order: they
// return in order, so a chunk's wait then leaves those of the chunks behind it in flight.
template <int NT, int AHEAD, bool DELTA>
__global__ void __launch_bounds__(320) __attribute__((amdgpu_waves_per_eu(2, 2))) channel_walk_kernel(ChunkArgs p) {
    __shared__ f32x4_t share_w[DELTA ? 2 : 1][4][DELTA ? WAVE : 1], share_o[2][4][WAVE];         // [chunk parity][wave][lane]
    const int head = blockIdx.x, seg = blockIdx.z, wave = threadIdx.x / WAVE, lane = threadIdx.x % WAVE;
    const int t0 = p.seg_start[seg], t1 = p.seg_start[seg + 1];
    if (t1 <= t0) return;
    const int base = t0 / CHUNK + seg, chunks = (t1 - t0 + CHUNK - 1) / CHUNK;
    const int first = max(base, p.slot0), last = min(base + chunks, p.slot0 + p.slots);
    if (first >= last) return;
    const int m = lane % 16, kg = lane / 16, R = p.R, C = p.C, Rp = p.Rp;
    const int c = blockIdx.y * 16 + m;
    const ChunkLayout<DELTA> at(Rp, p.Cp);
    const size_t per = (size_t)at.floats;
    auto operands = [&](int slot) { return (const char*)(p.work + ((size_t)(min(slot, last - 1) - p.slot0) * p.heads + head) * per); };
    // byte offsets of this lane's words from a chunk's operands (a uniform address): 32 bits
    const unsigned at_u = (at.u + (blockIdx.y * WAVE + lane) * 4) * 4u;
    auto writes = [&](f32x4_t u, int par) {          // the rows' writes: M V - M Kg S0
        if (!DELTA) return u;
        return u - ((share_w[par][0][lane] + share_w[par][1][lane]) + (share_w[par][2][lane] + share_w[par][3][lane]));
    };
    if (wave == 4) {
        const unsigned at_p = (at.pr + lane * 4) * 4u;
        struct Result { f32x4_t u, pr; } ring[AHEAD];
        auto fetch = [&](Result& r, int slot) {
            const char* w = operands(slot);
            r.u = *(const f32x4_t*)(w + at_u);
            r.pr = *(const f32x4_t*)(w + at_p);
        };
#pragma unroll
        for (int d = 0; d < AHEAD; ++d) fetch(ring[d], first + d);
        f32x4_t u = {0.f, 0.f, 0.f, 0.f}, pr = u;
        auto finish = [&](int slot, int par) {       // o of the chunk before, whose shares are there now
            f32x4_t own = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int i = 0; i < 4; ++i) own = __builtin_amdgcn_mfma_f32_16x16x4f32(pr[i], u[i], own, 0, 0, 0);
            if (__builtin_expect(__any((own[0] * 0.f + own[1] * 0.f) + (own[2] * 0.f + own[3] * 0.f) != 0.f), 0)) {
                // a write that is no finite number, times the zeros of P, reaches the rows before it: once more, row by row
                own = (f32x4_t){0.f, 0.f, 0.f, 0.f};
#pragma unroll 1
                for (int b = 0; b < 4; ++b)
#pragma unroll
                    for (int j = 0; j < 4; ++j) {        // slot 4 b + j, row 4 j + b of the chunk
                        const float write = __shfl(u[j], 16 * b + m, WAVE);
#pragma unroll
                        for (int i = 0; i < 4; ++i) {
                            const float score = __shfl(pr[j], 16 * b + 4 * kg + i, WAVE);
                            if (4 * j + b <= 4 * i + kg) own[i] += score * write;
                        }
                    }
            }
            const f32x4_t y = ((share_o[par][0][lane] + share_o[par][1][lane]) + (share_o[par][2][lane] + share_o[par][3][lane])) + own;
            const int row = t0 + (slot - base) * CHUNK + kg;
#pragma unroll
            for (int i = 0; i < 4; ++i)                  // (slot 4 kg + i of the chunk)
                if (row + 4 * i < t1 && c < C) p.out[(size_t)(row + 4 * i) * p.ldo + (size_t)head * C + c] = y[i];
        };
        for (int turn = first; turn < last; turn += AHEAD)
#pragma unroll
            for (int d = 0; d < AHEAD; ++d) {
                if (turn + d < last) {
                    __syncthreads();
                    if (turn + d > first) finish(turn + d - 1, (d + 1) & 1);
                    u = writes(ring[d].u, d & 1);
                    pr = ring[d].pr;
                }
                fetch(ring[d], turn + d + AHEAD);
            }
        __syncthreads();
        finish(last - 1, (last - 1 - first) & 1);
        return;
    }
    float* state = p.state + (long long)p.state_slots[seg] * p.slot_stride + (size_t)head * R * C;
    f32x4_t S[NT];
#pragma unroll
    for (int j = 0; j < NT; ++j)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int r = (wave * NT + j) * 16 + 4 * kg + i;
            S[j][i] = r < R && c < C ? state[(size_t)r * C + c] : 0.f;
        }
    struct Operands { f32x4_t kg[DELTA ? NT : 1], qg[NT], kd[NT], g[NT], u; } ring[AHEAD];
    unsigned at_k[NT], at_g[NT];
    float mine[NT];
    const unsigned q_words = at.q * 4u, d_words = at.kd * 4u;
#pragma unroll
    for (int j = 0; j < NT; ++j) {
        const unsigned r = min((wave * NT + j) * 16, Rp - 16);          // (a wave without this tile reads another: its S stays zero)
        mine[j] = (wave * NT + j) * 16 < Rp ? 1.f : 0.f;
        at_k[j] = (r * 4 + lane) * 16u;
        at_g[j] = (at.g + r + 4 * kg) * 4u;
    }
    auto fetch = [&](Operands& o, int slot) {
        const char* w = operands(slot);
        if (DELTA) {
#pragma unroll
            for (int j = 0; j < NT; ++j) o.kg[j] = *(const f32x4_t*)(w + at_k[j]);
        }
#pragma unroll
        for (int j = 0; j < NT; ++j) o.qg[j] = *(const f32x4_t*)(w + q_words + at_k[j]);
        o.u = *(const f32x4_t*)(w + at_u);
#pragma unroll
        for (int j = 0; j < NT; ++j) {
            o.g[j] = *(const f32x4_t*)(w + at_g[j]);
            o.kd[j] = *(const f32x4_t*)(w + d_words + at_k[j]);
        }
    };
    auto walk = [&](Operands& now, int par) {
        const f32x4_t zero = {0.f, 0.f, 0.f, 0.f};
        // (a sum a tile of sixteen rows of S, then theirs)
        auto with_state = [&](const f32x4_t (&left)[NT]) {
            f32x4_t part[NT];
#pragma unroll
            for (int j = 0; j < NT; ++j) part[j] = zero;
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int j = 0; j < NT; ++j) part[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(left[j][i], S[j][i], part[j], 0, 0, 0);
            if constexpr (NT == 4) return (part[0] + part[1]) + (part[2] + part[3]);
            else if constexpr (NT == 3) return (part[0] + part[1]) + part[2];
            else if constexpr (NT == 2) return part[0] + part[1];
            else return part[0];
        };
        if constexpr (DELTA) share_w[par][wave][lane] = with_state(now.kg);
        __syncthreads();           // (the other parity's shares were read before the barrier before this one's writes)
        const f32x4_t u = writes(now.u, par);
        share_o[par][wave][lane] = with_state(now.qg);
        // what the chunk's rows write is summed apart from S, eight rows and eight: S is rounded twice a chunk instead of sixteen times
        f32x4_t early[NT], late[NT];
#pragma unroll
        for (int j = 0; j < NT; ++j) early[j] = late[j] = zero;
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int j = 0; j < NT; ++j) {
                early[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(now.kd[j][i] * mine[j], u[i], early[j], 0, 0, 0);
                late[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(now.kd[j][2 + i] * mine[j], u[2 + i], late[j], 0, 0, 0);
            }
#pragma unroll
        for (int j = 0; j < NT; ++j)
#pragma unroll
            for (int i = 0; i < 4; ++i) S[j][i] = fmaf(S[j][i], now.g[j][i], early[j][i]) + late[j][i];
    };
#pragma unroll
    for (int d = 0; d < AHEAD; ++d) {
        fetch(ring[d], first + d);
        __builtin_amdgcn_sched_barrier(0);
    }
    // (a turn past the last chunk loads a chunk again and does nothing: no way out of the unrolled loop, so that the waits of
    // every turn stay exact)
    for (int turn = first; turn < last; turn += AHEAD)
#pragma unroll
        for (int d = 0; d < AHEAD; ++d) {
            if (turn + d < last) walk(ring[d], d & 1);          // (uniform over the block)
            __builtin_amdgcn_sched_barrier(0);
            fetch(ring[d], turn + d + AHEAD);
            __builtin_amdgcn_sched_barrier(0);
        }
    __syncthreads();               // (the last chunk's shares of (D q) S0 are there)
#pragma unroll
    for (int j = 0; j < NT; ++j)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int r = (wave * NT + j) * 16 + 4 * kg + i;
            if (r < R && c < C) state[(size_t)r * C + c] = S[j][i];
        }
}

// Chunk slots of a step, and floats of `work` a slot takes.
extern "C" int cisr_channel_chunk_slots(int rows, int segments) { return rows / CHUNK + segments; }
extern "C" long long cisr_channel_chunk_floats(int heads, int R, int C, int delta) {
    const int Rp = (R + 15) / 16 * 16, Cp = (C + 15) / 16 * 16;
    return (long long)heads * (delta ? ChunkLayout<true>(Rp, Cp).floats : ChunkLayout<false>(Rp, Cp).floats);
}

template <bool DELTA, bool VEC>
static int launch_chunks(ChunkArgs p, int rows, int slab, hipStream_t stream) {
    const int total = rows / CHUNK + p.segments, nt = (p.Rp / 16 + 3) / 4;
    const size_t lds = (size_t)3 * CHUNK * (p.Rp + 4) * sizeof(float);
    for (p.slot0 = 0; p.slot0 < total; p.slot0 += slab) {
        p.slots = min(slab, total - p.slot0);
        channel_chunk_kernel<DELTA, VEC><<<dim3(p.heads, p.slots), 256, lds, stream>>>(p);
        int err = CISR_LAUNCH_CHECK();
        if (err) return err;
        const dim3 grid(p.heads, p.Cp / 16, p.segments);
        if (nt == 1) channel_walk_kernel<1, 4, DELTA><<<grid, 320, 0, stream>>>(p);
        else if (nt == 2) channel_walk_kernel<2, 4, DELTA><<<grid, 320, 0, stream>>>(p);
        else if (nt == 3) channel_walk_kernel<3, 2, DELTA><<<grid, 320, 0, stream>>>(p);
        else channel_walk_kernel<4, 2, DELTA><<<grid, 320, 0, stream>>>(p);
        err = CISR_LAUNCH_CHECK();
        if (err) return err;
    }
    return 0;
}

// The step's rows in launches of `slab` chunk slots each (two kernels a slab); work: slab * cisr_channel_chunk_floats floats.
// `delta`: the delta rule (b: its write strengths before the sigmoid); else the linear scan (b: null or its step sizes).
// `vec`: a decay a head and key channel; else one a head.
extern "C" int cisr_channel_chunks(const float* q, int ldq, const float* k, int ldk, const float* v, int ldv, const float* g, int ldg,
                                   const float* b, int ldb, float* out, int ldo, float* state, long long slot_stride,
                                   const int* seg_start, const int* state_slots, int rows, int segments, int heads, int R, int C,
                                   int share, float q_scale, int delta, int vec, float* work, int slab, hipStream_t stream) {
    if (rows <= 0 || segments <= 0 || heads <= 0) return 0;
    if (R <= 0 || R > 256 || C <= 0 || share <= 0 || heads % share || segments > 65535 || (C + 15) / 16 > 65535 || slab <= 0 || slab > 65535 ||
        (delta && !b) || (uintptr_t)work % 16)
        return (int)hipErrorInvalidValue;
    const ChunkArgs p{q, ldq, k, ldk, v, ldv, g, ldg, b, ldb, out, ldo, state, slot_stride, seg_start, state_slots, R, C, share, heads, segments,
                      q_scale, (R + 15) / 16 * 16, (C + 15) / 16 * 16, 0, 0, work};
    if (delta) return vec ? launch_chunks<true, true>(p, rows, slab, stream) : launch_chunks<true, false>(p, rows, slab, stream);
    return vec ? launch_chunks<false, true>(p, rows, slab, stream) : launch_chunks<false, false>(p, rows, slab, stream);
}
