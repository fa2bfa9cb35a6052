// Kernels of mixers that carry a fixed-size state per request instead of keys and values:
//
//   linear scan     S_t = diag(a_t) S_(t-1) + k_t v_t^T,  o_t = S_t^T q_t   per head, S [R, C] float in the state slot
//                   of the row's request; a_t a vector over the R rows (a decay per key channel) or one number a head
//                   (state-space duality), q and k of a group of heads shared or not, v optionally times a step size
//   short conv      a causal convolution per channel over the last `taps` inputs, the taps - 1 inputs before a portion
//                   taken from the state slot, + bias, silu; with it the step sizes softplus(dt + bias) and the decays
//                   exp(-exp(A_log) dt) of a state-space layer
//   decay gates     a = sigmoid(z + bias)^(1 / tau) as exp(log sigmoid / tau)
//   group norm gate the output of such a mixer: RMS norm over equal parts of a row, times a weight, with a silu gate
//                   before or after the norm and an optional skip term D x
//
// Every kernel takes a step's rows as they come: portions of several requests side by side, single tokens among
// them.  seg_start[s] .. seg_start[s + 1] are the rows of segment s, state_slots[s] its request's slot; a segment
// without rows (padding of a captured step) touches nothing.  All of it is float arithmetic on float data: what
// enters a recurrence is 32-bit in every mode.
#include "common.h"
#include "recurrence_scan.inc"

// ------------------------------------------------------------------------------------------------ linear scan
// (the kernel: recurrence_scan.inc; one source file a tile width)
// Floats of `carry` and of `carry_decay` that a launch over `rows` rows in pieces of `piece` rows needs.
extern "C" long long cisr_linear_scan_carry(int rows, int piece, int heads, int R, int C, int vec, long long* decay_floats) {
    const long long pieces = piece > 0 ? (rows + piece - 1) / piece : 0;     // (the segments' pieces but their last are at most rows / piece)
    if (decay_floats) *decay_floats = pieces * heads * (vec ? R : 1);
    return pieces * heads * R * C;
}

int cisr_scan_launch_c4(const ScanArgs& p, int segments, bool vec, hipStream_t stream);
int cisr_scan_launch_c8(const ScanArgs& p, int segments, bool vec, hipStream_t stream);
int cisr_scan_launch_c16(const ScanArgs& p, int segments, bool vec, hipStream_t stream);

// silu 1: q, k and v are silu of what is stored.  lda 0: decays that do not change from row to row.
// cols: 4, 8 or 16 columns a wave (the caller's rule: fewer columns are more waves for the same head).  piece > 0:
// segments longer than `piece` rows are walked in pieces of that many rows side by side (three launches; `rows` is the
// number of rows of the step, carry / carry_decay as cisr_linear_scan_carry says); piece 0: a wave walks a whole segment.
extern "C" int cisr_linear_scan(const float* q, int ldq, const float* k, int ldk, const float* v, int ldv,
                                const float* a, int lda, int vec, const float* vs, int ldvs, float* out, int ldo,
                                float* state, long long slot_stride, const int* seg_start, const int* state_slots,
                                int segments, int heads, int R, int C, int share, float q_scale, int silu, int cols,
                                int rows, int piece, float* carry, float* carry_decay, hipStream_t stream) {
    if (segments <= 0 || heads <= 0) return 0;
    if (R <= 0 || C <= 0 || share <= 0 || heads % share || heads > 65535 || (cols != 4 && cols != 8 && cols != 16) ||
        piece < 0 || (piece > 0 && (!carry || !carry_decay || rows <= 0)))
        return (int)hipErrorInvalidValue;
    ScanArgs p{q, ldq, k, ldk, v, ldv, a, lda, vs, ldvs, out, ldo, state, slot_stride, seg_start, state_slots, R, C, share, heads,
               q_scale, silu, piece, piece > 0 ? (rows + piece - 1) / piece : 1, 0, carry, carry_decay};
    if ((C + cols - 1) / cols > 65535 || R > 256 || (piece > 0 && segments > 65535)) return (int)hipErrorInvalidValue;
    if (cols == 4) return cisr_scan_launch_c4(p, segments, vec, stream);
    if (cols == 8) return cisr_scan_launch_c8(p, segments, vec, stream);
    return cisr_scan_launch_c16(p, segments, vec, stream);
}

// ------------------------------------------------------------------------------------------------ short conv
#define MAX_TAPS 16

// in[t * ld + first + ch], ch < channels: the convolution's inputs of row t.  conv_state[slot * slot_stride +
// j * channels + ch], j < taps - 1: the inputs of the request's last taps - 1 tokens, oldest first.
// out[t * channels + ch] = silu(bias[ch] + sum_j w[ch * taps + j] * input(t - (taps - 1) + j)).
// Index channels + h, h < heads (if heads > 0): step[t * heads + h] = softplus(in[t * ld + dt_first + h] + dt_bias[h]),
// decay[t * heads + h] = exp(-exp(a_log[h]) * step).
// UNIT (unit.channels > 0): the first `unit.channels` results are heads of unit.dim (a power of two from 16 to 256) channels, each of which
// becomes x / sqrt(sum(x^2) + eps): the queries and keys of a delta rule, otherwise a kernel of their own (recurrence_delta.hip) that
// reads and writes them once more.  A head's squares are added neighbour by neighbour, pair by pair, in either kernel.  Of 8,192 channels
// 4,096 in heads of 128, us of the convolution / with the kernel behind it / so: 1,999 rows 40.6 / 58.7 / 40.6, 300 rows 17.5 / 23.7 / 17.0, 8 single
// rows 3.4 / 5.8 / 3.7, 64 6.2 / 9.0 / 6.2.
// SINGLE: every segment has one row (a step of single tokens), so the thread of a (row, channel) is the only one that
// reads that channel of its request's state, and it moves the state on itself: no second launch.
struct ConvUnit { int channels, dim; float eps; };

template <int CTRL>
__device__ __forceinline__ float conv_moved(float x) { return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), CTRL, 0xf, 0xf, false)); }

// the sum over the aligned group of `lanes` (1, 2, 4, ... 64) neighbours, in all of them, without a trip through LDS
__device__ __forceinline__ float conv_neighbours(float x, int lanes) {
    if (lanes >= 2) x += conv_moved<0xb1>(x);                  // quad_perm [1, 0, 3, 2]
    if (lanes >= 4) x += conv_moved<0x4e>(x);                  // quad_perm [2, 3, 0, 1]
    if (lanes >= 8) x += conv_moved<0x141>(x);                 // row_half_mirror (the quads' sums are the same in all four)
    if (lanes >= 16) x += conv_moved<0x140>(x);                // row_mirror
    if (lanes >= 32) {
        const auto a = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
        x = __uint_as_float(a[0]) + __uint_as_float(a[1]);
    }
    if (lanes >= 64) {
        const auto a = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
        x = __uint_as_float(a[0]) + __uint_as_float(a[1]);
    }
    return x;
}

template <bool SINGLE, bool UNIT>
__global__ void __launch_bounds__(256)
conv_silu_kernel(const float* __restrict__ in, int ld, int first, const float* __restrict__ w, const float* __restrict__ bias,
                 float* conv_state, long long slot_stride, float* __restrict__ out,
                 const int* __restrict__ seg_of_row, const int* __restrict__ seg_start, const int* __restrict__ state_slots,
                 int channels, int taps, int heads, int dt_first, const float* __restrict__ dt_bias,
                 const float* __restrict__ a_log, float* __restrict__ step, float* __restrict__ decay, ConvUnit unit) {
    const int t = blockIdx.x;
    const int idx = blockIdx.y * 256 + threadIdx.x;
    const int seg = seg_of_row[t];
    const bool units = UNIT && (int)blockIdx.y * 256 < unit.channels;       // (uniform: a block that meets in the end, and all of its threads come)
    if (seg < 0 || (idx >= channels + heads && !units)) return;
    if (idx >= channels && idx < channels + heads) {
        const int h = idx - channels;
        const float z = in[(size_t)t * ld + dt_first + h] + dt_bias[h];
        const float dt = z > 20.f ? z : log1pf(expf(z));
        step[(size_t)t * heads + h] = dt;
        decay[(size_t)t * heads + h] = expf(-expf(a_log[h]) * dt);
        if (!units) return;
    }
    float y = 0.f;
    if (idx < channels) {
        const int rel = t - seg_start[seg];
        float* st = conv_state + (long long)state_slots[seg] * slot_stride;
        y = bias ? bias[idx] : 0.f;
        for (int j = 0; j < taps; ++j) {
            const int src = rel - (taps - 1) + j;
            const float x = src >= 0 ? in[(size_t)(t - rel + src) * ld + first + idx] : st[(size_t)(taps - 1 + src) * channels + idx];
            y += w[(size_t)idx * taps + j] * x;
            if (SINGLE && j > 0) st[(size_t)(j - 1) * channels + idx] = x;     // (input j of this row is input j - 1 of the next)
        }
        y = y / (1.0f + expf(-y));
    }
    if (units) {
        __shared__ float red[4];
        float sum = conv_neighbours(y * y, min(unit.dim, WAVE));
        if (unit.dim > WAVE) {
            const int wave = threadIdx.x / WAVE;
            if (threadIdx.x % WAVE == 0) red[wave] = sum;
            __syncthreads();
            sum = red[wave & ~1] + red[wave | 1];
            if (unit.dim > 2 * WAVE) sum = (red[0] + red[1]) + (red[2] + red[3]);
        }
        if (idx < unit.channels) y *= rsqrtf(sum + unit.eps);
    }
    if (idx < channels) out[(size_t)t * channels + idx] = y;
}

// The same for portions, four channels a thread and CONV_ROWS rows of the step a block: an input is read once (the taps - 1
// before a block's first row again), eight rows' 16-byte loads are on their way together.  The same sums in the same order.
// Channels, row stride and first column multiples of 4, pointers 16-byte aligned.  The last blocks of y make the gates.
// A block all of whose rows are one portion's, none of them within the portion's first, looks nothing up row by row and asks for a
// row eight rows before its turn; in the others a portion that begins inside brings its state when its first row comes.  (With the
// state's rows chosen input by input a wave of four taps held 174 registers, two waves a SIMD; so 82, and the stream of
// memory is what bounds it.)  2,048 rows of 8,192 channels, four taps (134 MB): 90 us with a thread a (row, channel), 45 with rows looked
// up and the state chosen input by input, 34 so; fifty portions of 40 rows 42.5 / 39.0, 2,368 rows of 6,144 35.3 / 29.0, 4,096 of 8,192
// 76 / 60 (both with the state's own kernel).  A block's walk takes 12 to 14 us
// however few blocks there are, more where it meets portions that begin (their first rows wait for the state, one after the
// other; 16 single rows 22 us).  Steps of fewer inputs than that is worth keep a thread a (row, channel): 128 rows of 8,192 channels
// 10.1 us against 13.1 (200 rows 14.8 against 13.9), 1,024 of 1,024 9.6 against 12.7 (1,500 rows 13.2 against 12.8); 24 single
// rows beside 256, 8,192 channels, 18.9 against 25.2 (beside 512 28.8 against 26.9).
#define CONV_ROWS 16
#define CONV_WORDS (3ll << 19)               // inputs of a step of one portion
#define CONV_WORDS_A_PORTION 170000ll        // and for each of up to sixteen more
typedef __attribute__((ext_vector_type(4))) float conv_f32x4;
template <int TAPS, bool UNIT>
__global__ void __launch_bounds__(256)
conv_silu_rows_kernel(const float* __restrict__ in, int ld, int first, const float* __restrict__ w, const float* __restrict__ bias,
                      const float* __restrict__ conv_state, long long slot_stride, float* __restrict__ out,
                      const int* __restrict__ seg_of_row, const int* __restrict__ seg_start, const int* __restrict__ state_slots,
                      int rows, int channels, int heads, int dt_first, const float* __restrict__ dt_bias,
                      const float* __restrict__ a_log, float* __restrict__ step, float* __restrict__ decay, ConvUnit unit) {
    const int t0 = blockIdx.x * CONV_ROWS, t1 = min(t0 + CONV_ROWS, rows);
    const int channel_blocks = (channels / 4 + 255) / 256;
    if ((int)blockIdx.y >= channel_blocks) {
        const int h = ((int)blockIdx.y - channel_blocks) * 256 + threadIdx.x;
        if (h >= heads) return;
        for (int t = t0; t < t1; ++t) {
            if (seg_of_row[t] < 0) continue;
            const float z = in[(size_t)t * ld + dt_first + h] + dt_bias[h];
            const float dt = z > 20.f ? z : log1pf(expf(z));
            step[(size_t)t * heads + h] = dt;
            decay[(size_t)t * heads + h] = expf(-expf(a_log[h]) * dt);
        }
        return;
    }
    const int c = ((int)blockIdx.y * 256 + threadIdx.x) * 4;
    if (c >= channels) return;
    const int wave_first = __builtin_amdgcn_readfirstlane(c);
    const float* x0 = in + first + c;
    float taps[4][TAPS];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < TAPS; ++j) taps[i][j] = w[(size_t)(c + i) * TAPS + j];
    const conv_f32x4 b = bias ? *(const conv_f32x4*)(bias + c) : (conv_f32x4){0.f, 0.f, 0.f, 0.f};
    auto row = [&](int t) { return *(const conv_f32x4*)(x0 + (size_t)t * ld); };
    auto finish = [&](int t, const conv_f32x4 (&use)[TAPS]) __attribute__((always_inline)) {
        conv_f32x4 y = b;
#pragma unroll
        for (int j = 0; j < TAPS; ++j)
#pragma unroll
            for (int k = 0; k < 4; ++k) y[k] += taps[k][j] * use[j][k];
#pragma unroll
        for (int k = 0; k < 4; ++k) y[k] = y[k] / (1.0f + expf(-y[k]));
        if constexpr (UNIT) {                            // (whole waves beyond the heads pass by)
            if (wave_first < unit.channels) {
                const float f = rsqrtf(conv_neighbours((y[0] * y[0] + y[1] * y[1]) + (y[2] * y[2] + y[3] * y[3]), unit.dim / 4) + unit.eps);
                if (c < unit.channels) y *= f;
            }
        }
        *(conv_f32x4*)(out + (size_t)t * channels + c) = y;
    };
    const int whose = seg_of_row[t0];
    if (whose >= 0 && t0 - seg_start[whose] >= TAPS - 1 && t0 + CONV_ROWS <= seg_start[whose + 1]) {
        // the block's rows are one portion's and reach back into rows of it only: nothing to look up row by row.  (Told from the
        // portion's ends, which all lanes read: of a row's last wave only the lanes that still have channels are left to vote.)
        conv_f32x4 x[CONV_ROWS + TAPS - 1];          // (a row is asked for eight rows before its turn)
#pragma unroll
        for (int i = 0; i < TAPS - 1 + 8; ++i) x[i] = row(t0 - (TAPS - 1) + i);
#pragma unroll
        for (int i = 0; i < CONV_ROWS; ++i) {
            conv_f32x4 use[TAPS];
#pragma unroll
            for (int j = 0; j < TAPS; ++j) use[j] = x[i + j];
            finish(t0 + i, use);
            if (i + 8 < CONV_ROWS) x[i + TAPS - 1 + 8] = row(t0 + i + 8);
            __builtin_amdgcn_sched_barrier(0);
        }
        return;
    }
    // the inputs of the TAPS - 1 rows before: a portion's first rows reach back into the request's state, rel of them behind it
    conv_f32x4 before[TAPS - 1];
    auto from_state = [&](int seg, int rel) __attribute__((always_inline)) {
        const float* st = conv_state + (long long)state_slots[seg] * slot_stride + c;
#pragma unroll
        for (int j = 0; j < TAPS - 1; ++j)
            if (rel + j < TAPS - 1) {
                const float* from = st + (size_t)(rel + j) * channels;
                before[j] = (conv_f32x4){from[0], from[1], from[2], from[3]};
            }
    };
#pragma unroll
    for (int j = 0; j < TAPS - 1; ++j) before[j] = row(max(t0 - (TAPS - 1) + j, 0));
    const int rel0 = whose < 0 ? 0 : t0 - seg_start[whose];
    if (rel0 > 0 && rel0 < TAPS - 1) from_state(whose, rel0);
    for (int tb = t0; tb < t1; tb += 8) {
        conv_f32x4 x[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) x[i] = row(min(tb + i, rows - 1));
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const int t = tb + i;
            if (t >= t1) break;                      // (uniform)
            const int seg = seg_of_row[t];
            if (seg >= 0 && t == seg_start[seg]) from_state(seg, 0);
            conv_f32x4 use[TAPS];
#pragma unroll
            for (int j = 0; j < TAPS - 1; ++j) use[j] = before[j];
            use[TAPS - 1] = x[i];
#pragma unroll
            for (int j = 0; j < TAPS - 1; ++j) before[j] = use[j + 1];
            if (seg >= 0) finish(t, use);
        }
    }
}

// After the convolution has read it: the state becomes the last taps - 1 inputs of (state, portion).
__global__ void __launch_bounds__(256)
conv_state_kernel(const float* __restrict__ in, int ld, int first, float* __restrict__ conv_state, long long slot_stride,
                  const int* __restrict__ seg_start, const int* __restrict__ state_slots, int channels, int taps) {
    const int seg = blockIdx.x, ch = blockIdx.y * 256 + threadIdx.x;
    const int t0 = seg_start[seg], count = seg_start[seg + 1] - t0;
    if (count <= 0 || ch >= channels) return;
    float* st = conv_state + (long long)state_slots[seg] * slot_stride;
    float keep[MAX_TAPS];
#pragma unroll
    for (int i = 0; i < MAX_TAPS; ++i) {
        if (i >= taps - 1) break;
        const int src = count - (taps - 1) + i;
        keep[i] = src >= 0 ? in[(size_t)(t0 + src) * ld + first + ch] : st[(size_t)(taps - 1 + src) * channels + ch];
    }
#pragma unroll
    for (int i = 0; i < MAX_TAPS; ++i) {
        if (i >= taps - 1) break;
        st[(size_t)i * channels + ch] = keep[i];
    }
}

extern "C" int cisr_conv_silu(const float* in, int ld, int first, const float* w, const float* bias, float* conv_state,
                              long long slot_stride, float* out, const int* seg_of_row, const int* seg_start,
                              const int* state_slots, int rows, int segments, int channels, int taps, int heads,
                              int dt_first, const float* dt_bias, const float* a_log, float* step, float* decay,
                              int single_rows, int unit_channels, int unit_dim, float unit_eps, hipStream_t stream) {
    if (rows <= 0 || segments <= 0) return 0;
    const ConvUnit unit{unit_channels, unit_dim, unit_eps};
    if (unit_channels < 0 || unit_channels > channels ||
        (unit_channels && (unit_dim < 16 || unit_dim > 256 || (unit_dim & (unit_dim - 1)) || unit_channels % unit_dim)))
        return (int)hipErrorInvalidValue;
    if (channels <= 0 || taps < 1 || taps > MAX_TAPS || heads < 0 || segments > 65535) return (int)hipErrorInvalidValue;
    const dim3 grid(rows, (channels + heads + 255) / 256);
#define CONV_FEW_AS(SINGLE, UNIT) conv_silu_kernel<SINGLE, UNIT><<<grid, 256, 0, stream>>>(in, ld, first, w, bias, conv_state, slot_stride, \
        out, seg_of_row, seg_start, state_slots, channels, taps, heads, dt_first, dt_bias, a_log, step, decay, unit)
#define CONV_FEW(SINGLE) do { if (unit_channels) CONV_FEW_AS(SINGLE, true); else CONV_FEW_AS(SINGLE, false); } while (0)
    if (single_rows) {       // `single_rows`: the caller knows that no segment has more than one row
        CONV_FEW(true);
        return CISR_LAUNCH_CHECK();
    }
    const bool enough = (long long)rows * channels >= CONV_WORDS + CONV_WORDS_A_PORTION * min(segments - 1, 16);
    if (enough && taps >= 2 && taps <= 4 && channels % 4 == 0 && ld % 4 == 0 && first % 4 == 0 && (uintptr_t)in % 16 == 0 && (uintptr_t)out % 16 == 0 &&
        (!bias || (uintptr_t)bias % 16 == 0)) {
        const dim3 blocks((rows + CONV_ROWS - 1) / CONV_ROWS, (channels / 4 + 255) / 256 + (heads + 255) / 256);
#define CONV_ROWS_AS(TAPS, UNIT) conv_silu_rows_kernel<TAPS, UNIT><<<blocks, 256, 0, stream>>>(in, ld, first, w, bias, conv_state, slot_stride, \
            out, seg_of_row, seg_start, state_slots, rows, channels, heads, dt_first, dt_bias, a_log, step, decay, unit)
#define CONV_ROWS_OF(TAPS) do { if (unit_channels) CONV_ROWS_AS(TAPS, true); else CONV_ROWS_AS(TAPS, false); } while (0)
        if (taps == 2) CONV_ROWS_OF(2);
        else if (taps == 3) CONV_ROWS_OF(3);
        else CONV_ROWS_OF(4);
#undef CONV_ROWS_OF
#undef CONV_ROWS_AS
    } else {
        CONV_FEW(false);
    }
#undef CONV_FEW
#undef CONV_FEW_AS
    int err = CISR_LAUNCH_CHECK();
    if (err || taps == 1) return err;
    conv_state_kernel<<<dim3(segments, (channels + 255) / 256), 256, 0, stream>>>(in, ld, first, conv_state, slot_stride, seg_start,
        state_slots, channels, taps);
    return CISR_LAUNCH_CHECK();
}

// ------------------------------------------------------------------------------------------------ decay gates
// a[i] = sigmoid(z[t * ld + c] + bias[c])^(1 / tau) = exp(log sigmoid(.) / tau), log sigmoid(u) = min(u, 0) - log1p(exp(-|u|))
__global__ void decay_gate_kernel(const float* __restrict__ z, int ld, const float* __restrict__ bias, float* __restrict__ a,
                                  int cols, size_t n, float inv_tau) {
    const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    const size_t t = i / cols;
    const int c = (int)(i % cols);
    const float u = z[t * ld + c] + (bias ? bias[c] : 0.f);
    a[i] = expf((fminf(u, 0.f) - log1pf(expf(-fabsf(u)))) * inv_tau);
}

// The same with z = up . low made on the way: z[t, c] = sum_r up_t[r * cols + c] * low[t * ld + r] (the second half of a
// low-rank projection, its matrix transposed so that neighbouring lanes read neighbouring words; the first half came
// out of the mixer's fused input product).
__global__ void decay_gate_low_rank_kernel(const float* __restrict__ low, int ld, int rank, const float* __restrict__ up,
                                           const float* __restrict__ bias, float* __restrict__ a, int cols, size_t n, float inv_tau) {
    const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    const size_t t = i / cols;
    const int c = (int)(i % cols);
    const float* lo = low + t * ld;
    const float* w = up + c;
    float u = bias ? bias[c] : 0.f;
#pragma unroll 4
    for (int r = 0; r < rank; ++r) u += w[(size_t)r * cols] * lo[r];
    a[i] = expf((fminf(u, 0.f) - log1pf(expf(-fabsf(u)))) * inv_tau);
}

// The same with GATE_ROWS rows a thread, which share the matrix's words: 2,368 rows of 1,024 decays through a rank of 16 20 us a
// decay a thread, 14 so.  The same sums in the same order.
#define GATE_ROWS 8
__global__ void __launch_bounds__(256)
decay_gate_low_rank_rows_kernel(const float* __restrict__ low, int ld, int rank, const float* __restrict__ up,
                                const float* __restrict__ bias, float* __restrict__ a, int rows, int cols, float inv_tau) {
    const int c = blockIdx.x * 256 + threadIdx.x, t0 = blockIdx.y * GATE_ROWS;
    if (c >= cols) return;
    float u[GATE_ROWS];
    const float b = bias ? bias[c] : 0.f;
#pragma unroll
    for (int i = 0; i < GATE_ROWS; ++i) u[i] = b;
#pragma unroll 4
    for (int r = 0; r < rank; ++r) {
        const float w = up[(size_t)r * cols + c];
#pragma unroll
        for (int i = 0; i < GATE_ROWS; ++i) u[i] += w * low[(size_t)min(t0 + i, rows - 1) * ld + r];     // (uniform over the block)
    }
#pragma unroll
    for (int i = 0; i < GATE_ROWS; ++i)
        if (t0 + i < rows) a[(size_t)(t0 + i) * cols + c] = expf((fminf(u[i], 0.f) - log1pf(expf(-fabsf(u[i])))) * inv_tau);
}

extern "C" int cisr_decay_gate_low_rank(const float* low, int ld, int rank, const float* up, const float* bias, float* a,
                                        int rows, int cols, float tau, hipStream_t stream) {
    const size_t n = (size_t)rows * cols;
    if (n == 0) return 0;
    if (!(tau > 0.f) || rank <= 0) return (int)hipErrorInvalidValue;
    // From a block for every compute unit on, and from about 12,000 blocks times rank on.  A decay a thread / so: rank 16, 512 rows of
    // 1,024 (256 blocks) 5.5 / 6.9, 782 of 2,048 (784) 11.3 / 10.8; rank 32, 300 rows of 2,048 (304) 8.3 / 8.9, 512 (512) 11.3 /
    // 9.2; rank 128, 64 rows of 4,096 (128) 11.4 / 12.3, 130 (272) 21.7 / 12.9.
    const long long blocks = (long long)((cols + 255) / 256) * ((rows + GATE_ROWS - 1) / GATE_ROWS);
    if (blocks >= 256 && blocks * rank >= 12000 && rows <= 65535 * GATE_ROWS)
        decay_gate_low_rank_rows_kernel<<<dim3((cols + 255) / 256, (rows + GATE_ROWS - 1) / GATE_ROWS), 256, 0, stream>>>(low, ld, rank, up, bias, a, rows, cols, 1.0f / tau);
    else
        decay_gate_low_rank_kernel<<<(unsigned)((n + 255) / 256), 256, 0, stream>>>(low, ld, rank, up, bias, a, cols, n, 1.0f / tau);
    return CISR_LAUNCH_CHECK();
}

extern "C" int cisr_decay_gate(const float* z, int ld, const float* bias, float* a, int rows, int cols, float tau,
                               hipStream_t stream) {
    const size_t n = (size_t)rows * cols;
    if (n == 0) return 0;
    if (!(tau > 0.f)) return (int)hipErrorInvalidValue;
    decay_gate_kernel<<<(unsigned)((n + 255) / 256), 256, 0, stream>>>(z, ld, bias, a, cols, n, 1.0f / tau);
    return CISR_LAUNCH_CHECK();
}

// ------------------------------------------------------------------------------------------------ group norm gate
// Row t of y [T, groups * size] in `groups` equal parts; part g, element d, i = g * size + d:
//   u = y[t, i] + (skip ? skip[i / skip_span] * x[t * ldx + i] : 0)
//   GATE_FIRST:  u *= silu(gate[t * ldg + i]);  out = u / rms(part) * w[shared ? d : i]
//   else:        out = u / rms(part) * w[shared ? d : i] * silu(gate[t * ldg + i])
// with `sigmoid` the gate's law is sigmoid instead of silu.
// A block of NT threads a (row, part): a wave for parts of up to 256 elements, four waves up to 2,048, sixteen beyond.
// KEEP: the part's elements (after the skip term and the gate before the norm) wait in LDS for their scale, so every
// input is read once; else (parts of more than 12,288 elements) they are made a second time.
template <typename T, bool GATE_FIRST, int NT, bool KEEP>
__global__ void __launch_bounds__(NT)
group_norm_gate_kernel(const float* __restrict__ y, const float* __restrict__ gate, int ldg, const float* __restrict__ w,
                       int shared, const float* __restrict__ skip, int skip_span, const float* __restrict__ x, int ldx,
                       T* __restrict__ out, int size, float eps, int sigmoid) {
    __shared__ float red[NT / WAVE];
    extern __shared__ float kept[];
    const int t = blockIdx.x, g = blockIdx.y, groups = gridDim.y, lane = threadIdx.x;
    const size_t base = (size_t)t * groups * size + (size_t)g * size;
    const int col0 = g * size;
    auto element = [&](int d) {
        float u = y[base + d];
        if (skip) u += skip[(col0 + d) / skip_span] * x[(size_t)t * ldx + col0 + d];
        if (GATE_FIRST) { const float z = gate[(size_t)t * ldg + col0 + d]; u *= (sigmoid ? 1.0f : z) / (1.0f + expf(-z)); }
        return u;
    };
    float ss = 0.f;
    for (int d = lane; d < size; d += NT) {
        const float u = element(d);
        if (KEEP) kept[d] = u;
        ss += u * u;
    }
    const float scale = 1.0f / sqrtf((NT == WAVE ? wave_sum(ss) : block_sum<NT>(ss, red)) / (float)size + eps);
    for (int d = lane; d < size; d += NT) {
        float u = (KEEP ? kept[d] : element(d)) * scale * w[shared ? d : col0 + d];     // (a thread reads back what it wrote)
        if (!GATE_FIRST) { const float z = gate[(size_t)t * ldg + col0 + d]; u *= (sigmoid ? 1.0f : z) / (1.0f + expf(-z)); }
        store_f32(out + base + d, u);
    }
}

// The same in 16-byte words with a part's elements in registers: NT neighbouring threads (half a wave, a wave or the block of
// 256) a part of up to 4 NT E elements.  Parts, row strides and the skip's span multiples of 4, pointers
// 16-byte aligned.  2,048 rows of 32 parts of 128 31 us with a word a lane, 18.6 so; 2,368 rows of one part of 4,096 44 and 27.5.
typedef __attribute__((ext_vector_type(4))) float gng_f32x4;
template <typename T, bool GATE_FIRST, int NT, int E>
__global__ void __launch_bounds__(256)
group_norm_gate_words_kernel(const float* __restrict__ y, const float* __restrict__ gate, int ldg, const float* __restrict__ w,
                             int shared, const float* __restrict__ skip, int skip_span, const float* __restrict__ x, int ldx,
                             T* __restrict__ out, int groups, int size, float eps, int sigmoid, long long parts) {
    __shared__ float red[4];
    const int lane = threadIdx.x % NT;
    const long long own = (long long)blockIdx.x * (256 / NT) + threadIdx.x / NT, part = own < parts ? own : parts - 1;
    const long long t = part / groups;
    const int col0 = (int)(part % groups) * size;
    gng_f32x4 u[E], z[E], wt[E], s[E];
#pragma unroll
    for (int e = 0; e < E; ++e) {
        const int d = min(4 * (lane + NT * e), size - 4);
        u[e] = *(const gng_f32x4*)(y + part * size + d);
        z[e] = *(const gng_f32x4*)(gate + t * ldg + col0 + d);
        wt[e] = *(const gng_f32x4*)(w + (shared ? d : col0 + d));
        s[e] = (gng_f32x4){0.f, 0.f, 0.f, 0.f};
        if (skip) {
            const float f = skip[(col0 + d) / skip_span];
            s[e] = *(const gng_f32x4*)(x + t * ldx + col0 + d);
#pragma unroll
            for (int k = 0; k < 4; ++k) s[e][k] *= f;
        }
    }
    float ss = 0.f;
#pragma unroll
    for (int e = 0; e < E; ++e) {
        const bool in = 4 * (lane + NT * e) < size;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const float g = (sigmoid ? 1.0f : z[e][k]) / (1.0f + expf(-z[e][k]));
            float v = u[e][k] + s[e][k];
            if (GATE_FIRST) v *= g;
            ss += in ? v * v : 0.f;
            u[e][k] = v;
            z[e][k] = g;
        }
    }
    float sum = ss;
    if constexpr (NT == 256) sum = block_sum<256>(ss, red);
    else
#pragma unroll
        for (int off = NT / 2; off > 0; off >>= 1) sum += __shfl_xor(sum, off, WAVE);
    if (own >= parts) return;
    const float scale = 1.0f / sqrtf(sum / (float)size + eps);
#pragma unroll
    for (int e = 0; e < E; ++e) {
        const int d = 4 * (lane + NT * e);
        if (d >= size) continue;
        gng_f32x4 v;
#pragma unroll
        for (int k = 0; k < 4; ++k) v[k] = u[e][k] * scale * wt[e][k] * (GATE_FIRST ? 1.0f : z[e][k]);
        T* o = out + part * size + d;
        if constexpr (sizeof(T) == 4) *(gng_f32x4*)o = v;
        else *(uint2*)o = make_uint2(pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3]));
    }
}

template <typename T, bool GATE_FIRST>
static void launch_group_norm_gate(const float* y, const float* gate, int ldg, const float* w, int shared, const float* skip,
                                   int skip_span, const float* x, int ldx, T* out, int rows, int groups, int size, float eps,
                                   int sigmoid, hipStream_t stream) {
    const bool words = size % 4 == 0 && size <= 4096 && ldg % 4 == 0 && (!skip || (ldx % 4 == 0 && skip_span % 4 == 0 && (uintptr_t)x % 16 == 0)) &&
                       (uintptr_t)y % 16 == 0 && (uintptr_t)gate % 16 == 0 && (uintptr_t)w % 16 == 0 && (uintptr_t)out % (4 * sizeof(T)) == 0;
    const long long parts = (long long)rows * groups;
    // (a step of few rows keeps the blocks of a part each, which spread it over more compute units: from a part for each on)
    if (words && parts >= 256 && parts < 0x7fffffff) {
#define GNGW(NT, E) group_norm_gate_words_kernel<T, GATE_FIRST, NT, E><<<(unsigned)((parts + 256 / NT - 1) / (256 / NT)), 256, 0, stream>>>(y, gate, ldg, w, shared, skip, \
        skip_span, x, ldx, out, groups, size, eps, sigmoid, parts)
        if (size <= 128) GNGW(32, 1);
        else if (size <= 256) GNGW(64, 1);
        else if (size <= 512) GNGW(64, 2);
        else if (size <= 1024) GNGW(256, 1);
        else if (size <= 2048) GNGW(256, 2);
        else GNGW(256, 4);
#undef GNGW
        return;
    }
    const dim3 grid(rows, groups);
    const size_t lds = (size_t)size * sizeof(float);
#define GNG(NT, KEEP) group_norm_gate_kernel<T, GATE_FIRST, NT, KEEP><<<grid, NT, KEEP ? lds : 0, stream>>>(y, gate, ldg, w, shared, skip, skip_span, x, ldx, out, size, eps, sigmoid)
    if (size <= 256) GNG(64, true);
    else if (size <= 2048) GNG(256, true);
    else if (size <= 12288) GNG(1024, true);
    else GNG(1024, false);
#undef GNG
}

extern "C" int cisr_group_norm_gate(const float* y, const float* gate, int ldg, const float* w, int shared, const float* skip,
                                    int skip_span, const float* x, int ldx, void* out, int rows, int groups, int size,
                                    float eps, int gate_first, int sigmoid, int dtype, hipStream_t stream) {
    if (rows <= 0) return 0;
    if (groups <= 0 || groups > 65535 || size <= 0 || (skip && (skip_span <= 0 || !x))) return (int)hipErrorInvalidValue;
    if (dtype == DT_F32) {
        if (gate_first) launch_group_norm_gate<float, true>(y, gate, ldg, w, shared, skip, skip_span, x, ldx, (float*)out, rows, groups, size, eps, sigmoid, stream);
        else launch_group_norm_gate<float, false>(y, gate, ldg, w, shared, skip, skip_span, x, ldx, (float*)out, rows, groups, size, eps, sigmoid, stream);
    } else {
        if (gate_first) launch_group_norm_gate<bf16_t, true>(y, gate, ldg, w, shared, skip, skip_span, x, ldx, (bf16_t*)out, rows, groups, size, eps, sigmoid, stream);
        else launch_group_norm_gate<bf16_t, false>(y, gate, ldg, w, shared, skip, skip_span, x, ldx, (bf16_t*)out, rows, groups, size, eps, sigmoid, stream);
    }
    return CISR_LAUNCH_CHECK();
}
