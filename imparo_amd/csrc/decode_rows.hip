// Products for a step of at most 16 tokens (a decode step's rows), bfloat16 weights, plain or with the work that
// surrounds a product on the residual stream folded in, so that a layer of such a step is a chain of four to six
// launches instead of six to eight:
//
//   * the result may be added to the residual stream in place, and the block leaves the sum of
//     squares of its columns of the new rows: x += y, ssq[block][row] -- no add, and what the next
//     norm needs is there. Told the weight of the norm that reads the stream next, it also leaves
//     the new rows times that weight in bfloat16. A block adds the whole of K (no slices of K over
//     blocks): nothing meets across blocks, so there are no counters and no fences;
//     Where that norm has no statistic (dynamic tanh), the block leaves the rows behind it: every element is its own, and
//     nothing is left for the reader to do;
//   * the first columns may be channels of a causal conv with SiLU behind it: the lane that ends up with a channel's sum has
//     its history and taps by then, and shifts the history;
//   * the activations may be such rows (the stream times a norm's weight, not yet scaled) with the
//     partial sums of squares beside them: the block multiplies each row's result by the row's scale
//     rsqrt(sum / K + eps) at the end, in float32 -- no norm launch.
//
// The reference fuses the same neighbours: add + norm as one op, the gate/up pair with its
// activation (/root/reference/crates/imparo-backend/src/lib.rs:2603-2609, 1835-1869).
//
// Such a product is bound by reading its weights, and a short one by the trips to memory that follow one another. So
// every wave asks for all it needs at once, activations first (they are few and near), then weights, straight into the
// registers that the matrix products read, and waits once; nothing goes through LDS but the waves' sums at the end, which
// are added in wave order. A block takes RT tiles of 16 weight rows, which share the activations of a wave's chunks: with
// one tile every 64 KB of weights (K of 2,048) draw 32 KB of activations of 8 rows through the CU's load path again. Which
// RT, how many waves and chunks a wave: rows_shape. Measured, cold weights, launch behind launch (before: walks along K
// in steps of 128 to 1,024 with the activations through LDS):
//
//   rows, weight                               before      now
//   1, 9,216 by 1,024, gated, scaled           8.3 us      6.8 us
//   8 / 16, 16,384 by 2,048, gated, scaled     17.3 / 17.3 15.4 / 15.9
//   1, 65,536 by 1,024                         32.7        24.9
//   8 / 16, 65,536 by 2,048                    55.9 / 57.2 54.0 / 56.0
//   1, 1,024 by 4,608, 8 slices                6.1         4.5
//   8 / 16, 2,048 by 8,192, 4 slices           10.2 / 10.5 9.2 / 9.8
//   8 / 16, 3,072 by 2,048                     6.5 / 7.4   5.9 / 6.4
//   8 / 16, 2,048 by 2,048, into the stream    5.8 / 6.8   5.4 / 5.9
//   16, 9,216 by 3,072                         24.6        15.3
//   8, 12,288 by 4,608                         26.1        23.6
//   16, 16,384 by 4,096                        41.5        27.6
//   8, 16,384 by 11,008                        69.0        67.7
//
// (a kernel that only reads 8 / 34 / 67 / 134 / 268 MB takes 3.8 / 7.4 / 12.3 / 22 / 48 us).
#include "common.h"

#include <algorithm>
#include <type_traits>
#include "api.h"
#include "rows.h"

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

union RowFrag {
    uint4 u;
    bf16x8 v;
};

#define ROWS_STORE 0
#define ROWS_SWIGLU 1
#define ROWS_RESID 2
#define ROWS_TANH 3          // into the stream, and the rows behind a norm without a statistic
#define ROWS_CONV 4          // the first columns through a causal conv a channel and SiLU
#define ROWS_WAVES 8         // of a block at most
#define ROWS_TURNED 8192     // from this K on blocks start their walks at different places

// ROWS_CONV: columns 0 .. channels - 1 are channels of a causal conv (at most ROWS_TAPS taps, the last one the current row's) whose
// last inputs a request keeps: hist [slots, taps - 1, channels], row r in slot[r], shifted in place by the lane that owns the channel.
#define ROWS_TAPS 4
struct RowsConv {
    const float* w;          // [channels, taps]
    float* hist;
    const int32_t* slot;
    int taps, channels;
};

// K_KIND
#define ROWS_WHOLE 0         // K is a multiple of 128, and every wave has as many chunks of it as its rounds ask for
#define ROWS_UNEVEN 1        // K is a multiple of 128
#define ROWS_RAGGED 2        // any other K: addresses are clamped into the row, and what a chunk has beyond K counts as zeros
#define ROWS_HUGE 3          // K from 2^25 on: the same, with 64-bit offsets inside a block's rows

__device__ __forceinline__ uint4 rows_zero_if(bool out, uint4 v) {
    return make_uint4(out ? 0u : v.x, out ? 0u : v.y, out ? 0u : v.z, out ? 0u : v.w);
}

// Four results of a token, columns n .. n + 3 of N (n a multiple of 4), in one store where rows keep it aligned
template <typename TOut> __device__ __forceinline__ void rows_store(TOut* dst, const float (&v)[4], int n, int N, bool whole) {
    if (whole) {
        if (n >= N) return;
        if constexpr (sizeof(TOut) == 4)
            *reinterpret_cast<float4*>(dst) = make_float4(v[0], v[1], v[2], v[3]);
        else
            *reinterpret_cast<uint2*>(dst) = make_uint2(f32x2_to_bf16x2(v[0], v[1]), f32x2_to_bf16x2(v[2], v[3]));
        return;
    }
#pragma unroll
    for (int i = 0; i < 4; ++i)
        if (n + i < N) store_f32<TOut>(dst, i, v[i]);
}

// CHAINS: sums that a wave's chunks go into by turns; the chains' sums are added in the order of their first chunks.
// RB: weight rows of a tile, 16, 8 or 4 (the other lanes ask for nothing; RT 1). CH: chunks of 128 of K that a wave has in
// flight at once. SCALED: ssq_in is there. With slices (gridDim.y > 1) block (x, y) sums K range [y * k_per, (y+1) * k_per)
// into Y + y * M * N and the consumer adds the slices.
template <typename TOut, int RB, int RT, int CH, int CHAINS, int EPI, int K_KIND, bool SCALED>
__global__ __launch_bounds__(ROWS_WAVES * 64) void k_rows_gemm(
    const bf16_t* __restrict__ X, const float* __restrict__ ssq_in, int n_parts, float eps,
    const bf16_t* __restrict__ W, const float* __restrict__ bias, TOut* __restrict__ Y, float* __restrict__ x_io,
    float* __restrict__ ssq_out, bf16_t* __restrict__ weighted_out, const float* __restrict__ weighted_by,
    const float* __restrict__ tanh_bias, float tanh_alpha, int M, int N, int K_all, int k_per, int rounds, int turned, Epilogue unit,
    RowsConv conv) {
    static_assert(RB == 16 || RT == 1, "half tiles one by one");
    constexpr bool RAGGED = K_KIND == ROWS_RAGGED || K_KIND == ROWS_HUGE;
    extern __shared__ float4 red[];                     // [CHAINS][waves][RT][64]
    __shared__ __attribute__((aligned(16))) float part[ROWS_WAVES * 16];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), waves = blockDim.x >> 6;
    const int r16 = lane & 15, g = lane >> 4;
    const int n0 = blockIdx.x * (RB * RT);
    const int k_lo = blockIdx.y * k_per;
    const int K = min(K_all, k_lo + k_per) - k_lo;      // this block's part of K, re-based to 0
    Y += (size_t)blockIdx.y * M * N;
    if (blockIdx.y > 0) bias = nullptr;                 // the bias belongs to one slice only
    const int token = min(r16, M - 1);
    const int n_chunks = (K + 127) / 128;
    // uniform bases and 32-bit byte offsets inside a block's rows: a load costs next to no address arithmetic
    typedef typename std::conditional<K_KIND == ROWS_HUGE, size_t, unsigned>::type Offset;
    const bf16_t* xbase = X + k_lo;
    const bf16_t* wbase = W + (size_t)n0 * K_all + k_lo;
    const Offset xoff = (Offset)token * (unsigned)K_all * 2u;
    Offset woff[RT];
#pragma unroll
    for (int t = 0; t < RT; ++t) woff[t] = (Offset)min(t * 16 + (r16 & (RB - 1)), N - 1 - n0) * (unsigned)K_all * 2u;
    RowFrag x[CH][4], w[RT][CH][4];
    // This wave's chunks are first, first + waves, ...: CH of them a round. No load under a branch (the compiler would wait
    // for every load in flight at the next use of any): past the last chunk the last one again, which no product reads.
    // A long walk starts at a round that goes by the block's place: rows of a long K lie so far apart that blocks in step keep
    // asking the same few channels (8 rows of 16,384 by 11,008 82 us in step, 68 so; of 8,192 by 16,384 68 and 53). The
    // place is hashed, as rounds that follow the row's number undo what the address's own hash does (8 rows of 8,192 by
    // 8,192: in step 32 us, hashed 28, by the row 46).
    const int turn = waves * CH;
    int round = (int)__umulhi((unsigned)(n0 / 64) * 2654435761u, (unsigned)turned);      // (no branch in front of the loads)
    auto at = [&](const bf16_t* base, Offset row, int chunk, int s) __attribute__((always_inline)) {
        if constexpr (RAGGED)
            return reinterpret_cast<const uint4*>(reinterpret_cast<const char*>(base) +
                                                  (row + (Offset)min(chunk * 128 + s * 32 + g * 8, K - 8) * 2u));
        else
            return reinterpret_cast<const uint4*>(reinterpret_cast<const char*>(base + chunk * 128) + (row + g * 16) + s * 64);
    };
    // (A tile's chunks one after the other: chunk after chunk over all tiles, every block would read the first half of its
    // rows and then the second, at any time half of the memory's channels: 8 rows of 16,384 by 2,048 15.1 us and not 13.9.)
    auto ask_some = [&](int first, int n) __attribute__((always_inline)) {     // (n: known when this is compiled)
#pragma unroll
        for (int j = 0; j < n; ++j)
#pragma unroll
            for (int s = 0; s < 4; ++s) x[j][s].u = *at(xbase, xoff, min(first + j * waves, n_chunks - 1), s);
#pragma unroll
        for (int t = 0; t < RT; ++t)
#pragma unroll
            for (int j = 0; j < n; ++j)
#pragma unroll
                for (int s = 0; s < 4; ++s) {
                    // (lanes of weight rows beyond RB ask for nothing: their rows of the tile are nobody's)
                    if (RB < 16) w[t][j][s].u = make_uint4(0u, 0u, 0u, 0u);
                    if (RB == 16 || r16 < RB) w[t][j][s].u = *at(wbase, woff[t], min(first + j * waves, n_chunks - 1), s);
                }
    };
    auto ask = [&](int first) __attribute__((always_inline)) {
        if constexpr (CH > 1 && K_KIND != ROWS_WHOLE) {      // (a wave may have a chunk less than others)
            if (first + (CH - 1) * waves < n_chunks) ask_some(first, CH);
            else ask_some(first, CH - 1);
        } else {
            ask_some(first, CH);
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    // the rows' sums of squares first: they are added up while the weights are on their way
    RowsSsq early;
    if (SCALED) rows_ssq_ask(early, ssq_in, n_parts, 0);
    __builtin_amdgcn_sched_barrier(0);
    ask(wave + round * turn);
    if (SCALED) rows_ssq_share(part, early, ssq_in, n_parts);
    // needed when the walk is over: what the finishing lanes add to
    float x_old[4] = {0.f, 0.f, 0.f, 0.f}, by[4] = {0.f, 0.f, 0.f, 0.f}, plus[4] = {0.f, 0.f, 0.f, 0.f};
    if ((EPI == ROWS_RESID || EPI == ROWS_TANH) && wave == 0 && g * 4 < RB && r16 < M) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int n = min(n0 + g * 4 + i, N - 1);
            x_old[i] = x_io[(size_t)r16 * N + n];
            if (weighted_by) by[i] = weighted_by[n];
            if (EPI == ROWS_TANH && tanh_bias) plus[i] = tanh_bias[n];
        }
    }
    // (and what a conv's channels had before, for the tile that this wave finishes first)
    float taps_of[EPI == ROWS_CONV ? 4 : 1][ROWS_TAPS], old[EPI == ROWS_CONV ? ROWS_TAPS - 1 : 1][4];
    auto ask_conv = [&](int t) __attribute__((always_inline)) {
        const int n = n0 + t * 16 + g * 4, history = conv.taps - 1;
        if (n >= conv.channels || r16 >= M) return;
        const float* hist = conv.hist + (size_t)conv.slot[r16] * history * conv.channels + n;
#pragma unroll
        for (int i = 0; i < ROWS_TAPS - 1; ++i)
#pragma unroll
            for (int j = 0; j < 4; ++j) old[EPI == ROWS_CONV ? i : 0][j] = i < history ? hist[(size_t)i * conv.channels + j] : 0.f;
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
            for (int i = 0; i < ROWS_TAPS; ++i)
                taps_of[EPI == ROWS_CONV ? j : 0][i] = i < conv.taps ? conv.w[(size_t)(n + j) * conv.taps + i] : 0.f;
    };
    if (EPI == ROWS_CONV && wave < RT) ask_conv(wave);
    f32x4 acc[CHAINS][RT];
#pragma unroll
    for (int c = 0; c < CHAINS; ++c)
#pragma unroll
        for (int t = 0; t < RT; ++t) acc[c][t] = f32x4{0.f, 0.f, 0.f, 0.f};
    int left = rounds;                                   // (at least one)
    do {
        const int first = wave + round * turn;
        if constexpr (RAGGED) {                              // what the last steps of 32 have beyond K counts as zeros
#pragma unroll
            for (int j = 0; j < CH; ++j)
#pragma unroll
                for (int s = 0; s < 4; ++s) {
                    const int k0 = (first + j * waves) * 128 + s * 32;
                    if (k0 >= K || k0 + 32 <= K) continue;
                    x[j][s].u = rows_zero_if(k0 + g * 8 >= K, x[j][s].u);
#pragma unroll
                    for (int t = 0; t < RT; ++t) w[t][j][s].u = rows_zero_if(k0 + g * 8 >= K, w[t][j][s].u);
                }
        }
        auto multiply = [&](int odd) __attribute__((always_inline)) {       // (a wave's chunks by turns into its chains)
#pragma unroll
            for (int t = 0; t < RT; ++t)
#pragma unroll
                for (int j = 0; j < CH; ++j) {
                    if (first + j * waves >= n_chunks) continue;
                    f32x4& sum = acc[(j + odd) % CHAINS][t];
#pragma unroll
                    for (int s = 0; s < 4; ++s) {
                        if (RAGGED && (first + j * waves) * 128 + s * 32 >= K) continue;
                        sum = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[t][j][s].v, x[j][s].v, sum, 0, 0, 0);
                    }
                }
        };
        if (CHAINS == 2 && CH % 2 == 1 && (round & 1)) multiply(1);
        else multiply(0);
        round = round + 1 == rounds ? 0 : round + 1;
        if (left > 1 && wave + round * turn < n_chunks) ask(wave + round * turn);
    } while (--left > 0);
    // into the stream in one piece stands for slices of K and may not be further from 64 bits than they are: a wave's chains are
    // added in pairs here, the waves' sums in pairs below
    if constexpr (EPI == ROWS_TANH) {
#pragma unroll
        for (int c = 0; c + 1 < CHAINS; c += 2) acc[c][0] += acc[c + 1][0];
        if constexpr (CHAINS > 2) acc[0][0] += acc[2][0];
    }
    constexpr int LEFT = EPI == ROWS_TANH ? 1 : CHAINS;      // sums a wave leaves
#pragma unroll
    for (int c = 0; c < LEFT; ++c)
#pragma unroll
        for (int t = 0; t < RT; ++t)
            red[((c * waves + wave) * RT + t) * 64 + lane] = make_float4(acc[c][t][0], acc[c][t][1], acc[c][t][2], acc[c][t][3]);
    __syncthreads();
    if (g * 4 >= RB) return;
    // D layout of the 16x16 tile: lane holds column lane % 16 (a token), rows 4 * (lane / 16) + i (weight rows)
    for (int t = wave; t < RT; t += waves) {
        float4 sums[LEFT * ROWS_WAVES];
#pragma unroll
        for (int q = 0; q < LEFT * ROWS_WAVES; ++q) sums[q] = red[(min(q, LEFT * waves - 1) * RT + t) * 64 + lane];
        const float scale = SCALED ? rows_scale(part, token, K, eps) : 1.f;
        if constexpr (EPI == ROWS_TANH) {
#pragma unroll
            for (int w = 1; w < ROWS_WAVES; ++w)
                if (w >= waves) sums[w] = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
            for (int half = ROWS_WAVES / 2; half > 0; half /= 2)
#pragma unroll
                for (int w = 0; w < half; ++w)
                    sums[w].x += sums[w + half].x, sums[w].y += sums[w + half].y, sums[w].z += sums[w + half].z, sums[w].w += sums[w + half].w;
        }
        float v[4] = {sums[0].x, sums[0].y, sums[0].z, sums[0].w};
        if constexpr (EPI != ROWS_TANH) {
#pragma unroll
            for (int q = 1; q < CHAINS * ROWS_WAVES; ++q)
                if (q < CHAINS * waves) v[0] += sums[q].x, v[1] += sums[q].y, v[2] += sums[q].z, v[3] += sums[q].w;
        }
        const int n = n0 + t * 16 + g * 4;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            // each step rounded on its own (no fused multiply-add), so that every epilogue gives the same bits
            if (SCALED) v[i] = __fmul_rn(v[i], scale);
            if (bias && n + i < N) v[i] = __fadd_rn(v[i], bias[n + i]);
        }
        const bool live = r16 < M;
        if (EPI == ROWS_SWIGLU) {
            if (!live) continue;
            const float a = gated_mul_fast(unit, v[0], v[1]), b = gated_mul_fast(unit, v[2], v[3]);
            TOut* dst = Y + (size_t)r16 * (N / 2) + n / 2;
            if (n + 3 < N && N % 4 == 0 && ((uintptr_t)Y & (2 * sizeof(TOut) - 1)) == 0) {
                if constexpr (sizeof(TOut) == 4)
                    *reinterpret_cast<float2*>(dst) = make_float2(a, b);
                else
                    *reinterpret_cast<uint32_t*>(dst) = f32x2_to_bf16x2(a, b);
            } else {
                if (n + 1 < N) store_f32<TOut>(dst, 0, a);
                if (n + 3 < N) store_f32<TOut>(dst, 1, b);
            }
        } else if (EPI == ROWS_CONV) {
            if (!live) continue;
            if (n < conv.channels) {                     // (channels are a multiple of 4)
                if (t != wave) ask_conv(t);
                const int history = conv.taps - 1;
                float* hist = conv.hist + (size_t)conv.slot[r16] * history * conv.channels + n;
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const float now = v[j];
                    float sum = 0.f, last = taps_of[EPI == ROWS_CONV ? j : 0][0];
#pragma unroll
                    for (int i = 0; i < ROWS_TAPS - 1; ++i) {          // (what lies past the history is zero)
                        const int at = EPI == ROWS_CONV ? i : 0;
                        sum = fmaf(i < history ? taps_of[EPI == ROWS_CONV ? j : 0][i] : 0.f, old[at][j], sum);
                        last = i + 1 == history ? taps_of[EPI == ROWS_CONV ? j : 0][i + 1] : last;
                        if (i < history)
                            hist[(size_t)i * conv.channels + j] = i + 1 < history ? old[EPI == ROWS_CONV && i + 1 < ROWS_TAPS - 1 ? i + 1 : 0][j] : now;
                    }
                    const float z = fmaf(last, now, sum);
                    v[j] = z / (1.0f + expf(-z));
                }
            }
            rows_store<TOut>(Y + (size_t)r16 * N + n, v, n, N, N % 4 == 0 && ((uintptr_t)Y & (4 * sizeof(TOut) - 1)) == 0);
        } else if (EPI == ROWS_STORE) {
            if (live) rows_store<TOut>(Y + (size_t)r16 * N + n, v, n, N, N % 4 == 0 && ((uintptr_t)Y & (4 * sizeof(TOut) - 1)) == 0);
        } else {
            // the stream takes the result; the block leaves the sum of squares of its columns
            float sq = 0.f;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                if (live && n + i < N) {
                    const float xn = __fadd_rn(x_old[i], v[i]);
                    x_io[(size_t)r16 * N + n + i] = xn;
                    sq = fmaf(xn, xn, sq);
                    if (weighted_out)
                        weighted_out[(size_t)r16 * N + n + i] =
                            f32_to_bf16(EPI == ROWS_TANH ? fmaf(tanhf(tanh_alpha * xn), by[i], plus[i]) : xn * by[i]);
                }
            }
            if (EPI == ROWS_TANH) continue;
            sq += __shfl_xor(sq, 16, WAVE);             // the two lanes of a token sit 16 apart
            if (g == 0) ssq_out[(size_t)blockIdx.x * ROWS_PARTS + r16] = sq;
        }
    }
}

// How a product is shared out, measured against the kernels before over 2,500 random forms of 1 to 16 rows (1.25 times as
// fast on average, 1 in 100 slower by more than 3 % and 0.1 us: K below 540 and no multiple of 128, by 0.2 us at the most, and
// into the stream over K of 14,336, by 9 %).
//
// Waves: as many as there are chunks, eight at most. Chains: two a wave from 17 chunks on (into the stream from 33), where the
// kernels before had sixteen sums, too. The more chains a column is summed in, the nearer it is to 64 bits: fewer waves with
// more chunks each were 1.12e-7 off at K of 1,152, where eight are 8.8e-8, and eight with three chunks in one chain 1.21e-7 at
// 3,072, in two 1.14e-7. Waves, chains and where a walk starts do not go by the rows: a row has the same bits among others
// and by itself. (Weights of 12,288 rows and more had one chain a column, 3.4e-7 at 3,072; one a wave, 1.2e-7, saves registers.)
//
// Tiles a block: as many (up to four) as still load the CUs evenly, as they share the activations: 16 rows of 9,216 by 3,072
// three tiles (192 blocks) 15.2 us, two (288 blocks, some CUs with two) 21.5; of 24,576 by 4,608 three (two blocks a CU) 47.5,
// four 54.1. One or two chunks of K have nothing to share, and a block a tile is there sooner (8 rows of 9,216 by 128: one tile
// 3.4 us, three 4.2); nor do short slices of K (1,024 by 4,608 in eight) or up to four rows of a weight of many rows (1 row of
// 65,536 by 1,536: one 38.7, four 41.1), unless their walk is turned, for that goes by the block.
//
// Chunks in flight: all that a wave has, up to four, where a block is alone on its CU. With three or four tiles and in a walk
// of more than one round one, or two where rows lie a multiple of 4 KB apart and every wave has whole pairs: blocks of few
// registers share a CU, and one's loads cover the other's waits (16 rows of 65,536 by 4,608: one 115 us, two 122, four 160;
// of 16,384 by 4,096: one 31.1, two 27.9, four 31.5: rows that far apart lie on the same few channels, and longer pieces of
// each spread the load).
//
// Turned: 16 rows of 8,192 by 8,192 in step 35.0 us, turned 29.5; of 12,288 by 5,504 42.3 and 34.3, as whenever rows are an odd
// multiple of 256 or 512 bytes apart; of 6,144 by 4,608 16.3 and 17.6, so not below 8,192 otherwise.
struct RowsShape {
    int waves, ch, rt, chains;
    bool turned;
};
static RowsShape rows_shape(int m, int n, int k, int k_per, int slices, int rb) {
    const int chunks = (k_per + 127) / 128, waves = std::min(chunks, ROWS_WAVES), a_wave = (chunks + waves - 1) / waves;
    const bool ragged = k % 128 != 0;
    RowsShape sh{waves, 1, 1, 1, k >= ROWS_TURNED || (chunks > 32 && !ragged && k % 512 != 0)};
    // a whole number of pairs of chunks for every wave, and rows a multiple of 4 KB apart
    const int pairs = k % 2048 == 0 && k_per % (256 * waves) == 0 && k % k_per == 0 ? 2 : 1;
    bool spread = a_wave > 4;                            // one or two chunks at a time
    if (rb == 16) {
        const long long tiles = (long long)((n + 15) / 16) * slices;
        auto a_cu = [&](int rt) { return ((tiles + rt - 1) / rt + 255) / 256 * rt; };
        const long long least = a_cu(1);
        for (int rt = 2; rt <= 4; ++rt)
            if (a_cu(rt) * 6 <= least * 7) sh.rt = rt;
        if (chunks <= 2 && tiles <= 1024) sh.rt = 1;
        if (slices > 1 && tiles <= 512 && chunks <= 8) sh.rt = 1;
        // (a launch holds fewer than 2^32 threads along x: a tile a block of several waves would pass that at 2^29 rows)
        if (m <= 4 && tiles > 1024 && tiles < (1 << 22) && !sh.turned) sh.rt = 1;
        if (tiles > 768 && a_wave > 2) spread = true;
        if (m <= 4 && tiles > 1024) spread = true;
        if (sh.rt > 2 && !(sh.rt == 3 && a_wave == 3 && tiles <= 768 && !ragged)) spread = true;
        if (slices > 1 && a_wave == 4 && pairs == 2) spread = true;
        sh.ch = spread ? pairs : a_wave;
        sh.chains = chunks > 2 * ROWS_WAVES && (n < 12288 || sh.ch > 2) ? 2 : 1;
    } else {
        // half tiles: one chunk at a time where a CU has several blocks, else two of four, which leaves room for a second block
        if (n > 4096 || (n > 2048 && a_wave == 4)) sh.ch = spread ? pairs : 1;
        else sh.ch = spread || (a_wave == 4 && pairs == 2) ? pairs : a_wave;
        sh.chains = chunks > 4 * ROWS_WAVES ? 2 : 1;
    }
    return sh;
}

struct RowsCall {
    const bf16_t* x;
    const float* ssq_in;
    int n_parts;
    float eps;
    const bf16_t* w;
    const float* bias;
    void* y;
    float* x_io;
    float* ssq_out;
    bf16_t* weighted_out;
    const float* weighted_by;
    const float* tanh_bias;
    float tanh_alpha;
    int m, n, k, slices;
    Epilogue unit;
    RowsConv conv;
};

template <typename TOut, int RB, int EPI, bool SCALED>
static void rows_launch_as(const RowsCall& c, hipStream_t s) {
    const int k_per = ((c.k + c.slices - 1) / c.slices + 127) / 128 * 128;
    const bool huge = c.k >= (1 << 25), ragged = c.k % 128 != 0 || huge;      // (byte offsets inside 64 rows stay in 32 bits)
    RowsShape sh = rows_shape(c.m, c.n, c.k, std::min(k_per, c.k), c.slices, RB);
    if (EPI == ROWS_CONV && sh.rt > 2) sh.rt = 2;
    if (huge) sh.rt = 1, sh.ch = 1, sh.chains = 1;
    const dim3 grid((unsigned)((c.n + (long long)RB * sh.rt - 1) / (RB * sh.rt)), (unsigned)((c.k + k_per - 1) / k_per));
    const int rounds = ((std::min(k_per, c.k) + 127) / 128 + sh.waves * sh.ch - 1) / (sh.waves * sh.ch);
    const int turned = sh.turned ? rounds : 0;
    const bool even = c.k % (128 * sh.waves * sh.ch) == 0 && k_per % (128 * sh.waves * sh.ch) == 0;
    const size_t lds = (size_t)sh.chains * sh.waves * sh.rt * 64 * sizeof(float4);          // (48 KB at most)
#define ROWS_GO(RT, CH, CHAINS, KIND)                                                                                \
    k_rows_gemm<TOut, RB, RT, CH, CHAINS, EPI, KIND, SCALED><<<grid, sh.waves * 64, lds, s>>>(                         \
        c.x, c.ssq_in, c.n_parts, c.eps, c.w, c.bias, (TOut*)c.y, c.x_io, c.ssq_out, c.weighted_out, c.weighted_by, \
        c.tanh_bias, c.tanh_alpha, c.m, c.n, c.k, k_per, rounds, turned, c.unit, c.conv)
#define ROWS_CHAINS(RT, CH, KIND)                                                                                    \
    do {                                                                                                             \
        if (sh.chains == 2) ROWS_GO(RT, CH, 2, KIND);                                                                \
        else ROWS_GO(RT, CH, 1, KIND);                                                                               \
    } while (0)
// (three and four chunks a wave are a walk of one round: two chains, but into the stream)
#define ROWS_LONG(RT, CH, KIND)                                                                                      \
    do {                                                                                                             \
        if constexpr (RB == 8) ROWS_CHAINS(RT, CH, KIND);                                                            \
        else ROWS_GO(RT, CH, 2, KIND);                                                                               \
    } while (0)
#define ROWS_CH(RT)                                                                                                  \
    do {                                                                                                             \
        if (sh.ch == 1 && ragged) ROWS_CHAINS(RT, 1, ROWS_RAGGED);                                                   \
        else if (sh.ch == 1) ROWS_CHAINS(RT, 1, ROWS_WHOLE);                                                         \
        else if (sh.ch == 2 && ragged) ROWS_GO(RT, 2, 1, ROWS_RAGGED);                                               \
        else if (sh.ch == 2 && even) ROWS_CHAINS(RT, 2, ROWS_WHOLE);                                                 \
        else if (sh.ch == 2) ROWS_GO(RT, 2, 1, ROWS_UNEVEN);                                                         \
        else if (sh.ch == 3 && ragged) ROWS_LONG(RT, 3, ROWS_RAGGED);                                                \
        else if (sh.ch == 3 && even) ROWS_LONG(RT, 3, ROWS_WHOLE);                                                   \
        else if (sh.ch == 3) ROWS_LONG(RT, 3, ROWS_UNEVEN);                                                          \
        else if (ragged) ROWS_LONG(RT, 4, ROWS_RAGGED);                                                              \
        else if (even) ROWS_LONG(RT, 4, ROWS_WHOLE);                                                                 \
        else ROWS_LONG(RT, 4, ROWS_UNEVEN);                                                                          \
    } while (0)
    if (huge) {
        ROWS_GO(1, 1, 1, ROWS_HUGE);
    } else if constexpr (RB == 8) {
        ROWS_CH(1);
    } else if (sh.rt == 1) {
        ROWS_CH(1);
    } else if (EPI == ROWS_CONV || sh.rt == 2) {
        ROWS_CH(2);
    } else if constexpr (EPI == ROWS_CONV) {
    } else if (sh.rt == 3) {
        if (ragged) ROWS_CHAINS(3, 1, ROWS_RAGGED);
        else if (sh.ch == 1) ROWS_CHAINS(3, 1, ROWS_WHOLE);
        else if (sh.ch == 2) ROWS_CHAINS(3, 2, ROWS_WHOLE);
        else if (even) ROWS_GO(3, 3, 2, ROWS_WHOLE);
        else ROWS_GO(3, 3, 2, ROWS_UNEVEN);
    } else {
        if (ragged) ROWS_GO(4, 1, 1, ROWS_RAGGED);
        else if (sh.ch == 1) ROWS_GO(4, 1, 1, ROWS_WHOLE);
        else ROWS_GO(4, 2, 1, ROWS_WHOLE);
    }
#undef ROWS_LONG
#undef ROWS_CHAINS
#undef ROWS_CH
#undef ROWS_GO
}

// A sum for every chunk a wave has in flight (up to four; K of 4,096 is one round), added in pairs: errors of 1,024 weight rows
// against 64 bits 7.7e-8 over K of 1,024 and 8.7e-8 over 3,072, where a chain a wave, added one after the other, had 8.3e-8 and
// 1.2e-7 and slices of K that the norm adds have 7.8e-8 and 8.7e-8.
template <int RB, int CH>
static void rows_launch_tanh(const RowsCall& c, const RowsShape& sh, hipStream_t s) {
    const int rounds = ((c.k + 127) / 128 + sh.waves * CH - 1) / (sh.waves * CH), turned = sh.turned ? rounds : 0;
    const dim3 grid((unsigned)((c.n + RB - 1LL) / RB));
    const size_t lds = (size_t)sh.waves * 64 * sizeof(float4);
#define ROWS_GO(KIND)                                                                                                  \
    k_rows_gemm<float, RB, 1, CH, CH, ROWS_TANH, KIND, false><<<grid, sh.waves * 64, lds, s>>>(                          \
        c.x, nullptr, 0, 0.f, c.w, c.bias, nullptr, c.x_io, nullptr, c.weighted_out, c.weighted_by, c.tanh_bias, c.tanh_alpha, \
        c.m, c.n, c.k, c.k, rounds, turned, c.unit, c.conv)
    if (c.k % 128) ROWS_GO(ROWS_RAGGED);
    else if (CH == 1 || c.k % (128 * sh.waves * CH) == 0) ROWS_GO(ROWS_WHOLE);
    else ROWS_GO(ROWS_UNEVEN);
#undef ROWS_GO
}

template <typename TOut, int RB, int EPI>
static void rows_launch(const RowsCall& c, hipStream_t s) {
    if (c.ssq_in) rows_launch_as<TOut, RB, EPI, true>(c, s);
    else rows_launch_as<TOut, RB, EPI, false>(c, s);
}

int imparo_few_rows(const bf16_t* x, const bf16_t* w, const float* bias, void* y, int out_dtype, int m, int n, int k,
                    const Epilogue& epilogue, int slices, const float* ssq_in, int n_parts, float eps, hipStream_t s) {
    const RowsCall c{x, ssq_in, n_parts, eps, w, bias, y, nullptr, nullptr, nullptr, nullptr, nullptr, 0.f, m, n, k, slices,
                     epilogue, {}};
    if (m <= 0 || m > ROWS_MAX || n <= 0 || k < 8 || k % 8 || slices < 1) return IMPARO_BAD_ARGUMENT;
    if (epilogue == EPI_SWIGLU && out_dtype == IMPARO_BF16)
        rows_launch<bf16_t, 16, ROWS_SWIGLU>(c, s);
    else if (epilogue == EPI_SWIGLU)
        rows_launch<float, 16, ROWS_SWIGLU>(c, s);
    else if (out_dtype == IMPARO_BF16)
        rows_launch<bf16_t, 16, ROWS_STORE>(c, s);
    else
        rows_launch<float, 16, ROWS_STORE>(c, s);
    return launch_status();
}

// blocks of a ROWS_RESID product with `n` weight rows: the partial sums of squares it leaves
extern "C" int imparo_rows_parts(int n) { return (n + 7) / 8; }

extern "C" int imparo_rows_gemm(const void* x, const float* ssq_in, int n_parts, float eps, const void* w,
                                const float* bias, void* y, int out_dtype, float* x_io, float* ssq_out,
                                void* weighted_out, const float* weighted_by, int m, int n, int k, int epilogue,
                                imparo_stream stream) {
    if (!x || !w || m < 0 || m > ROWS_MAX || n <= 0 || k <= 0 || k % 8 != 0) return IMPARO_BAD_ARGUMENT;
    if (ssq_in && (n_parts <= 0 || !(eps > 0.f))) return IMPARO_BAD_ARGUMENT;
    if (((uintptr_t)w & 15) || ((uintptr_t)x & 15)) return IMPARO_BAD_ARGUMENT;
    if (epilogue == ROWS_RESID) {
        if (!x_io || !ssq_out || ((weighted_out == nullptr) != (weighted_by == nullptr))) return IMPARO_BAD_ARGUMENT;
    } else if (epilogue == ROWS_STORE || epilogue == ROWS_SWIGLU) {
        if (!y || (out_dtype != IMPARO_F32 && out_dtype != IMPARO_BF16)) return IMPARO_BAD_ARGUMENT;
        if (epilogue == ROWS_SWIGLU && n % 2 != 0) return IMPARO_BAD_ARGUMENT;
    } else {
        return IMPARO_BAD_ARGUMENT;
    }
    if (m == 0) return IMPARO_OK;
    hipStream_t s = (hipStream_t)stream;
    const bf16_t* xb = (const bf16_t*)x;
    const bf16_t* wb = (const bf16_t*)w;
    bf16_t* wo = (bf16_t*)weighted_out;
    if (epilogue == ROWS_RESID) {
        rows_launch<float, 8, ROWS_RESID>(RowsCall{xb, ssq_in, n_parts, eps, wb, bias, nullptr, x_io, ssq_out, wo, weighted_by, nullptr,
                                                   0.f, m, n, k, 1, Epilogue(EPI_NONE), {}}, s);
        return launch_status();
    }
    return imparo_few_rows(xb, wb, bias, y, out_dtype, m, n, k, Epilogue(epilogue == ROWS_SWIGLU ? EPI_SWIGLU : EPI_NONE), 1, ssq_in,
                           n_parts, eps, s);
}

extern "C" int imparo_rows_gemm_conv(const void* x, const void* w, float* y, const float* conv_w, float* hist, const int32_t* slot,
                                     int taps, int channels, int m, int n, int k, imparo_stream stream) {
    if (!x || !w || !y || !conv_w || !slot || m < 0 || m > ROWS_MAX || n <= 0 || k <= 0 || k % 8 != 0 || k >= (1 << 25))
        return IMPARO_BAD_ARGUMENT;
    if (taps < 1 || taps > ROWS_TAPS || (taps > 1 && !hist) || channels < 0 || channels > n || channels % 4)
        return IMPARO_BAD_ARGUMENT;
    if (((uintptr_t)w & 15) || ((uintptr_t)x & 15)) return IMPARO_BAD_ARGUMENT;
    if (m == 0) return IMPARO_OK;
    rows_launch_as<float, 16, ROWS_CONV, false>(
        RowsCall{(const bf16_t*)x, nullptr, 0, 0.f, (const bf16_t*)w, nullptr, y, nullptr, nullptr, nullptr, nullptr, nullptr, 0.f, m, n,
                 k, 1, Epilogue(EPI_NONE), RowsConv{conv_w, hist, slot, taps, channels}},
        (hipStream_t)stream);
    return launch_status();
}

extern "C" int imparo_rows_gemm_tanh(const void* x, const void* w, const float* bias, float* x_io, void* out, float alpha,
                                     const float* norm_w, const float* norm_b, int m, int n, int k, imparo_stream stream) {
    if (!x || !w || !x_io || m < 0 || m > ROWS_MAX || n <= 0 || k <= 0 || k % 8 != 0) return IMPARO_BAD_ARGUMENT;
    if ((out != nullptr) != (norm_w != nullptr) || (out != nullptr) != (norm_b != nullptr)) return IMPARO_BAD_ARGUMENT;
    if (((uintptr_t)w & 15) || ((uintptr_t)x & 15) || k >= (1 << 25)) return IMPARO_BAD_ARGUMENT;
    if (m == 0) return IMPARO_OK;
    const RowsCall c{(const bf16_t*)x, nullptr, 0, 0.f, (const bf16_t*)w, bias, nullptr, x_io, nullptr, (bf16_t*)out, norm_w, norm_b,
                     alpha, m, n, k, 1, Epilogue(EPI_NONE), {}};
    const RowsShape sh = rows_shape(m, n, k, k, 1, 8);
    const int a_wave = ((k + 127) / 128 + sh.waves - 1) / sh.waves;
    hipStream_t s = (hipStream_t)stream;
    // four weight rows a block while those make no more blocks than CUs: 4 rows of 1,024 by 3,072 5.9 -> 5.5 us, by 1,024 4.1 -> 3.8; of
    // 1,536 by 3,072 6.3 -> 8.8
#define ROWS_TANH_GO(RB)                                     \
    do {                                                     \
        if (a_wave == 1) rows_launch_tanh<RB, 1>(c, sh, s);  \
        else if (a_wave == 2) rows_launch_tanh<RB, 2>(c, sh, s); \
        else if (a_wave == 3) rows_launch_tanh<RB, 3>(c, sh, s); \
        else rows_launch_tanh<RB, 4>(c, sh, s);              \
    } while (0)
    if (n <= 1024) ROWS_TANH_GO(4);
    else ROWS_TANH_GO(8);
#undef ROWS_TANH_GO
    return launch_status();
}

// Asks the runtime about one kernel of this file, which makes it load the file's code onto the
// current device (it loads a file's kernels when one of them is first used; a stream under capture
// cannot do that).
int imparo_load_code_decode_rows() {
    hipFuncAttributes attributes;
    return hipFuncGetAttributes(&attributes, reinterpret_cast<const void*>(&k_rows_gemm<float, 8, 1, 1, 1, ROWS_RESID, ROWS_WHOLE, false>)) ==
                   hipSuccess
               ? IMPARO_OK
               : IMPARO_LAUNCH_FAILED;
}
