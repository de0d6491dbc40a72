// Products for a step of at most 16 tokens (a decode step's rows), bfloat16 weights, plain or with the work that
// surrounds a product on the residual stream folded in, so that a layer of such a step is a chain of four to six
// launches instead of six to eight:
//
//   * the result may be added to the residual stream in place, and the block leaves the sum of
//     squares of its columns of the new rows: x += y, ssq[block][row] -- no add, and what the next
//     norm needs is there. Told the weight of the norm that reads the stream next, it also leaves
//     the new rows times that weight in bfloat16. A block adds the whole of K (no slices of K over
//     blocks): nothing meets across blocks, so there are no counters and no fences;
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
//   rows, weight (gated unless said)      before      now
//   1, 9,216 by 1,024, scaled             7.9 us      6.5 us
//   8, 16,384 by 2,048, scaled            16.0        13.9
//   1, 65,536 by 1,024, plain             31.4        23.7
//   8, 65,536 by 2,048, plain             51.8        51.2
//   1, 1,024 by 4,608, 8 slices           6.0         4.5
//   8, 2,048 by 8,192, 4 slices           9.6         8.8
//   8, 3,072 by 2,048, plain              6.4         5.7
//   8, 2,048 by 2,048, into the stream    5.8         5.4
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
#define ROWS_WAVES 8         // of a block at most

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
// RB: weight rows of a tile, 16 or 8 (the other lanes ask for nothing; RT 1). CH: chunks of 128 of K that a wave has in
// flight at once. RAGGED: K is no multiple of 128, or not all slices are alike: addresses are clamped into the row and
// what lies beyond K counts as zeros. With slices (gridDim.y > 1) block (x, y) sums K range [y * k_per, (y+1) * k_per) into
// Y + y * M * N and the consumer adds the slices.
template <typename TOut, int RB, int RT, int CH, int CHAINS, int EPI, bool RAGGED>
__global__ __launch_bounds__(ROWS_WAVES * 64) void k_rows_gemm(
    const bf16_t* __restrict__ X, const float* __restrict__ ssq_in, int n_parts, float eps,
    const bf16_t* __restrict__ W, const float* __restrict__ bias, TOut* __restrict__ Y, float* __restrict__ x_io,
    float* __restrict__ ssq_out, bf16_t* __restrict__ weighted_out, const float* __restrict__ weighted_by, int M, int N,
    int K_all, int k_per, Epilogue unit) {
    static_assert(RB == 16 || RT == 1, "half tiles one by one");
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
    // uniform bases and 32-bit offsets inside a block's rows: a load costs no address arithmetic (RAGGED: any K)
    typedef typename std::conditional<RAGGED, size_t, unsigned>::type Offset;
    const bf16_t* xbase = X + k_lo;
    const bf16_t* wbase = W + (size_t)n0 * K_all + k_lo;
    const Offset xoff = (Offset)token * (unsigned)K_all;
    Offset woff[RT];
#pragma unroll
    for (int t = 0; t < RT; ++t) woff[t] = (Offset)min(t * 16 + (r16 & (RB - 1)), N - 1 - n0) * (unsigned)K_all;
    RowFrag x[CH][4], w[RT][CH][4];
    // This wave's chunks are first, first + waves, ...: CH of them a round. No load under a branch (the compiler would wait
    // for every load in flight at the next use of any): past the last chunk the last one again, which no product reads.
    auto at = [&](const bf16_t* base, Offset row, int chunk, int s) __attribute__((always_inline)) {
        if constexpr (RAGGED)
            return reinterpret_cast<const uint4*>(base + row + min(chunk * 128 + s * 32 + g * 8, K - 8));
        else
            return reinterpret_cast<const uint4*>(reinterpret_cast<const char*>(base + chunk * 128) + (row + g * 8) * 2u + s * 64);
    };
    // (A tile's chunks one after the other: chunk after chunk over all tiles, every block would read the first half of its
    // rows and then the second, at any time half of the memory's channels: 8 rows of 16,384 by 2,048 15.1 us and not 13.9.)
    auto ask = [&](int first) __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < CH; ++j)
#pragma unroll
            for (int s = 0; s < 4; ++s) x[j][s].u = *at(xbase, xoff, min(first + j * waves, n_chunks - 1), s);
#pragma unroll
        for (int t = 0; t < RT; ++t)
#pragma unroll
            for (int j = 0; j < CH; ++j)
#pragma unroll
                for (int s = 0; s < 4; ++s) {
                    // (lanes of weight rows beyond RB ask for nothing: their rows of the tile are nobody's)
                    if (RB < 16) w[t][j][s].u = make_uint4(0u, 0u, 0u, 0u);
                    if (RB == 16 || r16 < RB) w[t][j][s].u = *at(wbase, woff[t], min(first + j * waves, n_chunks - 1), s);
                }
        __builtin_amdgcn_sched_barrier(0);
    };
    // the rows' sums of squares first: they are added up while the weights are on their way
    RowsSsq early;
    if (ssq_in) rows_ssq_ask(early, ssq_in, n_parts, 0);
    __builtin_amdgcn_sched_barrier(0);
    ask(wave);
    if (ssq_in) rows_ssq_share(part, early, ssq_in, n_parts);
    // needed when the walk is over: what the finishing lanes add to
    float x_old[4] = {0.f, 0.f, 0.f, 0.f}, by[4] = {0.f, 0.f, 0.f, 0.f};
    if (EPI == ROWS_RESID && wave == 0 && g * 4 < RB && r16 < M) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int n = min(n0 + g * 4 + i, N - 1);
            x_old[i] = x_io[(size_t)r16 * N + n];
            if (weighted_by) by[i] = weighted_by[n];
        }
    }
    f32x4 acc[CHAINS][RT];
#pragma unroll
    for (int c = 0; c < CHAINS; ++c)
#pragma unroll
        for (int t = 0; t < RT; ++t) acc[c][t] = f32x4{0.f, 0.f, 0.f, 0.f};
    for (int first = wave; first < n_chunks;) {
#pragma unroll
        for (int t = 0; t < RT; ++t)
#pragma unroll
            for (int j = 0; j < CH; ++j) {
                if (first + j * waves >= n_chunks) continue;
#pragma unroll
                for (int s = 0; s < 4; ++s) {
                    if (RAGGED && (first + j * waves) * 128 + s * 32 + g * 8 >= K)
                        w[t][j][s].u = x[j][s].u = make_uint4(0u, 0u, 0u, 0u);       // (both: zero times infinity is none)
                    acc[j % CHAINS][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[t][j][s].v, x[j][s].v, acc[j % CHAINS][t], 0, 0, 0);
                }
            }
        first += waves * CH;
        if (first < n_chunks) ask(first);
    }
#pragma unroll
    for (int c = 0; c < CHAINS; ++c)
#pragma unroll
        for (int t = 0; t < RT; ++t)
            red[((c * waves + wave) * RT + t) * 64 + lane] = make_float4(acc[c][t][0], acc[c][t][1], acc[c][t][2], acc[c][t][3]);
    __syncthreads();
    if (g * 4 >= RB) return;
    // D layout of the 16x16 tile: lane holds column lane % 16 (a token), rows 4 * (lane / 16) + i (weight rows)
    for (int t = wave; t < RT; t += waves) {
        float4 sums[CHAINS * ROWS_WAVES];
#pragma unroll
        for (int q = 0; q < CHAINS * ROWS_WAVES; ++q) sums[q] = red[(min(q, CHAINS * waves - 1) * RT + t) * 64 + lane];
        const float scale = ssq_in ? rows_scale(part, token, K, eps) : 1.f;
        float v[4] = {sums[0].x, sums[0].y, sums[0].z, sums[0].w};
#pragma unroll
        for (int q = 1; q < CHAINS * ROWS_WAVES; ++q)
            if (q < CHAINS * waves) v[0] += sums[q].x, v[1] += sums[q].y, v[2] += sums[q].z, v[3] += sums[q].w;
        const int n = n0 + t * 16 + g * 4;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            // each step rounded on its own (no fused multiply-add), so that every epilogue gives the same bits
            if (ssq_in) v[i] = __fmul_rn(v[i], scale);
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
                    if (weighted_out) weighted_out[(size_t)r16 * N + n + i] = f32_to_bf16(xn * by[i]);
                }
            }
            sq += __shfl_xor(sq, 16, WAVE);             // the two lanes of a token sit 16 apart
            if (g == 0) ssq_out[(size_t)blockIdx.x * ROWS_PARTS + r16] = sq;
        }
    }
}

// How a product is shared out: as many waves as there are chunks, eight at most, with `ch` chunks of 128 in flight each;
// `rt` tiles of 16 weight rows a block so that there is a block a CU (1,024 by 1,024, 8 rows: one tile 3.5 us, four 6.2; 9,216
// by 1,024: one 7.1, three, which is 192 blocks, 6.0; 16,384 by 2,048: one 14.7, four, 256 blocks, 13.0). A weight of more rows
// than four tiles a CU runs several blocks one after the other on a CU: those of many short rows are then the smallest, whose
// ends the others' loads cover (65,536 by 1,024, one row: one tile 22 us, four 26), unless there are more activations to share
// (8 rows: 28 and 25). The more chains a column is summed in, the nearer it is to 64 bits: fewer waves with more chunks each
// were 1.12e-7 off at K of 1,152, where eight are 8.8e-8, and eight with three chunks in one chain 1.21e-7 at 3,072, in two 1.14e-7.
// Eight chains up to 16 chunks and sixteen beyond, in this order, are the sums of before there was this kernel.
struct RowsShape {
    int waves, ch, rt, chains;
};
static RowsShape rows_shape(int m, int n, int k_per, int slices, bool ragged, int rb) {
    const int chunks = (k_per + 127) / 128;
    RowsShape sh{std::min(chunks, ROWS_WAVES), 4, 1, 1};
    sh.ch = std::min((chunks + sh.waves - 1) / sh.waves, 4);
    if (sh.ch > 2 && (rb == 16 ? n < 12288 : chunks > 32)) sh.chains = 2;
    if (rb == 16) {
        const long long tiles = (long long)((n + 15) / 16) * slices;
        const int most = ragged || sh.ch > 2 ? 2 : 4;
        const int a_cu = slices > 1 && tiles <= 512 ? 1 : tiles <= 1024 ? (int)((tiles + 255) / 256) : k_per < 2048 && m <= 4 ? 1 : 4;
        sh.rt = std::max(1, std::min(a_cu, most));
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
    int m, n, k, slices;
    Epilogue unit;
};

template <typename TOut, int RB, int EPI>
static void rows_launch(const RowsCall& c, hipStream_t s) {
    const int k_per = ((c.k + c.slices - 1) / c.slices + 127) / 128 * 128;
    const bool ragged = c.k % 128 != 0 || c.k >= (1 << 25);      // (offsets inside 64 rows are kept in 32 bits)
    const RowsShape sh = rows_shape(c.m, c.n, std::min(k_per, c.k), c.slices, ragged, RB);
    const dim3 grid((unsigned)((c.n + (long long)RB * sh.rt - 1) / (RB * sh.rt)), (unsigned)((c.k + k_per - 1) / k_per));
    const size_t lds = (size_t)sh.chains * sh.waves * sh.rt * 64 * sizeof(float4);          // (32 KB at most)
#define ROWS_GO(RT, CH, CHAINS, RG)                                                                                  \
    k_rows_gemm<TOut, RB, RT, CH, CHAINS, EPI, RG><<<grid, sh.waves * 64, lds, s>>>(                                   \
        c.x, c.ssq_in, c.n_parts, c.eps, c.w, c.bias, (TOut*)c.y, c.x_io, c.ssq_out, c.weighted_out, c.weighted_by, c.m, \
        c.n, c.k, k_per, c.unit)
#define ROWS_CH(RT, RG)                                                                                              \
    do {                                                                                                             \
        if (sh.ch == 1) ROWS_GO(RT, 1, 1, RG);                                                                       \
        else if (sh.ch == 2) ROWS_GO(RT, 2, 1, RG);                                                                  \
        else if (sh.ch == 3 && sh.chains == 2) ROWS_GO(RT, 3, 2, RG);                                                \
        else if (sh.ch == 3) ROWS_GO(RT, 3, 1, RG);                                                                  \
        else if (sh.chains == 2) ROWS_GO(RT, 4, 2, RG);                                                              \
        else ROWS_GO(RT, 4, 1, RG);                                                                                  \
    } while (0)
    if constexpr (RB == 16) {
        if (ragged) {
            if (sh.rt == 1) ROWS_CH(1, true);
            else ROWS_CH(2, true);
        } else if (sh.rt == 1) {
            ROWS_CH(1, false);
        } else if (sh.rt == 2) {
            ROWS_CH(2, false);
        } else if (sh.rt == 3) {
            if (sh.ch == 1) ROWS_GO(3, 1, 1, false);
            else ROWS_GO(3, 2, 1, false);
        } else {
            if (sh.ch == 1) ROWS_GO(4, 1, 1, false);
            else ROWS_GO(4, 2, 1, false);
        }
    } else {
        if (ragged) ROWS_CH(1, true);
        else ROWS_CH(1, false);
    }
#undef ROWS_CH
#undef ROWS_GO
}

int imparo_few_rows(const bf16_t* x, const bf16_t* w, const float* bias, void* y, int out_dtype, int m, int n, int k,
                    const Epilogue& epilogue, int slices, const float* ssq_in, int n_parts, float eps, hipStream_t s) {
    const RowsCall c{x, ssq_in, n_parts, eps, w, bias, y, nullptr, nullptr, nullptr, nullptr, m, n, k, slices, epilogue};
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
        rows_launch<float, 8, ROWS_RESID>(RowsCall{xb, ssq_in, n_parts, eps, wb, bias, nullptr, x_io, ssq_out, wo, weighted_by, m, n,
                                                   k, 1, Epilogue(EPI_NONE)}, s);
        return launch_status();
    }
    return imparo_few_rows(xb, wb, bias, y, out_dtype, m, n, k, Epilogue(epilogue == ROWS_SWIGLU ? EPI_SWIGLU : EPI_NONE), 1, ssq_in,
                           n_parts, eps, s);
}

// Asks the runtime about one kernel of this file, which makes it load the file's code onto the
// current device (it loads a file's kernels when one of them is first used; a stream under capture
// cannot do that).
int imparo_load_code_decode_rows() {
    hipFuncAttributes attributes;
    return hipFuncGetAttributes(&attributes, reinterpret_cast<const void*>(&k_rows_gemm<float, 8, 1, 1, 1, ROWS_RESID, false>)) ==
                   hipSuccess
               ? IMPARO_OK
               : IMPARO_LAUNCH_FAILED;
}
