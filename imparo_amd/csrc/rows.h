// Shared by the products of a step of at most 16 tokens (decode_rows.hip) and of more (gemm.hip): what happens to a
// product before it is stored, and a norm of the residual stream folded into the products around it: the product that
// adds its result to the stream leaves the partial sums of squares of the new rows and the rows times the next norm's
// weight in bfloat16; the product behind that norm runs on those rows and multiplies each row's result at the end by
// scale[t] = rsqrt(sum_p ssq[p][t] / width + eps). The scale is one number a row, so the walk along K does not wait for
// the sums, and there is no launch for the norm.
#pragma once
#include "common.h"

typedef float f32x4_any __attribute__((ext_vector_type(4), aligned(4)));     // four floats wherever they lie

#define EPI_NONE 0
#define EPI_SWIGLU 1   // weight rows interleaved gate, up, gate, up...: out[m, j] = act(y[m, 2j], y[m, 2j+1])
#define EPI_ADD 2      // float32 out only: Y += y, what Y holds being read where the result is stored

// What happens to a product before it is stored: its kind (one of the above) and, for the gated kind, a constant
// the result is multiplied by in float32 before it is rounded (a factor on the whole sublayer, carried by the input
// of the product that follows), and the bound of a unit that has one: act(g, u) = silu(g) u with limit 0, else
// g' sigmoid(alpha g') (u' + 1) with g' = min(g, limit), u' = clamp(u, -limit, limit).
struct Epilogue {
    int kind;
    float scale, limit, alpha;
    __host__ __device__ Epilogue(int k, float s = 1.0f, float l = 0.0f, float a = 1.0f) : kind(k), scale(s), limit(l), alpha(a) {}
    __host__ __device__ operator int() const { return kind; }
};

__device__ __forceinline__ void gated_bounds(const Epilogue& e, float& g, float& u) {
    if (e.limit > 0.f) {
        g = fminf(g, e.limit);
        u = fminf(fmaxf(u, -e.limit), e.limit) + 1.0f;
    }
}
__device__ __forceinline__ float gated_mul(const Epilogue& e, float g, float u) {
    gated_bounds(e, g, u);
    return g / (1.0f + expf(-e.alpha * g)) * u * e.scale;
}
// The same with the hardware's exp2 and reciprocal (an ulp each) for the bfloat16 kernels: the exact
// division and exponential cost some thirty instructions per output, ten microseconds per 256x256 tile
__device__ __forceinline__ float gated_mul_fast(const Epilogue& e, float g, float u) {
    gated_bounds(e, g, u);
    return g * __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(-1.44269504f * e.alpha * g)) * u * e.scale;
}

#define ROWS_MAX 16          // tokens of a step these kernels take
#define ROWS_PARTS 16        // floats per partial sum of squares: one per token
#define ROWS_ASK 4           // partial sums of four tokens that a thread has in flight at once

struct RowsSsq {
    f32x4_any v[ROWS_ASK];
};

// Thread i gathers the partials p = first + i / 4, + threads / 4, ... of tokens 4 * (i % 4) to 4 * (i % 4) + 3: every block
// of a product reads all of them, 16 KB for a stream of 2,048, and in vectors that is a quarter of the loads.
__device__ __forceinline__ void rows_ssq_ask(RowsSsq& r, const float* __restrict__ ssq, int n_parts, int first) {
    const int at = first + (threadIdx.x >> 2), step = blockDim.x >> 2;
#pragma unroll
    for (int j = 0; j < ROWS_ASK; ++j)
        r.v[j] = *reinterpret_cast<const f32x4_any*>(ssq + (size_t)min(at + j * step, n_parts - 1) * ROWS_PARTS + (threadIdx.x & 3) * 4);
}

__device__ __forceinline__ float rows_fold(float v) {       // over the lanes 4, 8, 16 and 32 apart
    v += rotated_in_row<8>(v);
    v += rotated_in_row<4>(v);
    auto swapped = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    v = __uint_as_float(swapped[0]) + __uint_as_float(swapped[1]);
    swapped = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return __uint_as_float(swapped[0]) + __uint_as_float(swapped[1]);
}

// Lanes 0 to 3 of every wave put the wave's share of their four tokens' sums at part[wave][token]: `early` holds the first
// round, asked for before the walk along K; further rounds are fetched here. The order of the additions depends on the
// block size and the number of partials only.
__device__ __forceinline__ void rows_ssq_share(float* part, const RowsSsq& early, const float* __restrict__ ssq, int n_parts) {
    const int at = threadIdx.x >> 2, step = blockDim.x >> 2;
    float4 s = make_float4(0.f, 0.f, 0.f, 0.f);
    auto add = [&](const RowsSsq& r, int first) {
#pragma unroll
        for (int j = 0; j < ROWS_ASK; ++j) {
            const bool in = first + at + j * step < n_parts;
            s.x += in ? r.v[j][0] : 0.f, s.y += in ? r.v[j][1] : 0.f, s.z += in ? r.v[j][2] : 0.f, s.w += in ? r.v[j][3] : 0.f;
        }
    };
    add(early, 0);
    for (int first = ROWS_ASK * step; first < n_parts; first += ROWS_ASK * step) {
        RowsSsq r;
        rows_ssq_ask(r, ssq, n_parts, first);
        add(r, first);
    }
    s = make_float4(rows_fold(s.x), rows_fold(s.y), rows_fold(s.z), rows_fold(s.w));
    if ((threadIdx.x & 63) < 4) *reinterpret_cast<float4*>(part + (threadIdx.x >> 6) * 16 + (threadIdx.x & 3) * 4) = s;
}

// After rows_ssq_share, and once the block (at most 8 waves) has met: the waves' shares are added in wave order. All of
// them are read before the first is added: a loop that reads one after the other makes a trip to LDS for each (with 32
// shares it was 1.4 us of a product of 8).
__device__ __forceinline__ float rows_scale(const float* part, int token, int width, float eps) {
    const int waves = blockDim.x >> 6;
    float share[8];
#pragma unroll
    for (int w = 0; w < 8; ++w) share[w] = part[min(w, waves - 1) * 16 + token];
    float total = 0.f;
#pragma unroll
    for (int w = 0; w < 8; ++w) total += w < waves ? share[w] : 0.f;
    return 1.0f / sqrtf(total / (float)width + eps);
}

// (decode_rows.hip) Y = X . W^T of at most 16 rows, kinds EPI_NONE and EPI_SWIGLU; `slices` of K as imparo_gemm_slices
// says, each a float32 result of its own in Y; ssq_in (null: none): the rows are scaled at the end.
int imparo_few_rows(const bf16_t* x, const bf16_t* w, const float* bias, void* y, int out_dtype, int m, int n, int k,
                    const Epilogue& epilogue, int slices, const float* ssq_in, int n_parts, float eps, hipStream_t s);

// (some_rows.hip) Products of 17 to SOME_ROWS_MAX rows with a K that is a multiple of 128, any kind; `tile`: weight rows a block, 64, 32 or 16,
// as imparo_some_rows_tile says.
#define SOME_ROWS_MAX 128
bool imparo_some_rows_takes(int m, int n, int k);
int imparo_some_rows_tile(int m, int n, int slices);
int imparo_some_rows(const bf16_t* x, const bf16_t* w, const float* bias, void* y, int out_dtype, int m, int n, int k,
                     const Epilogue& epilogue, int slices, int tile, hipStream_t s);
