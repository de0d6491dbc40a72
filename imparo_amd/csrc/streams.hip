// The residual stream as several copies of a row (hyper-connections), and norms that read it. One launch between
// two sublayers does all of it, row by row:
//   d    = the sublayer's result: the sum of its slices, or of a routed feed-forward's experts, or of both;
//   x'_t = sum_s mix[s, t] x_s + join[t] d                  (all copies from the old ones; written back)
//   u    = sum_t read[t] x'_t
//   out  = norm(u), a layer norm or an RMS norm with weight and maybe bias, or u itself.
// With one copy, and mix, join and read left out (one each), this is a residual add and the norm behind it.
// Sums in float32, in an order that the width alone decides.
#include "common.h"
#include "api.h"
#include "moe_route.h"

#define STREAM_MAX 16              // copies
#define STREAM_MAX_WIDTH 16384
#define STREAM_MAX_TOP 24          // experts a token uses

#define STREAM_NORM_NONE 0
#define STREAM_NORM_RMS 1
#define STREAM_NORM_LAYER 2

// What a routed feed-forward leaves to be summed here: see imparo_post_norm_add_moe.
struct StreamExperts {
    const float* y;
    const void* h;
    const int32_t* choice;
    const float* weight;
    const int32_t* slot_of_entry;
    int h_is_bf16, top, n_experts;
};

template <int V> struct StreamPiece { float e[V]; };
template <int V>
__device__ __forceinline__ StreamPiece<V> stream_load(const float* __restrict__ p) {
    StreamPiece<V> r;
    if constexpr (V == 4) {
        const float4 f = *reinterpret_cast<const float4*>(p);
        r.e[0] = f.x; r.e[1] = f.y; r.e[2] = f.z; r.e[3] = f.w;
    } else {
#pragma unroll
        for (int i = 0; i < V; ++i) r.e[i] = p[i];
    }
    return r;
}
template <int V>
__device__ __forceinline__ void stream_store(float* __restrict__ p, const float (&v)[V]) {
    if constexpr (V == 4) {
        *reinterpret_cast<float4*>(p) = make_float4(v[0], v[1], v[2], v[3]);
    } else {
#pragma unroll
        for (int i = 0; i < V; ++i) p[i] = v[i];
    }
}

// One block a row; a thread keeps PER pieces of V neighbouring values of u in registers. S: at least `streams`.
template <int S, int V, int PER, bool EARLY>
__global__ __launch_bounds__(1024) void k_stream_norm(
    const float* x, int in_streams, float* x_out, const float* __restrict__ delta, int n_delta,
    size_t delta_stride, StreamExperts moe, const int32_t* __restrict__ rows, int streams,
    const float* __restrict__ mix, const float* __restrict__ join, const float* __restrict__ read, int norm,
    const float* __restrict__ weight, const float* __restrict__ bias, float eps, void* __restrict__ out,
    int out_is_bf16, int width) {
    __shared__ float scratch[16];
    __shared__ float mixes[S][S], joins[S], reads[S];
    __shared__ int slot[STREAM_MAX_TOP];
    __shared__ float wt[STREAM_MAX_TOP];
    const int i_out = blockIdx.x, tid = threadIdx.x;
    const size_t t = rows ? rows[i_out] : i_out;
    const bool adds = moe.y || n_delta;
    const int pieces = width / V;
    // What depends on nothing is asked for first (EARLY), all of it before anything is waited for: with few rows (a decode step)
    // this kernel is a chain of trips to memory, and these are then one. (8 rows of 1,024 on four copies: 6.0 us where
    // it took 7.8 with the weights, the experts' places and the row one after the other.) Threads that keep several
    // pieces of a wide row ask for each piece's row where they use it.
    static_assert(!EARLY || PER == 1, "a thread's only piece");
    // Experts' rows are asked for without a branch (FREE), but for many single values a thread: sixteen times the code in
    // the unrolled pieces pushes 16 copies out of the registers (one row of 2,048 by 16 copies 421 us with the branch, 505
    // without).
    constexpr bool FREE = PER == 1 || V == 4;
    const int c_own = min(tid, pieces - 1) * V;
    auto passed = [&](int c) __attribute__((always_inline)) {          // what an expert that passes its input through gives
        StreamPiece<V> r;
#pragma unroll
        for (int i = 0; i < V; ++i)
            r.e[i] = moe.h_is_bf16 ? load_f32<bf16_t>((const bf16_t*)moe.h, t * width + c + i)
                                   : load_f32<float>((const float*)moe.h, t * width + c + i);
        return r;
    };
    StreamPiece<V> v_own[S], w_own, b_own, d_own;
    if (EARLY) {
#pragma unroll
        for (int s = 0; s < S; ++s)
            v_own[s] = stream_load<V>(x + (t * in_streams + (in_streams == 1 ? 0 : min(s, streams - 1))) * width + c_own);
        d_own = stream_load<V>((n_delta ? delta : x) + t * (n_delta ? 1 : in_streams) * width + c_own);
        const float* some = weight ? weight : bias ? bias : x;     // (read where there is none to keep loads off branches)
        w_own = stream_load<V>((weight ? weight : some) + c_own);
        b_own = stream_load<V>((bias ? bias : some) + c_own);
    }
    for (int i = tid; i < S * S; i += blockDim.x) {
        const int from = i / S, to = i % S;
        mixes[from][to] = (from >= streams || to >= streams) ? 0.f : mix ? mix[from * streams + to] : from == to ? 1.f : 0.f;
    }
    if (tid < S) {
        joins[tid] = tid >= streams ? 0.f : join ? join[tid] : 1.f;
        reads[tid] = tid >= streams ? 0.f : read ? read[tid] : 1.f;
    }
    if (moe.y && tid < moe.top) {
        const int e = moe.choice[t * moe.top + tid], at = moe.slot_of_entry[t * moe.top + tid];
        slot[tid] = e < moe.n_experts ? at : -1;
        wt[tid] = moe.weight ? moe.weight[t * moe.top + tid] : 1.0f;
    }
    __syncthreads();
    float u[PER][V];
    float sum = 0.f;
#pragma unroll
    for (int p = 0; p < PER; ++p) {
        const int piece = tid + p * blockDim.x;
        const bool in = piece < pieces;
        const int c = min(piece, pieces - 1) * V;
        StreamPiece<V> v[S];
#pragma unroll
        for (int s = 0; s < S; ++s)
            v[s] = EARLY ? v_own[s]
                         : stream_load<V>(x + (t * in_streams + (in_streams == 1 ? 0 : min(s, streams - 1))) * width + c);
        float d[V];
#pragma unroll
        for (int i = 0; i < V; ++i) d[i] = 0.f;
        if (moe.y) {
            for (int k0 = 0; k0 < moe.top; k0 += 4) {           // four experts' rows under way at once
                StreamPiece<V> y[4];
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const int sl = slot[min(k0 + j, moe.top - 1)];
                    if (FREE || sl >= 0) y[j] = stream_load<V>(moe.y + (size_t)max(sl, 0) * width + c);
                    else y[j] = passed(c);
                }
                if (FREE)
#pragma unroll
                    for (int j = 0; j < 4; ++j)
                        if (__builtin_amdgcn_readfirstlane(slot[min(k0 + j, moe.top - 1)]) < 0) y[j] = passed(c);
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const float w = k0 + j < moe.top ? wt[k0 + j] : 0.f;
#pragma unroll
                    for (int i = 0; i < V; ++i) d[i] = k0 + j < moe.top ? fmaf(w, y[j].e[i], d[i]) : d[i];
                }
            }
        }
        if (n_delta) {
            float e[V];
#pragma unroll
            for (int i = 0; i < V; ++i) e[i] = 0.f;
            for (int s0 = 0; s0 < n_delta; s0 += 4) {
                StreamPiece<V> y[4];
#pragma unroll
                for (int j = 0; j < 4; ++j)
                    y[j] = EARLY && s0 + j == 0 ? d_own
                                                : stream_load<V>(delta + (size_t)min(s0 + j, n_delta - 1) * delta_stride + t * width + c);
#pragma unroll
                for (int j = 0; j < 4; ++j)
#pragma unroll
                    for (int i = 0; i < V; ++i) e[i] += s0 + j < n_delta ? y[j].e[i] : 0.f;
            }
#pragma unroll
            for (int i = 0; i < V; ++i) d[i] += e[i];
        }
#pragma unroll
        for (int i = 0; i < V; ++i) u[p][i] = 0.f;
#pragma unroll
        for (int to = 0; to < S; ++to) {
            float n[V];
            if (adds) {
#pragma unroll
                for (int i = 0; i < V; ++i) n[i] = joins[to] * d[i];
#pragma unroll
                for (int s = 0; s < S; ++s)
#pragma unroll
                    for (int i = 0; i < V; ++i) n[i] = fmaf(mixes[s][to], v[s].e[i], n[i]);
                if (x_out && in && to < streams) stream_store<V>(x_out + (t * streams + to) * width + c, n);
            } else {
#pragma unroll
                for (int i = 0; i < V; ++i) n[i] = v[to].e[i];
            }
#pragma unroll
            for (int i = 0; i < V; ++i) u[p][i] = fmaf(reads[to], n[i], u[p][i]);
        }
#pragma unroll
        for (int i = 0; i < V; ++i) {
            if (!in) u[p][i] = 0.f;
            sum += norm == STREAM_NORM_RMS ? u[p][i] * u[p][i] : u[p][i];
        }
    }
    if (!out) return;
    float mean = 0.f, scale = 1.0f;
    if (norm == STREAM_NORM_RMS) {
        scale = 1.0f / sqrtf(block_sum(sum, scratch) / (float)width + eps);
    } else if (norm == STREAM_NORM_LAYER) {
        mean = block_sum(sum, scratch) / (float)width;
        float ss = 0.f;
#pragma unroll
        for (int p = 0; p < PER; ++p) {
            if (tid + p * (int)blockDim.x >= pieces) continue;
#pragma unroll
            for (int i = 0; i < V; ++i) ss = fmaf(u[p][i] - mean, u[p][i] - mean, ss);
        }
        scale = 1.0f / sqrtf(block_sum(ss, scratch) / (float)width + eps);
    }
#pragma unroll
    for (int p = 0; p < PER; ++p) {
        const int piece = tid + p * blockDim.x;
        if (piece >= pieces) continue;
        const int c = piece * V;
        float y[V];
#pragma unroll
        for (int i = 0; i < V; ++i) y[i] = (u[p][i] - mean) * scale;
        if (weight) {
            const StreamPiece<V> w = EARLY ? w_own : stream_load<V>(weight + c);
#pragma unroll
            for (int i = 0; i < V; ++i) y[i] *= w.e[i];
        }
        if (bias) {
            const StreamPiece<V> b = EARLY ? b_own : stream_load<V>(bias + c);
#pragma unroll
            for (int i = 0; i < V; ++i) y[i] += b.e[i];
        }
        const size_t dst = (size_t)i_out * width + c;
        if (out_is_bf16) {
            if constexpr (V == 4) {
                *reinterpret_cast<uint2*>((bf16_t*)out + dst) =
                    make_uint2(f32x2_to_bf16x2(y[0], y[1]), f32x2_to_bf16x2(y[2], y[3]));
            } else {
#pragma unroll
                for (int i = 0; i < V; ++i) store_f32<bf16_t>((bf16_t*)out, dst + i, y[i]);
            }
        } else {
            stream_store<V>((float*)out + dst, y);
        }
    }
}

// ---------------------------------------------------------------- a decode step's rows
// The same for the few rows of a decode step, whose sublayer left slices of a product, or experts' rows that lie by entry
// (token * used + place in the token's list: no places to look up first). Such a launch is a chain of trips to memory, so everything
// is asked for at once, the small constants through the scalar cache, and the rows' sums run as in k_stream_norm, so that a row has the same bits.
// ROUTE: the row goes on through a mixture's router in the same launch: its outputs (at most 16) are matrix products over the
// rounded row in LDS, chunks of 128 of K summed as the product of few rows sums them (decode_rows.hip: a wave a chunk, or two, the
// waves' sums in order), and the first wave chooses. 8 rows of 1,024 on four copies, one of 33 such launches of a step: behind a
// mixture 6.0 -> 4.7 us; behind attention, with a router of 8 outputs, 7.7, where norm, product and choice took 6.0 + 4.2 + 4.0.
// 8 chats of a mixture of 8 experts 32.0 -> 28.4 ms.
// (A block of the framework norms the mixer's result before its mixture, so no router rides behind experts' rows there; the entry takes it.)
#define STREAM_STEP_DELTAS 4
#define STREAM_STEP_TOP 8
#define STREAM_STEP_ROUTER 16
struct StreamRouter {
    const bf16_t* w;            // [n_router, width]
    const float* bias;          // [n_router] or null
    const float* correction;    // [n_router] or null
    int32_t* choice;            // [rows, top + always]
    float* weight;
    int n_router, top, scoring;
    MoeRouteRules rules;
};

template <int S, bool MOE, bool ROUTE>
__global__ __launch_bounds__(ROUTE ? 512 : 1024) void k_stream_step(
    const float* x, int in_streams, float* x_out, const float* __restrict__ delta, int n_delta, size_t delta_stride,
    StreamExperts moe, int streams, const float* __restrict__ mix, const float* __restrict__ join,
    const float* __restrict__ read, int norm, const float* __restrict__ weight, const float* __restrict__ bias, float eps,
    void* __restrict__ out, int out_is_bf16, int width, StreamRouter router) {
    typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
    typedef float f32x4 __attribute__((ext_vector_type(4)));
    typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
    constexpr int V = 4;
    __shared__ float scratch[16];
    __shared__ __attribute__((aligned(16))) bf16_t row_lds[ROUTE ? 2048 : 8];
    __shared__ float z_part[ROUTE ? 8 : 1][STREAM_STEP_ROUTER];
    const int tid = threadIdx.x, lane = tid & (WAVE - 1), wave = __builtin_amdgcn_readfirstlane(tid / WAVE);
    const size_t t = blockIdx.x;
    const int c = tid * V;                               // (a thread has one piece: blocks have width / 4 threads)
    StreamPiece<V> v[S], y[MOE ? STREAM_STEP_TOP : STREAM_STEP_DELTAS];
#pragma unroll
    for (int s = 0; s < S; ++s)
        v[s] = stream_load<V>(x + (t * in_streams + (in_streams == 1 ? 0 : min(s, streams - 1))) * width + c);
    if constexpr (MOE) {
#pragma unroll
        for (int k = 0; k < STREAM_STEP_TOP; ++k) y[k] = stream_load<V>(moe.y + (t * moe.top + min(k, moe.top - 1)) * width + c);
    } else {
#pragma unroll
        for (int k = 0; k < STREAM_STEP_DELTAS; ++k) y[k] = stream_load<V>(delta + min(k, n_delta - 1) * delta_stride + t * width + c);
    }
    const float* some = weight ? weight : bias ? bias : x;
    const StreamPiece<V> w = stream_load<V>((weight ? weight : some) + c), b = stream_load<V>((bias ? bias : some) + c);
    u32x4 rw[ROUTE ? 2 : 1][4];
    const int waves = blockDim.x / WAVE, r16 = lane & 15, g = lane >> 4;
    if constexpr (ROUTE) {                               // two chunks of 128 of the router's rows a wave
        const bf16_t* at = router.w + (size_t)min(r16, router.n_router - 1) * width + g * 8;
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int s = 0; s < 4; ++s) rw[h][s] = *reinterpret_cast<const u32x4*>(at + (wave + h * waves) * 128 + s * 32);
    }
    float mixes[S][S], joins[S], reads[S];
#pragma unroll
    for (int i = 0; i < S; ++i) {
        const int from = min(i, streams - 1);
        joins[i] = i >= streams ? 0.f : join ? join[from] : 1.f;
        reads[i] = i >= streams ? 0.f : read ? read[from] : 1.f;
#pragma unroll
        for (int to = 0; to < S; ++to)
            mixes[i][to] = (i >= streams || to >= streams) ? 0.f : mix ? mix[from * streams + min(to, streams - 1)] : i == to ? 1.f : 0.f;
    }
    float d[V];
#pragma unroll
    for (int i = 0; i < V; ++i) d[i] = 0.f;
    if constexpr (MOE) {
        float wt[STREAM_STEP_TOP];
        bool passes[STREAM_STEP_TOP];
#pragma unroll
        for (int k = 0; k < STREAM_STEP_TOP; ++k) {
            const size_t entry = t * moe.top + min(k, moe.top - 1);
            const int e = moe.choice[entry];
            wt[k] = moe.weight ? moe.weight[entry] : 1.0f;
            passes[k] = e < 0 || e >= moe.n_experts;
        }
#pragma unroll
        for (int k = 0; k < STREAM_STEP_TOP; ++k)
            if (k < moe.top && passes[k]) {              // an expert that hands its input on
#pragma unroll
                for (int i = 0; i < V; ++i)
                    y[k].e[i] = moe.h_is_bf16 ? load_f32<bf16_t>((const bf16_t*)moe.h, t * width + c + i)
                                              : load_f32<float>((const float*)moe.h, t * width + c + i);
            }
#pragma unroll
        for (int k = 0; k < STREAM_STEP_TOP; ++k)
#pragma unroll
            for (int i = 0; i < V; ++i) d[i] = k < moe.top ? fmaf(wt[k], y[k].e[i], d[i]) : d[i];
    } else {
        float e[V];
#pragma unroll
        for (int i = 0; i < V; ++i) e[i] = 0.f;
#pragma unroll
        for (int k = 0; k < STREAM_STEP_DELTAS; ++k)
#pragma unroll
            for (int i = 0; i < V; ++i) e[i] += k < n_delta ? y[k].e[i] : 0.f;
#pragma unroll
        for (int i = 0; i < V; ++i) d[i] += e[i];
    }
    float u[V];
    float sum = 0.f;
#pragma unroll
    for (int i = 0; i < V; ++i) u[i] = 0.f;
#pragma unroll
    for (int to = 0; to < S; ++to) {
        float n[V];
#pragma unroll
        for (int i = 0; i < V; ++i) n[i] = joins[to] * d[i];
#pragma unroll
        for (int s = 0; s < S; ++s)
#pragma unroll
            for (int i = 0; i < V; ++i) n[i] = fmaf(mixes[s][to], v[s].e[i], n[i]);
        if (x_out && to < streams) stream_store<V>(x_out + (t * streams + to) * width + c, n);
#pragma unroll
        for (int i = 0; i < V; ++i) u[i] = fmaf(reads[to], n[i], u[i]);
    }
#pragma unroll
    for (int i = 0; i < V; ++i) sum += norm == STREAM_NORM_RMS ? u[i] * u[i] : u[i];
    float mean = 0.f, scale = 1.0f;
    if (norm == STREAM_NORM_RMS) {
        scale = 1.0f / sqrtf(block_sum(sum, scratch) / (float)width + eps);
    } else if (norm == STREAM_NORM_LAYER) {
        mean = block_sum(sum, scratch) / (float)width;
        float ss = 0.f;
#pragma unroll
        for (int i = 0; i < V; ++i) ss = fmaf(u[i] - mean, u[i] - mean, ss);
        scale = 1.0f / sqrtf(block_sum(ss, scratch) / (float)width + eps);
    }
    float o[V];
#pragma unroll
    for (int i = 0; i < V; ++i) {
        o[i] = (u[i] - mean) * scale;
        if (weight) o[i] *= w.e[i];
        if (bias) o[i] += b.e[i];
    }
    const size_t dst = t * width + c;
    const uint2 packed = make_uint2(f32x2_to_bf16x2(o[0], o[1]), f32x2_to_bf16x2(o[2], o[3]));
    if (out_is_bf16) *reinterpret_cast<uint2*>((bf16_t*)out + dst) = packed;
    else stream_store<V>((float*)out + dst, o);
    if constexpr (ROUTE) {
        *reinterpret_cast<uint2*>(row_lds + c) = packed;
        __syncthreads();
        // every column of the products is this row; the router's rows are theirs. Up to eight chunks each has a sum of its own, of
        // sixteen a wave adds its two
        const bool pairs = 2 * waves > 8;
        f32x4 acc[2];
        acc[0] = acc[1] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            if (h == 1 && pairs) acc[1] = acc[0];
#pragma unroll
            for (int s = 0; s < 4; ++s) {
                const u32x4 a = *reinterpret_cast<const u32x4*>(row_lds + (wave + h * waves) * 128 + s * 32 + g * 8);
                acc[h] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, rw[h][s]), __builtin_bit_cast(bf16x8, a), acc[h], 0, 0, 0);
            }
        }
        if (r16 == 0) {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                if (!pairs) z_part[wave][4 * g + i] = acc[0][i];
                z_part[pairs ? wave : wave + waves][4 * g + i] = acc[1][i];
            }
        }
        __syncthreads();
        if (wave == 0) {
            const int parts = pairs ? waves : 2 * waves, e = min(lane, router.n_router - 1);
            float p[8];                                  // (asked for together)
#pragma unroll
            for (int q = 0; q < 8; ++q) p[q] = z_part[min(q, parts - 1)][e];
            float z = p[0];
#pragma unroll
            for (int q = 1; q < 8; ++q) z = q < parts ? z + p[q] : z;
            if (router.bias) z = __fadd_rn(z, router.bias[e]);
            moe_route_lanes(z, router.correction, router.choice, router.weight, (int)t, router.n_router, router.top, router.scoring,
                            router.rules, nullptr);
        }
    }
}

// Which steps imparo_stream_step takes: few rows of copies that a block keeps in registers, a piece of four a thread.
extern "C" int imparo_stream_step_takes(int n_rows, int streams, int width, int n_delta, int top) {
    return n_rows >= 1 && n_rows <= 16 && streams >= 1 && streams <= 4 && width >= 256 && width <= 4096 && width % 256 == 0 &&
           (top > 0 ? top <= STREAM_STEP_TOP && n_delta == 0 : n_delta >= 1 && n_delta <= STREAM_STEP_DELTAS);
}
// ... and where that is the faster way without a router: a thread's copies and all that joins them, asked for at once, fit the registers
// of a block of 1,024 threads in part only. One row, us here | k_stream_norm: a tensor joins, four copies of 1,024 3.45 | 3.62, of 1,280
// 3.96 | 3.72, of 4,096 5.60 | 4.59, two of 4,096 3.98 | 4.04; eight experts' rows join, four copies of 1,280 4.96 | 4.56, of 4,096
// 7.31 | 5.65, one or two of 2,048 faster here, one of 2,304 4.43 | 4.09, of 4,096 5.15 | 4.65.
extern "C" int imparo_stream_step_pays(int streams, int width, int top) {
    return streams > 2 ? width <= 1024 : top == 0 || width <= 2048;
}
// ... and whether a router of so many outputs rides: widths whose chunks of 128 come out as the product of few rows sums them.
extern "C" int imparo_stream_step_routes(int width, int n_router, int top) {
    return width % 256 == 0 && (width <= 1024 || width == 2048) && n_router >= 1 && n_router <= STREAM_STEP_ROUTER && top >= 1 &&
           top <= n_router;
}

extern "C" int imparo_stream_step(const float* x, int in_streams, float* x_out, const float* delta, int n_delta, const float* y,
                                  const void* h, int h_dtype, const int32_t* choice, const float* choice_weight, int top,
                                  int n_experts, int n_rows, int streams, const float* mix, const float* join, const float* read,
                                  int norm, const float* weight, const float* bias, float eps, void* out, int out_dtype,
                                  int width, const void* router_w, const float* router_bias, const float* correction,
                                  int n_router, int route_top, int scoring, int normalize, float route_scale, int always,
                                  int32_t* route_choice, float* route_weight, imparo_stream stream) {
    if (!x || !x_out || !out || n_rows < 0 || n_delta < 0 || (n_delta && !delta) || (!y && top) || (y && top < 1)) return IMPARO_BAD_ARGUMENT;
    if (n_rows == 0) return IMPARO_OK;
    if (!imparo_stream_step_takes(n_rows, streams, width, n_delta, y ? top : 0)) return IMPARO_BAD_ARGUMENT;
    if ((in_streams != streams && in_streams != 1) || (in_streams != streams && x_out == x)) return IMPARO_BAD_ARGUMENT;
    if (y && (!h || !choice || n_experts < 0 || (h_dtype != IMPARO_F32 && h_dtype != IMPARO_BF16))) return IMPARO_BAD_ARGUMENT;
    if (norm < STREAM_NORM_NONE || norm > STREAM_NORM_LAYER) return IMPARO_BAD_ARGUMENT;
    if (out_dtype != IMPARO_F32 && out_dtype != IMPARO_BF16) return IMPARO_BAD_ARGUMENT;
    if (((uintptr_t)x | (uintptr_t)x_out | (uintptr_t)delta | (uintptr_t)y | (uintptr_t)out | (uintptr_t)weight | (uintptr_t)bias |
         (uintptr_t)router_w) & 15)
        return IMPARO_BAD_ARGUMENT;
    const MoeRouteRules rules{n_router, 1, 1, normalize, route_scale, always};
    const StreamRouter router{(const bf16_t*)router_w, router_bias, correction, route_choice, route_weight, n_router, route_top, scoring, rules};
    if (router_w) {
        if (!imparo_stream_step_routes(width, n_router, route_top) || out_dtype != IMPARO_BF16) return IMPARO_BAD_ARGUMENT;
        if (!route_choice || !route_weight || always < 0 || route_top + always > MOE_MAX_USED || !(route_scale == route_scale))
            return IMPARO_BAD_ARGUMENT;
        if (scoring < MOE_SCORE_SOFTMAX || scoring > MOE_SCORE_CHOSEN) return IMPARO_BAD_ARGUMENT;
        // a block reads its row of the choices that join and writes its row of the new ones: where both lie in one buffer the rows have
        // to be the same ones, or a block would write what another has yet to read
        const int used = route_top + always;
        auto crosses = [&](const void* joins, const void* chosen) {
            const uintptr_t a = (uintptr_t)joins, b = (uintptr_t)chosen, rows = (uintptr_t)n_rows * 4;
            return joins && a < b + rows * used && b < a + rows * top && !(a == b && used == top);
        };
        if (y && (crosses(choice, route_choice) || crosses(choice_weight, route_weight))) return IMPARO_BAD_ARGUMENT;
    }
    hipStream_t s = (hipStream_t)stream;
    const StreamExperts moe{y, h, choice, choice_weight, nullptr, h_dtype == IMPARO_BF16, top, n_experts};
    const size_t stride = (size_t)n_rows * width;
    const int out_is_bf16 = out_dtype == IMPARO_BF16;
#define STREAM_STEP(S, MOE, ROUTE)                                                                                   \
    k_stream_step<S, MOE, ROUTE><<<n_rows, width / 4, 0, s>>>(x, in_streams, x_out, delta, n_delta, stride, moe, streams, mix, join, \
                                                              read, norm, weight, bias, eps, out, out_is_bf16, width, router)
#define STREAM_STEP_OF(S)                                                                                            \
    if (y && router_w) STREAM_STEP(S, true, true);                                                                   \
    else if (y) STREAM_STEP(S, true, false);                                                                         \
    else if (router_w) STREAM_STEP(S, false, true);                                                                  \
    else STREAM_STEP(S, false, false)
    if (streams == 1) { STREAM_STEP_OF(1); }
    else if (streams == 2) { STREAM_STEP_OF(2); }
    else { STREAM_STEP_OF(4); }
#undef STREAM_STEP_OF
#undef STREAM_STEP
    return launch_status();
}

extern "C" int imparo_stream_max() { return STREAM_MAX; }

extern "C" int imparo_stream_norm(const float* x, int in_streams, float* x_out, const float* delta, int n_delta,
                                  const float* y, const void* h, int h_dtype, const int32_t* choice,
                                  const float* choice_weight, const int32_t* slot_of_entry, int top, int n_experts,
                                  int n_rows_x, const int32_t* rows, int streams, const float* mix, const float* join,
                                  const float* read, int norm, const float* weight, const float* bias, float eps,
                                  void* out, int out_dtype, int n_out, int width, imparo_stream stream) {
    if (!x || n_rows_x < 0 || n_out < 0 || n_delta < 0 || (n_delta && !delta)) return IMPARO_BAD_ARGUMENT;
    if (width < 1 || width > STREAM_MAX_WIDTH || streams < 1 || streams > STREAM_MAX) return IMPARO_BAD_ARGUMENT;
    if (in_streams != streams && in_streams != 1) return IMPARO_BAD_ARGUMENT;
    if (y && (!h || !choice || !slot_of_entry || top < 1 || top > STREAM_MAX_TOP || n_experts < 0 ||
              (h_dtype != IMPARO_F32 && h_dtype != IMPARO_BF16)))
        return IMPARO_BAD_ARGUMENT;
    if (norm < STREAM_NORM_NONE || norm > STREAM_NORM_LAYER) return IMPARO_BAD_ARGUMENT;
    if (!out && !x_out) return IMPARO_BAD_ARGUMENT;
    if (out && out_dtype != IMPARO_F32 && out_dtype != IMPARO_BF16) return IMPARO_BAD_ARGUMENT;
    // the copies are written where something joins them, for every row; copies that were one are written elsewhere
    if (x_out && (rows || (!y && !n_delta) || (in_streams != streams && x_out == x))) return IMPARO_BAD_ARGUMENT;
    if (!rows && n_out != n_rows_x) return IMPARO_BAD_ARGUMENT;
    if (n_out == 0) return IMPARO_OK;
    hipStream_t s = (hipStream_t)stream;
    const StreamExperts moe{y, h, choice, choice_weight, slot_of_entry, h_dtype == IMPARO_BF16, top, n_experts};
    const size_t stride = (size_t)n_rows_x * width;
    const bool four = width % 4 == 0 && streams <= 8 && !(((uintptr_t)x | (uintptr_t)x_out | (uintptr_t)delta | (uintptr_t)y |
                                           (uintptr_t)out | (uintptr_t)weight | (uintptr_t)bias) & 15);
    const int pieces = four ? width / 4 : width;
    const int threads = pieces >= 1024 ? 1024 : (pieces + WAVE - 1) / WAVE * WAVE;
    const int per = (pieces + threads - 1) / threads;
    const int out_is_bf16 = out_dtype == IMPARO_BF16;
    // Once there are several rounds of blocks, how many of them a CU holds is what counts, and what is asked for early takes
    // registers, of more copies more. Late where that costs more than the wait for memory: without a norm to wait for; and of
    // several copies, while blocks have at most 512 threads (of 1,024 a CU holds two either way) and few slices of a
    // pending result, which late are asked for one trip later than the row. us early | late, layer norm unless said, 2,048 rows of 2,048:
    // one slice by 2 copies 18.8 | 17.4, by 5 37.5 | 33.3, by 8 56.6 | 52.1; by one copy 13.2 | 13.8; four slices by 4 31.6 | 34.7, by 8
    // 68.6 | 72.9, two by 4 27.9 | 29.4, by 5 39.0 | 36.0; no norm, by 4 26.6 | 25.0. Rows of 4,096, two slices by 4 copies, 1,200 rows: 33.0 | 35.0,
    // but 8,192 rows, one slice by 2 copies 145 | 138. From few rows on by many copies (600 of 2,048 by 5 14.5 | 13.8, by 4 with 1,200
    // rows still 17.1 | 17.6, without a norm 600 9.0 | 9.6), two slices of few copies from more rows on (8,192 of 1,024 by 2 36.3 |
    // 34.7). With experts' rows early is the faster way at any count (2,048 rows of 2,048 by 8 copies 74 | 86).
    const long long at_work = (long long)n_out * threads;
    const bool late = !y && per <= 1 &&
                      (norm == STREAM_NORM_NONE ? at_work >= (streams == 3 || streams == 4 ? 600000 : 1 << 18)
                                                : at_work >= (streams > 4 ? 1 << 18 : 1 << 20) && streams > 1 &&
                                                      n_delta <= (streams > 4 || at_work >= 1 << 21 ? 2 : 1) &&
                                                      (threads <= 512 || (streams == 2 && n_delta == 1)));
#define STREAM_NORM(S, V, PER)                                                                                       \
    k_stream_norm<S, V, PER, (PER == 1)><<<n_out, threads, 0, s>>>(x, in_streams, x_out, delta, n_delta, stride, moe, rows, streams, \
                                                       mix, join, read, norm, weight, bias, eps, out, out_is_bf16, width)
#define STREAM_WIDTHS(S)                                                                                             \
    if (four) {                                                                                                      \
        if (late) k_stream_norm<S, 4, 1, false><<<n_out, threads, 0, s>>>(                                           \
            x, in_streams, x_out, delta, n_delta, stride, moe, rows, streams, mix, join, read, norm, weight, bias,   \
            eps, out, out_is_bf16, width);                                                                           \
        else if (per <= 1) STREAM_NORM(S, 4, 1);                                                                     \
        else STREAM_NORM(S, 4, 4);                                                                                   \
    } else {                                                                                                         \
        if (per <= 1) STREAM_NORM(S, 1, 1);                                                                          \
        else STREAM_NORM(S, 1, 16);                                                                                  \
    }
    if (streams == 1) { STREAM_WIDTHS(1) }
    else if (streams == 2) { STREAM_WIDTHS(2) }
    else if (streams <= 4) { STREAM_WIDTHS(4) }
    else if (streams <= 8) { STREAM_WIDTHS(8) }
    else if (per <= 1) { STREAM_NORM(16, 1, 1); }
    else { STREAM_NORM(16, 1, 16); }
#undef STREAM_WIDTHS
#undef STREAM_NORM
    return launch_status();
}

int imparo_load_code_streams() {
    hipFuncAttributes attributes;
    return hipFuncGetAttributes(&attributes, reinterpret_cast<const void*>(&k_stream_norm<4, 4, 1, true>)) == hipSuccess
               ? IMPARO_OK : IMPARO_LAUNCH_FAILED;
}
