// Y[m, n] = X[m, k] . W[n, k]^T with float32 accumulation.
//
// float32: kernels on the matrix cores' float32 products; every output element sums
// its products in the order k = 0, 1, 2, ... whatever the tile it falls in, so a row's
// result does not depend on how many other rows are in the batch.
// bfloat16: MFMA kernels, LDS-tiled ones for many rows and weight-streaming ones for some
// (17 to 128 rows: some_rows.hip; at most 16: decode_rows.hip).
#include "common.h"

#include <algorithm>
#include "api.h"
#include "rows.h"

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

union Frag8 {
    uint4 u;
    bf16x8 v;
};

__device__ __forceinline__ uint4 zero_if(bool out, uint4 v) {
    return make_uint4(out ? 0u : v.x, out ? 0u : v.y, out ? 0u : v.z, out ? 0u : v.w);
}

// ------------------------------------------------------------------ float32
// The float32 matrix instructions round exactly as a chain of fused multiply-adds over k = 0, 1, 2, ... does
// (checked against fmaf on normal, widely spread and subnormal values: the same bits everywhere), so both kernels
// below run on the matrix cores, at twice the vector units' rate, and still sum every output in that order.
//
// Many rows: a tile of 64x64 or 32x32 per block of four waves, a quarter each, K in steps of 32 or 64 through LDS; a thread
// brings 8 neighbouring k of a row of each operand, the loads of four further steps in flight.
// 64x64: a wave has 32x32 on the 32x32x2 product, 32 cycles a k. Of 8 neighbouring k the even ones lie together in LDS
// and then the odd ones: lane / 32 picks a half of each product's two k, so one 16-byte read feeds four products.
// 32x32: a wave has 16x16 on the 16x16x4 product, whose chain takes 8 cycles a k; k = 4p + lane / 16 of product p comes out
// of LDS as it lies there, value by value (rows 68 floats apart: 64 lanes, 64 banks).
// A step's operands go to LDS while the products of the step before run, and the barrier stands before its last four products, with
// the next step's first operands asked for behind it, so that neither is waited for.
// Bound by the matrix cores where there are enough tiles, and with few by the chain of a wave's products (64x64) or what a CU
// brings in, 30 to 40 GB/s (32x32). Measured, 666 rows: 131 us by 9,216 by 1,024 (96 TFLOP/s; 140 when a step's writes, barrier and
// reads stood between its products and the last step's), 89 by 1,024 by 4,608 (107); 64 rows by 1,024 by 4,608 41 (106).
template <bool SMALL>
struct F32Tile {
    static constexpr int M = SMALL ? 32 : 64, K = SMALL ? 64 : 32;
    static constexpr int LD = SMALL ? 68 : 40;      // (40: 32 bytes beyond a row's own keep 16-byte reads free of conflicts)
    static constexpr int SUB = K / 4;               // k of four products
    using Acc = typename std::conditional<SMALL, f32x4, f32x16>::type;
};

// lane: token m, weight rows n .. n + 3
template <typename TOut>
__device__ __forceinline__ void f32_rows_out(const f32x4& acc, const float* __restrict__ bias, TOut* __restrict__ Y, int m, int n, int M,
                                             int N, const Epilogue& epilogue) {
    if (m >= M) return;
    float v[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] = bias && n + i < N ? acc[i] + bias[n + i] : acc[i];
    if (epilogue == EPI_SWIGLU) {
#pragma unroll
        for (int i = 0; i < 4; i += 2)
            if (n + i + 1 < N) store_f32<TOut>(Y, (size_t)m * (N / 2) + (n + i) / 2, gated_mul(epilogue, v[i], v[i + 1]));
        return;
    }
#pragma unroll
    for (int i = 0; i < 4; ++i)
        if (n + i < N) store_f32<TOut>(Y, (size_t)m * N + n + i, v[i]);
}

// VEC: K is at least 4, and rows are read in vectors of four floats that may start anywhere; the end of a K that is no
// multiple of 4, and a shorter K, value by value. (666 rows by 9,216 by 1,024 that start 4 bytes off 16:
// 136 us, 395 value by value.)
template <typename TOut, bool VEC, bool SMALL>
__global__ __launch_bounds__(256, VEC ? 4 : 3) void k_gemm_f32(const float* __restrict__ X, const float* __restrict__ W,
                                                  const float* __restrict__ bias, TOut* __restrict__ Y,
                                                  int M, int N, int K, int tiles_m, int tiles_n, Epilogue epilogue) {
    using T = F32Tile<SMALL>;
    __shared__ __attribute__((aligned(16))) float xs[2][T::M * T::LD];
    __shared__ __attribute__((aligned(16))) float ws[2][T::M * T::LD];
    // blocks that share weight rows are neighbours on one XCD (they go to the 8 XCDs in turn, each has an L2)
    const int total = tiles_m * tiles_n;
    const int per_xcd = (total + 7) / 8;
    const int block = blockIdx.y * gridDim.x + blockIdx.x;   // (a row of the grid is a multiple of 8)
    const int logical = (block % 8) * per_xcd + block / 8;
    if (block / 8 >= per_xcd || logical >= total) return;
    const int m0 = (logical % tiles_m) * T::M, n0 = (logical / tiles_m) * T::M;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int wm = (wave >> 1) * (T::M / 2), wn = (wave & 1) * (T::M / 2);
    const int row = tid / (T::K / 8), part = tid % (T::K / 8) * 8;
    const float* xrow = X + (size_t)min(m0 + row, M - 1) * K;
    const float* wrow = W + (size_t)min(n0 + row, N - 1) * K;
    struct Ahead {
        float x[8], w[8];
    };
    auto fetch_values = [&](int k0, Ahead& f) __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < 8; ++j) f.x[j] = xrow[min(k0 + part + j, K - 1)], f.w[j] = wrow[min(k0 + part + j, K - 1)];
    };
    auto fetch = [&](int k0, Ahead& f) __attribute__((always_inline)) {     // no load under a branch; what lies past K is zero
        const int k = k0 + part;
        if (VEC) {
#pragma unroll
            for (int j = 0; j < 8; j += 4) {
                const int at = min(k + j, K - 4);
                const f32x4_any a = *reinterpret_cast<const f32x4_any*>(xrow + at), b = *reinterpret_cast<const f32x4_any*>(wrow + at);
                f.x[j] = a.x, f.x[j + 1] = a.y, f.x[j + 2] = a.z, f.x[j + 3] = a.w;
                f.w[j] = b.x, f.w[j + 1] = b.y, f.w[j + 2] = b.z, f.w[j + 3] = b.w;
            }
        } else {
            fetch_values(k0, f);
        }
    };
    const int at = row * T::LD + part;
    auto put_row = [&](int k0, float* to, const float (&f)[8]) __attribute__((always_inline)) {
        float v[8];
#pragma unroll
        for (int j = 0; j < 8; ++j)                      // (the choice also where it always holds: without it the compiler
            v[SMALL ? j : (j & 1) * 4 + j / 2] = k0 + part + j < K ? f[j] : 0.f;   // sorts what comes as it comes, and waits there)
        *reinterpret_cast<float4*>(to) = make_float4(v[0], v[1], v[2], v[3]);
        *reinterpret_cast<float4*>(to + 4) = make_float4(v[4], v[5], v[6], v[7]);
    };
    auto put = [&](int k0, int buf, const Ahead& f) __attribute__((always_inline)) {
        put_row(k0, &xs[buf][at], f.x);
        __builtin_amdgcn_sched_barrier(0);               // (one after the other: registers)
        put_row(k0, &ws[buf][at], f.w);
    };
    struct Operands {
        float x[4], w[4];
    };
    const int get_x = SMALL ? (wm + (lane & 15)) * T::LD + (lane >> 4) : (wm + (lane & 31)) * T::LD + (lane >> 5) * 4;
    const int get_w = SMALL ? (wn + (lane & 15)) * T::LD + (lane >> 4) : (wn + (lane & 31)) * T::LD + (lane >> 5) * 4;
    auto get = [&](int buf, int sub, Operands& o) __attribute__((always_inline)) {
        if (SMALL) {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                o.x[i] = xs[buf][get_x + sub * T::SUB + i * 4];
                o.w[i] = ws[buf][get_w + sub * T::SUB + i * 4];
            }
        } else {
            const float4 a = *reinterpret_cast<const float4*>(&xs[buf][get_x + sub * T::SUB]);
            const float4 b = *reinterpret_cast<const float4*>(&ws[buf][get_w + sub * T::SUB]);
            o.x[0] = a.x, o.x[1] = a.y, o.x[2] = a.z, o.x[3] = a.w;
            o.w[0] = b.x, o.w[1] = b.y, o.w[2] = b.z, o.w[3] = b.w;
        }
    };
    typename T::Acc acc = {};
    auto multiply = [&](const Operands& o) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            if constexpr (SMALL)
                acc = __builtin_amdgcn_mfma_f32_16x16x4f32(o.w[i], o.x[i], acc, 0, 0, 0);
            else
                acc = __builtin_amdgcn_mfma_f32_32x32x2f32(o.x[i], o.w[i], acc, 0, 0, 0);
        }
    };
    Operands even, odd;
    // One step, whose first operands are in `even`; `next` holds the step behind it, which goes to LDS here (if it is not
    // the last), and is asked for the fourth step behind that one.
    auto step = [&](int k0, int buf, Ahead& next, const bool more, const bool puts) __attribute__((always_inline)) {
        get(buf, 1, odd);
        __builtin_amdgcn_sched_barrier(0);
        multiply(even);
        if (puts) put(k0 + T::K, buf ^ 1, next);
        if (more) fetch(k0 + 5 * T::K, next);
        __builtin_amdgcn_sched_barrier(0);   // (left alone, the compiler sinks these loads to where they are used)
        get(buf, 2, even);
        multiply(odd);
        __builtin_amdgcn_sched_barrier(0);
        get(buf, 3, odd);
        multiply(even);
        // (nobody reads the other buffer any more, nobody will read this one; the loads in flight are not waited for)
        __builtin_amdgcn_sched_barrier(0);
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        get(buf ^ 1, 0, even);               // (behind the last step: for nothing)
        __builtin_amdgcn_sched_barrier(0);
        multiply(odd);
        __builtin_amdgcn_sched_barrier(0);
    };
    const int steps = (K + T::K - 1) / T::K;
    Ahead s0, s1, s2, s3;
    // (in the order they are used: a first use whose loads were issued last would wait for all of them, every round)
    fetch(0, s0);
    __builtin_amdgcn_sched_barrier(0);
    fetch(T::K, s1);
    __builtin_amdgcn_sched_barrier(0);
    fetch(2 * T::K, s2);
    __builtin_amdgcn_sched_barrier(0);
    fetch(3 * T::K, s3);
    __builtin_amdgcn_sched_barrier(0);
    if (VEC && K % 4 && steps == 1) fetch_values(0, s0);
    put(0, 0, s0);
    fetch(4 * T::K, s0);
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    get(0, 0, even);
    // turns of four steps that two steps at least come behind, so that the last step, which may end inside a vector, is none that
    // a turn puts into LDS
    const int turns = steps < 2 ? 0 : (steps - 2) / 4 * 4 * T::K;
    for (int k0 = 0; k0 < turns; k0 += 4 * T::K) {
        step(k0, 0, s1, true, true);
        step(k0 + T::K, 1, s2, true, true);
        step(k0 + 2 * T::K, 0, s3, true, true);
        step(k0 + 3 * T::K, 1, s0, true, true);
    }
    // what is left of K, up to five steps, the last one filled up with zeros (a short K is nothing else: 4,096 rows by 1,024
    // by 8 9.3 us where steps to the end of the turn took 18 and steps of 16 on the vector units 11)
    auto rest = [&](int k0, int buf, Ahead& next) __attribute__((always_inline)) {
        if (k0 >= K) return;
        if (VEC && K % 4 && k0 + T::K < K && k0 + 2 * T::K > K) fetch_values(k0 + T::K, next);
        step(k0, buf, next, false, k0 + T::K < K);
    };
    rest(turns, 0, s1);
    rest(turns + T::K, 1, s2);
    rest(turns + 2 * T::K, 0, s3);
    rest(turns + 3 * T::K, 1, s0);
    rest(turns + 4 * T::K, 0, s1);
    if constexpr (SMALL) {
        f32_rows_out<TOut>(acc, bias, Y, m0 + wm + (lane & 15), n0 + wn + (lane >> 4) * 4, M, N, epilogue);
    } else {
        // a lane holds one column (a weight row) of 16 activation rows
        const int n = n0 + wn + (lane & 31);
        const float bn = bias && n < N ? bias[n] : 0.f;
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const int m = m0 + wm + (r >> 2) * 8 + (lane >> 5) * 4 + (r & 3);
            const float v = bias ? acc[r] + bn : acc[r];
            if (epilogue == EPI_SWIGLU) {
                const float up = lane_xor<1>(v);             // gate and up rows are neighbours
                if (m < M && !(lane & 1) && n + 1 < N) store_f32<TOut>(Y, (size_t)m * (N / 2) + n / 2, gated_mul(epilogue, v, up));
            } else if (m < M && n < N) {
                store_f32<TOut>(Y, (size_t)m * N + n, v);
            }
        }
    }
}

// At most 16 rows (a decode step in the float32 engine): a wave takes 16 weight rows and all the activation rows
// and walks K alone, operands from memory straight into registers, 16 bytes a lane: lane (row, g) asks for
// k = 4g .. 4g + 3 of 16, and a transposition over the four groups of lanes (four lane swaps) gives it
// k = g, 4 + g, 8 + g, 12 + g, which is how the products want them. Loads run seven chunks of 32 ahead in eight
// register sets. For any K and operands that start anywhere, as its loads ask for 4-byte alignment only (2 rows of 1,024 by
// 1,026 9.9 us, 65,536 by 1,022 44; value by value in tiles of 64 rows 50 and 144); a K that is a multiple of 64 goes
// through the ring below. Bound by the weight's bytes, or, where few rows leave most CUs idle, by one wave's walk: products
// that each wait for the one before them, 32 cycles for 4 k (16 us for K = 4,608), and about as much again for the lane swaps
// and waits between them.
#define F32R_BK 32
#define F32R_SETS 8
struct RowsF32Set {
    f32x4 w[F32R_BK / 16], x[F32R_BK / 16];     // (whole vectors until they are used)
};

__device__ __forceinline__ void swap_lanes_16(float& a, float& b) {
    const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(a), __float_as_uint(b), false, false);
    a = __uint_as_float(r[0]);
    b = __uint_as_float(r[1]);
}
__device__ __forceinline__ void swap_lanes_32(float& a, float& b) {
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(a), __float_as_uint(b), false, false);
    a = __uint_as_float(r[0]);
    b = __uint_as_float(r[1]);
}
// lane group g, component c  ->  lane group c, component g
__device__ __forceinline__ void transpose_over_groups(const f32x4& from, float (&v)[4]) {
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] = from[i];
    swap_lanes_32(v[0], v[2]);
    swap_lanes_32(v[1], v[3]);
    swap_lanes_16(v[0], v[1]);
    swap_lanes_16(v[2], v[3]);
}

template <typename TOut>
__global__ __launch_bounds__(64) void k_gemm_f32_rows(const float* __restrict__ X, const float* __restrict__ W,
                                                      const float* __restrict__ bias, TOut* __restrict__ Y,
                                                      int M, int N, int K, Epilogue epilogue) {
    const int lane = threadIdx.x, r16 = lane & 15, g = lane >> 4;
    const int n0 = blockIdx.x * 16;
    // (uniform bases and 32-bit offsets inside 16 rows: a load in the loop costs no address arithmetic)
    const float* wbase = W + (size_t)n0 * K;
    const unsigned woff = (unsigned)min(r16, N - 1 - n0) * (unsigned)K + g * 4, xoff = (unsigned)min(r16, M - 1) * (unsigned)K + g * 4;
    const int full = K / F32R_BK;                        // whole chunks; the rest of K comes last
    auto fetch = [&](int chunk, RowsF32Set& f) __attribute__((always_inline)) {
        const char* w0 = reinterpret_cast<const char*>(wbase + min(chunk, full - 1) * F32R_BK);
        const char* x0 = reinterpret_cast<const char*>(X + min(chunk, full - 1) * F32R_BK);
#pragma unroll
        for (int j = 0; j < F32R_BK / 16; ++j) {
            f.w[j] = *reinterpret_cast<const f32x4_any*>(w0 + woff * 4u + j * 64);
            f.x[j] = *reinterpret_cast<const f32x4_any*>(x0 + xoff * 4u + j * 64);
        }
    };
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
    auto multiply = [&](const RowsF32Set& f) __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < F32R_BK / 16; ++j) {
            float w[4], x[4];
            transpose_over_groups(f.w[j], w);
            transpose_over_groups(f.x[j], x);
#pragma unroll
            for (int i = 0; i < 4; ++i) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(w[i], x[i], acc, 0, 0, 0);
        }
    };
    if (full > 0) {
        RowsF32Set set[F32R_SETS];
        // (in the order they are used: a first use whose loads were issued last would wait for all of them, every round)
#pragma unroll
        for (int i = 0; i < F32R_SETS - 1; ++i) {
            fetch(i, set[i]);
            __builtin_amdgcn_sched_barrier(0);
        }
        const int rounds = full / F32R_SETS * F32R_SETS;
        for (int c = 0; c < rounds; c += F32R_SETS) {
#pragma unroll
            for (int i = 0; i < F32R_SETS; ++i) {
                fetch(c + i + F32R_SETS - 1, set[(i + F32R_SETS - 1) % F32R_SETS]);
                __builtin_amdgcn_sched_barrier(0);       // (left alone, the compiler sinks the loads to where they are used)
                multiply(set[i]);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
#pragma unroll
        for (int i = 0; i < F32R_SETS - 1; ++i)          // the chunks beyond whole rounds: their loads are on their way
            if (rounds + i < full) multiply(set[i]);
    }
    if (full * F32R_BK < K) {
        RowsF32Set f;
#pragma unroll
        for (int j = 0; j < F32R_BK / 16; ++j) {         // what lies past K counts as zeros
            const int k = full * F32R_BK + j * 16 + g * 4;
            if (K % 4 == 0) {
                const int at = min(k, K - 4) - g * 4;
                f.w[j] = *reinterpret_cast<const f32x4_any*>(wbase + ((long long)woff + at));
                f.x[j] = *reinterpret_cast<const f32x4_any*>(X + ((long long)xoff + at));
            } else {
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const int at = min(k + i, K - 1) - g * 4;
                    f.w[j][i] = wbase[(long long)woff + at];
                    f.x[j][i] = X[(long long)xoff + at];
                }
            }
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                f.w[j][i] = k + i < K ? f.w[j][i] : 0.f;
                f.x[j][i] = k + i < K ? f.x[j][i] : 0.f;
            }
        }
        multiply(f);
    }
    f32_rows_out<TOut>(acc, bias, Y, r16, n0 + g * 4, M, N, epilogue);
}

// The same with K a multiple of 64 and operands that start at multiples of 16 bytes: through a ring of S stages of 64 k in
// LDS that the loads go straight into, no more than the chain of products in the wave's way. A row's 16 pieces of four k lie
// in the order piece ^ (row % 16): product i wants k = 4 i + g of row r in lane (r, g), which are 64 different banks, so the
// operands come from LDS as the products want them, without lane swaps. A wave is a block and has its ring to itself: no
// barriers, it counts its own loads. XI: load instructions for the activations of a stage, four rows each. Bound by the
// chain, 32 cycles for 4 k, where the weight has few rows, by its bytes where it has many.
// Measured, cold weights, 2 rows (the kernel above): 1,024 by 1,024 6.5 us (9.0), 1,024 by 4,608 20 (33), 9,216 by 1,024 10.6
// (12.0), 65,536 by 1,024 51 (56); 16 rows of 9,216 by 1,024 11 (15.6).
template <typename TOut, int S, int XI>
__global__ __launch_bounds__(64) void k_gemm_f32_rows_ring(const float* __restrict__ X, const float* __restrict__ W,
                                                           const float* __restrict__ bias, TOut* __restrict__ Y,
                                                           int M, int N, int K, Epilogue epilogue) {
    constexpr int STAGE = (16 + 4 * XI) * 64;               // floats
    static_assert((S - 1) * (4 + XI) <= 63 && S * STAGE * 4 <= 65536, "loads a wave can count, and LDS in reach of an offset");
    __shared__ __attribute__((aligned(1024))) float ring[S * STAGE];
    const int lane = threadIdx.x, r16 = lane & 15, g = lane >> 4;
    const int n0 = blockIdx.x * 16;
    const int n_chunks = K / 64;
    // loading: an instruction fills four rows; lane -> row lane / 16, place lane % 16, where piece place ^ (row % 16) lies.
    // Uniform bases that walk along K and offsets inside 16 rows that stay: a load takes three instructions.
    unsigned offset[4 + XI];
#pragma unroll
    for (int q = 0; q < 4 + XI; ++q) {
        const int row = (q < 4 ? q * 4 : (q - 4) * 4) + (lane >> 4);
        offset[q] = ((unsigned)(q < 4 ? min(row, N - 1 - n0) : min(row, M - 1)) * (unsigned)K + ((lane & 15) ^ row) * 4) * 4u;
    }
    const float* wbase = W + (size_t)n0 * K;
    const unsigned lds = (unsigned)(size_t)(__attribute__((address_space(3))) float*)ring;
    auto load = [&](int stage, int chunk, int q) __attribute__((always_inline)) {      // (past the end: the last chunk again, nobody reads it)
        load_to_lds_uncounted((q < 4 ? wbase : X) + min(chunk, n_chunks - 1) * 64, offset[q],
                              __builtin_amdgcn_readfirstlane(lds + stage * STAGE * 4 + q * 1024));
    };
    const int x_row = min(r16, M - 1);
    int w_at[16], x_at[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        w_at[i] = r16 * 64 + ((i ^ r16) << 2) + g;
        x_at[i] = 1024 + x_row * 64 + ((i ^ x_row) << 2) + g;
    }
    struct Operands {
        float w[16], x[16];
    };
    auto read = [&](int stage, Operands& o, int i) __attribute__((always_inline)) {
        o.w[i] = ring[stage * STAGE + w_at[i]];
        o.x[i] = ring[stage * STAGE + x_at[i]];
    };
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
    Operands even, odd;
    // Chunk c of 16 products: its operands are in registers or about to be, chunks c + 1 to c + S - 1 are on their way.
    // Between one product and the next, which waits for it, the operands of chunk c + 1 are read and the loads of chunk
    // c + S go out into the stage that chunk c was read from.
    auto step = [&](int stage, int c, const Operands& now, Operands& next) __attribute__((always_inline)) {
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"((S - 2) * (4 + XI)) : "memory");
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            acc = __builtin_amdgcn_mfma_f32_16x16x4f32(now.w[i], now.x[i], acc, 0, 0, 0);
            if (i < 8) {                                  // (so early that the last of them is there when the chunk ends)
                read((stage + 1) % S, next, 2 * i);
                read((stage + 1) % S, next, 2 * i + 1);
            }
            if (i < 4 + XI) load(stage, c + S, i);
            __builtin_amdgcn_sched_barrier(0);
        }
    };
#pragma unroll
    for (int i = 0; i < S; ++i)
#pragma unroll
        for (int q = 0; q < 4 + XI; ++q) load(i, i, q);
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"((S - 1) * (4 + XI)) : "memory");
#pragma unroll
    for (int i = 0; i < 16; ++i) read(0, even, i);
    static_assert(S % 2 == 0, "two register sets in turn");
    for (int c = 0; c < n_chunks; c += S) {
#pragma unroll
        for (int i = 0; i < S; i += 2) {
            if (c + i < n_chunks) step(i, c + i, even, odd);
            if (c + i + 1 < n_chunks) step(i + 1, c + i + 1, odd, even);
        }
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");        // nothing may land in LDS that is another block's
    f32_rows_out<TOut>(acc, bias, Y, r16, n0 + g * 4, M, N, epilogue);
}

template <typename TOut>
static int launch_f32(const float* x, const float* w, const float* bias, TOut* y, int m, int n, int k, Epilogue epilogue,
                      hipStream_t s) {
    const unsigned rows_blocks = (unsigned)((n + 15) / 16);
    // (from K of 256 on: with less the ring is hardly filled before it is empty, 1 row of 512 by 64 2.6 us and 2.2 without, by 128
    // 3.1 and 2.9, by 256 3.6 and 3.8)
    if (m <= 16 && k % 64 == 0 && k >= 256 && k < (1 << 25) && !(((uintptr_t)x | (uintptr_t)w) & 15)) {
        // stages: as many as keep a wave alone on its CU supplied, fewer where more waves share the CU and its LDS (9,216 by
        // 1,024: 8 stages 11.1 us, 4 10.6)
        if (m <= 4 && rows_blocks <= 512)
            k_gemm_f32_rows_ring<TOut, 12, 1><<<rows_blocks, 64, 0, s>>>(x, w, bias, y, m, n, k, epilogue);
        else if (m <= 4)
            k_gemm_f32_rows_ring<TOut, 4, 1><<<rows_blocks, 64, 0, s>>>(x, w, bias, y, m, n, k, epilogue);
        else if (rows_blocks <= 512)
            k_gemm_f32_rows_ring<TOut, 8, 4><<<rows_blocks, 64, 0, s>>>(x, w, bias, y, m, n, k, epilogue);
        else
            k_gemm_f32_rows_ring<TOut, 4, 4><<<rows_blocks, 64, 0, s>>>(x, w, bias, y, m, n, k, epilogue);
        return launch_status();
    }
    if (m <= 16 && k < (1 << 25)) {                  // (offsets inside 16 rows are kept in 32 bits)
        k_gemm_f32_rows<TOut><<<(unsigned)((n + 15) / 16), 64, 0, s>>>(x, w, bias, y, m, n, k, epilogue);
        return launch_status();
    }
    if (m > 65535 * F32Tile<false>::M) return IMPARO_BAD_ARGUMENT;
    auto tiles = [](int rows, bool small) { return (rows - 1) / (small ? F32Tile<true>::M : F32Tile<false>::M) + 1; };
    // The smaller tile where it loads the CUs so much more evenly that its twice the operands a product cost less: what a launch takes
    // goes by the blocks of its fullest CU. 2,048 rows of weight by 8,192, us by blocks a CU: 64x64 one 162, two 284, three 424; 32x32 one
    // 70, two 110, three 154, four 197, six 292. (So 16 to 128 rows by 2,048 by 1,024 24.4 -> 12.3 us, 666 by 1,024 by 4,608 95 -> 89.)
    auto a_cu = [&](bool small) { return ((long long)tiles(m, small) * tiles(n, small) + 255) / 256; };
    // (With three blocks a CU it takes a longer K and rows on 16 bytes: 666 rows by 1,024 by 8 6.0 us and 4.7, by 300 11.3 and 11.7, 64
    // rows by 9,216 by 1,024 off 16 30.1 and 28.6. With two more than one step of the other tile: 541 rows by 768 by 4 to 32 4.3 us and
    // 3.9, by 48 4.3 and 4.8.)
    const bool at_16 = k % 4 == 0 && !(((uintptr_t)x | (uintptr_t)w) & 15);
    const bool small = k >= 4 && 5 * a_cu(true) + 3 < 14 * a_cu(false) + 5 && (a_cu(true) <= (k > 32 ? 2 : 1) || (k >= 256 && at_16));
    const int tiles_m = tiles(m, small), tiles_n = tiles(n, small);
    const long long total = (long long)tiles_m * tiles_n;
    if (total > 0x7f000000LL) return IMPARO_BAD_ARGUMENT;
    // (a launch holds fewer than 2^32 threads along x)
    const long long row = std::min<long long>((total + 7) / 8 * 8, 1LL << 23);
    const dim3 blocks((unsigned)row, (unsigned)((total + row - 1) / row));
    if (small)
        k_gemm_f32<TOut, true, true><<<blocks, 256, 0, s>>>(x, w, bias, y, m, n, k, tiles_m, tiles_n, epilogue);
    else if (k >= 4)
        k_gemm_f32<TOut, true, false><<<blocks, 256, 0, s>>>(x, w, bias, y, m, n, k, tiles_m, tiles_n, epilogue);
    else
        k_gemm_f32<TOut, false, false><<<blocks, 256, 0, s>>>(x, w, bias, y, m, n, k, tiles_m, tiles_n, epilogue);
    return launch_status();
}

// ------------------------------------------------------------------ bfloat16, many rows
// 128x128 output tile per block of four waves (2x2, 64x64 each as 2x2 MFMA
// tiles of 32x32x16), K in steps of 64. Global loads run three K-steps ahead
// in registers, LDS is double-buffered, one barrier per K-step. Blocks are
// numbered so that those sharing rows of X and W sit on the same XCD (blocks
// go to the 8 XCDs round-robin, each XCD has its own L2).
#define BG_BM 128
#define BG_BN 128
#define BG_BK 64
#define BG_LD 72   // LDS row stride in elements: 144 bytes keeps 16-byte reads of 16 rows on distinct banks
#define BG_PF 3    // K-steps in flight
#define BG_GROUP_M 8
#define N_XCD 8

template <typename TOut>
__global__ __launch_bounds__(256, 2) void k_gemm_bf16_tile(const bf16_t* __restrict__ X, const bf16_t* __restrict__ W,
                                                           const float* __restrict__ bias, TOut* __restrict__ Y,
                                                           int M, int N, int K_all, int tiles_m, int tiles_n,
                                                           Epilogue epilogue, int k_per) {
    __shared__ __attribute__((aligned(16))) bf16_t As[2][BG_BM * BG_LD];
    __shared__ __attribute__((aligned(16))) bf16_t Bs[2][BG_BN * BG_LD];
    // slices of K (gridDim.y > 1): block (x, y) sums K range [y * k_per, (y+1) * k_per) into Y + y * M * N
    const int k_lo = blockIdx.y * k_per;
    const int K = min(K_all, k_lo + k_per) - k_lo;
    X += k_lo;
    W += k_lo;
    Y += (size_t)blockIdx.y * M * N;
    if (blockIdx.y > 0) bias = nullptr;
    // block id -> tile: consecutive logical ids on one XCD, grouped over 8 tile rows
    const int total = tiles_m * tiles_n;
    const int per_xcd = (total + N_XCD - 1) / N_XCD;
    const int logical = (blockIdx.x % N_XCD) * per_xcd + blockIdx.x / N_XCD;
    if (logical >= total) return;
    const int per_group = BG_GROUP_M * tiles_n;
    const int first_m = (logical / per_group) * BG_GROUP_M;
    const int gsize = min(tiles_m - first_m, BG_GROUP_M);
    const int tile_m = first_m + (logical % per_group) % gsize;
    const int tile_n = (logical % per_group) / gsize;

    const int tid = threadIdx.x;
    const int lane = tid & 63, wave = tid >> 6;
    const int wm = wave >> 1, wn = wave & 1;
    const int m0 = tile_m * BG_BM, n0 = tile_n * BG_BN;

    // this thread's four 16-byte pieces of each operand tile: rows tid/8 + 32 j, columns (tid%8)*8
    const int kc8 = (tid & 7) * 8;
    const bf16_t* pa[4];
    const bf16_t* pb[4];
    int lds_off[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const int row = (tid >> 3) + 32 * j;
        pa[j] = X + (size_t)min(m0 + row, M - 1) * K_all;
        pb[j] = W + (size_t)min(n0 + row, N - 1) * K_all;
        lds_off[j] = row * BG_LD + kc8;
    }
    const int nk = (K + BG_BK - 1) / BG_BK;
    // three register sets, one per K-step in flight (named apart so that they stay in registers)
    uint4 a0[4], b0[4], a1[4], b1[4], a2[4], b2[4];

    // No load sits under a branch (the compiler would wait for every load in flight at the
    // next use of any): addresses are clamped into the row, a step past the end reads the
    // last one again, and what a cut step reads at or beyond K is zeroed on its way to LDS.
    auto fetch = [&](int kt, uint4 (&a)[4], uint4 (&b)[4]) {
        const int k = min(min(kt, nk - 1) * BG_BK + kc8, K - 8);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            a[j] = *reinterpret_cast<const uint4*>(pa[j] + k);
            b[j] = *reinterpret_cast<const uint4*>(pb[j] + k);
        }
    };
    auto stash = [&](int kt, int buf, uint4 (&a)[4], uint4 (&b)[4]) {
        if ((kt + 1) * BG_BK > K) {                               // only a cut step, or one past the end
            const bool out = kt * BG_BK + kc8 >= K;
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                a[j] = zero_if(out, a[j]);
                b[j] = zero_if(out, b[j]);
            }
        }
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            *reinterpret_cast<uint4*>(&As[buf][lds_off[j]]) = a[j];
            *reinterpret_cast<uint4*>(&Bs[buf][lds_off[j]]) = b[j];
        }
    };

    f32x16 acc[2][2];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;

    const int frag_row = lane & 31, frag_k = (lane >> 5) * 8;
    const int a_base = (wm * 64 + frag_row) * BG_LD + frag_k;
    const int b_base = (wn * 64 + frag_row) * BG_LD + frag_k;
    // The operand fragments of K-sub-step ks+1 are read from LDS while the products of sub-step ks
    // run: without that every sub-step waits a full LDS latency before its first product.
    auto read_frags = [&](int buf, int ks, Frag8 (&fa)[2], Frag8 (&fb)[2]) {
#pragma unroll
        for (int ii = 0; ii < 2; ++ii)
            fa[ii].u = *reinterpret_cast<const uint4*>(&As[buf][a_base + ii * 32 * BG_LD + ks * 16]);
#pragma unroll
        for (int jj = 0; jj < 2; ++jj)
            fb[jj].u = *reinterpret_cast<const uint4*>(&Bs[buf][b_base + jj * 32 * BG_LD + ks * 16]);
    };
    auto multiply = [&](const Frag8 (&fa)[2], const Frag8 (&fb)[2]) {
#pragma unroll
        for (int ii = 0; ii < 2; ++ii)
#pragma unroll
            for (int jj = 0; jj < 2; ++jj)
                acc[ii][jj] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[ii].v, fb[jj].v, acc[ii][jj], 0, 0, 0);
    };
    auto compute = [&](int buf) {
        Frag8 fa0[2], fb0[2], fa1[2], fb1[2];
        read_frags(buf, 0, fa0, fb0);
        read_frags(buf, 1, fa1, fb1);
        __builtin_amdgcn_sched_barrier(0);
        multiply(fa0, fb0);
        read_frags(buf, 2, fa0, fb0);
        __builtin_amdgcn_sched_barrier(0);
        multiply(fa1, fb1);
        read_frags(buf, 3, fa1, fb1);
        __builtin_amdgcn_sched_barrier(0);
        multiply(fa0, fb0);
        __builtin_amdgcn_sched_barrier(0);
        multiply(fa1, fb1);
    };
    // K-step i: the next step's tile goes from its registers to LDS, those registers
    // take the load of step i+1+BG_PF, then step i is multiplied out of LDS
    auto step = [&](int i, uint4 (&na)[4], uint4 (&nb)[4]) {
        const int buf = i & 1;
        stash(i + 1, buf ^ 1, na, nb);
        fetch(i + 1 + BG_PF, na, nb);
        compute(buf);
        __syncthreads();
    };

    fetch(0, a0, b0);
    fetch(1, a1, b1);
    fetch(2, a2, b2);
    stash(0, 0, a0, b0);
    fetch(3, a0, b0);
    __syncthreads();
    int kt = 0;
    for (; kt + BG_PF <= nk; kt += BG_PF) {        // whole rounds of the three sets, free of branches
        step(kt, a1, b1);
        step(kt + 1, a2, b2);
        step(kt + 2, a0, b0);
    }
    if (kt < nk) {
        step(kt, a1, b1);
        if (kt + 1 < nk) step(kt + 1, a2, b2);
    }
    // D layout of the 32x32 tile: lane holds column lane%32, rows 8*(r/4) + 4*(lane/32) + r%4
    float bns[2];
#pragma unroll
    for (int j = 0; j < 2; ++j) bns[j] = bias && n0 + wn * 64 + j * 32 + (lane & 31) < N ? bias[n0 + wn * 64 + j * 32 + (lane & 31)] : 0.f;
    asm volatile("" : "+v"(bns[0]), "+v"(bns[1]));     // waited for here: a store under a condition would wait for it, and for the store before
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const int n = n0 + wn * 64 + j * 32 + (lane & 31);
            const float bn = bns[j];
            if (epilogue == EPI_SWIGLU) {
                // gate and up of one output sit in neighbouring lanes (n even, n odd)
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    const float mine = acc[i][j][r] + bn;
                    const float other = lane_xor<1>(mine);
                    const int m = m0 + wm * 64 + i * 32 + (r >> 2) * 8 + (lane >> 5) * 4 + (r & 3);
                    if (!(lane & 1) && n + 1 < N && m < M)
                        store_f32<TOut>(Y, (size_t)m * (N / 2) + n / 2, gated_mul_fast(epilogue, mine, other));
                }
                continue;
            }
            if (n >= N) continue;
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const int m = m0 + wm * 64 + i * 32 + (r >> 2) * 8 + (lane >> 5) * 4 + (r & 3);
                if (m < M) store_f32<TOut>(Y, (size_t)m * N + n, acc[i][j][r] + bn);
            }
        }
}

// ------------------------------------------------------------------ bfloat16, many rows, large tiles
// The throughput of these tile kernels follows the number of products per fragment read from
// LDS: the 128x128 kernel's waves (2x2 MFMA tiles each) read one 1 KB fragment per product and
// reach 660-700 TFLOP/s, a 256x128 tile with the same ratio reaches the same, and this kernel's
// 256x256 tile (a WM x WN grid of waves, each TM x TN MFMA tiles of 32x32; with 4x2 tiles a wave
// reads three fragments per four products) reaches 830-900. Counters say the matrix pipes are
// busy a third of the time and LDS a quarter: what is exposed is the wait for fragments, with
// two waves per SIMD to hide it. One block per CU (its LDS holds two K-steps of both operands),
// global loads two K-steps ahead in registers. (Four waves of 128x128 each halve the reads per
// product again, but only fit the register file when the operands bypass it: the kernel after
// this one, which takes K in multiples of 128; this one takes the rest.)
template <typename TOut, int WM, int WN, int TM, int TN>
__global__ __launch_bounds__(WM * WN * 64) void k_gemm_bf16_big(const bf16_t* __restrict__ X,
                                                                const bf16_t* __restrict__ W,
                                                                const float* __restrict__ bias,
                                                                TOut* __restrict__ Y, int M, int N, int K,
                                                                int tiles_m, int tiles_n, Epilogue epilogue) {
    constexpr int BM = WM * TM * 32, BN = WN * TN * 32, NT = WM * WN * 64;
    constexpr int PA = BM * 8 / NT, PB = BN * 8 / NT;      // 16-byte pieces of a K-step per thread
    static_assert(BM * 8 % NT == 0 && BN * 8 % NT == 0, "tile rows must divide over the threads");
    extern __shared__ __attribute__((aligned(16))) bf16_t lds[];
    bf16_t* As = lds;                                      // [2][BM * BG_LD]
    bf16_t* Bs = lds + 2 * BM * BG_LD;                     // [2][BN * BG_LD]
    const int total = tiles_m * tiles_n;
    const int per_xcd = (total + N_XCD - 1) / N_XCD;
    const int logical = (blockIdx.x % N_XCD) * per_xcd + blockIdx.x / N_XCD;
    if (logical >= total) return;
    const int per_group = BG_GROUP_M * tiles_n;
    const int first_m = (logical / per_group) * BG_GROUP_M;
    const int gsize = min(tiles_m - first_m, BG_GROUP_M);
    const int tile_m = first_m + (logical % per_group) % gsize;
    const int tile_n = (logical % per_group) / gsize;

    const int tid = threadIdx.x;
    const int lane = tid & 63, wave = tid >> 6;
    const int wm = wave / WN, wn = wave % WN;
    const int m0 = tile_m * BM, n0 = tile_n * BN;
    const int kc8 = (tid & 7) * 8;
    const bf16_t* pa[PA];
    const bf16_t* pb[PB];
    int la[PA], lb[PB];
#pragma unroll
    for (int j = 0; j < PA; ++j) {
        const int row = (tid >> 3) + (NT / 8) * j;
        pa[j] = X + (size_t)min(m0 + row, M - 1) * K;
        la[j] = row * BG_LD + kc8;
    }
#pragma unroll
    for (int j = 0; j < PB; ++j) {
        const int row = (tid >> 3) + (NT / 8) * j;
        pb[j] = W + (size_t)min(n0 + row, N - 1) * K;
        lb[j] = row * BG_LD + kc8;
    }
    const int nk = (K + BG_BK - 1) / BG_BK;
    uint4 a0[PA], b0[PB], a1[PA], b1[PB];
    // as in the 128x128 kernel: no load under a branch, addresses clamped, cut steps zeroed on the way to LDS
    auto fetch = [&](int kt, uint4 (&a)[PA], uint4 (&b)[PB]) {
        const int k = min(min(kt, nk - 1) * BG_BK + kc8, K - 8);
#pragma unroll
        for (int j = 0; j < PA; ++j) a[j] = *reinterpret_cast<const uint4*>(pa[j] + k);
#pragma unroll
        for (int j = 0; j < PB; ++j) b[j] = *reinterpret_cast<const uint4*>(pb[j] + k);
    };
    auto stash = [&](int kt, int buf, uint4 (&a)[PA], uint4 (&b)[PB]) {
        if ((kt + 1) * BG_BK > K) {
            const bool out = kt * BG_BK + kc8 >= K;
#pragma unroll
            for (int j = 0; j < PA; ++j) a[j] = zero_if(out, a[j]);
#pragma unroll
            for (int j = 0; j < PB; ++j) b[j] = zero_if(out, b[j]);
        }
#pragma unroll
        for (int j = 0; j < PA; ++j) *reinterpret_cast<uint4*>(&As[buf * BM * BG_LD + la[j]]) = a[j];
#pragma unroll
        for (int j = 0; j < PB; ++j) *reinterpret_cast<uint4*>(&Bs[buf * BN * BG_LD + lb[j]]) = b[j];
    };
    f32x16 acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;
    const int frag_row = lane & 31, frag_k = (lane >> 5) * 8;
    const int a_base = (wm * TM * 32 + frag_row) * BG_LD + frag_k;
    const int b_base = (wn * TN * 32 + frag_row) * BG_LD + frag_k;
    // (reading the fragments of sub-step ks+1 by hand before the products of ks, as the 128x128
    // kernel does, costs registers this tile does not have: it spills and runs slower)
    auto compute = [&](int buf) {
#pragma unroll
        for (int ks = 0; ks < BG_BK / 16; ++ks) {
            Frag8 fa[TM], fb[TN];
#pragma unroll
            for (int i = 0; i < TM; ++i)
                fa[i].u = *reinterpret_cast<const uint4*>(&As[buf * BM * BG_LD + a_base + i * 32 * BG_LD + ks * 16]);
#pragma unroll
            for (int j = 0; j < TN; ++j)
                fb[j].u = *reinterpret_cast<const uint4*>(&Bs[buf * BN * BG_LD + b_base + j * 32 * BG_LD + ks * 16]);
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int j = 0; j < TN; ++j)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[i].v, fb[j].v, acc[i][j], 0, 0, 0);
        }
    };
    auto step = [&](int i, uint4 (&na)[PA], uint4 (&nb)[PB]) {
        const int buf = i & 1;
        stash(i + 1, buf ^ 1, na, nb);
        fetch(i + 3, na, nb);
        compute(buf);
        __syncthreads();
    };
    fetch(0, a0, b0);
    fetch(1, a1, b1);
    stash(0, 0, a0, b0);
    fetch(2, a0, b0);
    __syncthreads();
    for (int kt = 0; kt < nk; kt += 2) {           // rounds of the two sets, free of branches: with an odd
        step(kt, a1, b1);                          // number of K-steps the last round multiplies a step of zeros
        step(kt + 1, a0, b0);
    }
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) {
            const int n = n0 + (wn * TN + j) * 32 + (lane & 31);
            const float bn = (bias && n < N) ? bias[n] : 0.f;
            if (epilogue == EPI_SWIGLU) {
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    const float mine = acc[i][j][r] + bn;
                    const float other = lane_xor<1>(mine);
                    const int m = m0 + (wm * TM + i) * 32 + (r >> 2) * 8 + (lane >> 5) * 4 + (r & 3);
                    if (!(lane & 1) && n + 1 < N && m < M)
                        store_f32<TOut>(Y, (size_t)m * (N / 2) + n / 2, gated_mul_fast(epilogue, mine, other));
                }
                continue;
            }
            if (n >= N) continue;
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const int m = m0 + (wm * TM + i) * 32 + (r >> 2) * 8 + (lane >> 5) * 4 + (r & 3);
                if (m < M) store_f32<TOut>(Y, (size_t)m * N + n, acc[i][j][r] + bn);
            }
        }
}

template <typename TOut, int WM, int WN, int TM, int TN>
static int launch_big(const bf16_t* x, const bf16_t* w, const float* bias, TOut* y, int m, int n, int k, Epilogue epilogue,
                      hipStream_t s) {
    constexpr int BM = WM * TM * 32, BN = WN * TN * 32;
    constexpr size_t lds_bytes = (size_t)2 * (BM + BN) * BG_LD * sizeof(bf16_t);
    static bool configured = false;
    if (!configured) {
        if (hipFuncSetAttribute((const void*)k_gemm_bf16_big<TOut, WM, WN, TM, TN>,
                                hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds_bytes) != hipSuccess)
            return IMPARO_LAUNCH_FAILED;
        configured = true;
    }
    const int tiles_m = (m + BM - 1) / BM, tiles_n = (n + BN - 1) / BN;
    const long long total = (long long)tiles_m * tiles_n;
    const unsigned blocks = (unsigned)(((total + N_XCD - 1) / N_XCD) * N_XCD);
    k_gemm_bf16_big<TOut, WM, WN, TM, TN><<<blocks, WM * WN * 64, lds_bytes, s>>>(x, w, bias, y, m, n, k, tiles_m,
                                                                                 tiles_n, epilogue);
    return launch_status();
}

// ------------------------------------------------------------------ bfloat16, many rows, loads straight into LDS
// A tile of 256 or 128 activation rows by 256, 192 or 128 weight rows, or of 192 by 256, on eight waves, two per
// SIMD, so that one's products run while the other waits or writes its results (12% faster than
// four waves of 128x128 on the gate/up product at 2,048 rows, 5 to 15% on the narrower tiles).
// A wave has 128 (or 64) rows by 64 or 32 of it, 4x2 or 4x1 MFMA tiles of 32x32 (2x2, 2x1 with
// 128 activation rows); the 192 wide tile's waves 64 rows by 96 (2x3). The operands never pass through registers
// on their way in: global_load_lds writes 16 bytes per
// lane straight into LDS, a wave's 64 lanes to 1 KB in a row. LDS rows are the 128 bytes of
// a K-step without padding, so the eight 16-byte pieces of row r are stored in the order
// piece ^ swz(r), swz(r) = (r & 7) ^ ((r >> 3) & 1): the loading lane picks its global piece
// accordingly, and the 16 rows that a quarter of a wave reads for one fragment fall on
// distinct banks. Two stages of 64 KB are two separate arrays: the compiler can then tell
// that reads of one stage need not wait for loads in flight to the other. A wave keeps the
// fragments of the next K-sub-step in flight while it multiplies (two register sets), and the
// barrier of a K-step sits before the last sub-step's products, so the matrix pipe has
// work queued while the waves meet. Needs K a multiple of 128 (two K-steps).
#define DM_BK 64

// TMI, TN: MFMA tiles of 32x32 down a wave's part of the activation rows and across its part of
// the weight rows; NWM, NWN: waves down and across (eight in all). The launcher's plan chooses
// the tile so that the blocks come out in whole rounds of the CUs.
template <typename TOut, int TMI, int TN, int NWN, int NWM = 2, int STAGES = 2>
__global__ __launch_bounds__(64 * NWM * NWN) void k_gemm_bf16_dma(const bf16_t* __restrict__ X, const bf16_t* __restrict__ W,
                                                             const float* __restrict__ bias, TOut* __restrict__ Y,
                                                             int M, int N, int K_all, int k_per, int tiles_m,
                                                             int tiles_n, Epilogue epilogue) {
    constexpr int NW = NWM * NWN;                      // waves of the block
    constexpr int WN = 32 * TN;                        // weight rows of one wave's part
    constexpr int BN = NWN * WN;                       // of the block's tile
    constexpr int WM = 32 * TMI;                       // activation rows of one wave's part
    constexpr int BM = NWM * WM;                       // of the block's tile
    constexpr int LX = BM / (8 * NW), LW = BN / (8 * NW);   // load instructions per wave and K-step
    static_assert(BM % (8 * NW) == 0 && BN % (8 * NW) == 0, "the waves share the tile's rows evenly");
    __shared__ __attribute__((aligned(1024))) bf16_t stage0[(BM + BN) * DM_BK];   // X rows, then W rows
    __shared__ __attribute__((aligned(1024))) bf16_t stage1[(BM + BN) * DM_BK];
    // four stages (a block alone on its CU): the loads of three K-steps in flight while one is multiplied
    static_assert(STAGES == 2 || STAGES == 4, "two stages or four");
    __shared__ __attribute__((aligned(1024))) bf16_t stage2[STAGES == 4 ? (BM + BN) * DM_BK : 8];
    __shared__ __attribute__((aligned(1024))) bf16_t stage3[STAGES == 4 ? (BM + BN) * DM_BK : 8];
    const int total = tiles_m * tiles_n;
    const int per_xcd = (total + N_XCD - 1) / N_XCD;
    const int logical = (blockIdx.x % N_XCD) * per_xcd + blockIdx.x / N_XCD;
    if (logical >= total) return;
    const int per_group = BG_GROUP_M * tiles_n;
    const int first_m = (logical / per_group) * BG_GROUP_M;
    const int gsize = min(tiles_m - first_m, BG_GROUP_M);
    const int tile_m = first_m + (logical % per_group) % gsize;
    const int tile_n = (logical % per_group) / gsize;
    const int m0 = tile_m * BM, n0 = tile_n * BN;
    // slices of K (gridDim.y > 1): block (x, y) sums K range [y * k_per, (y+1) * k_per) into Y + y * M * N
    const int k_lo = blockIdx.y * k_per;
    const int K = min(K_all, k_lo + k_per) - k_lo;
    X += k_lo;
    W += k_lo;
    Y += (size_t)blockIdx.y * M * N;
    if (blockIdx.y > 0) bias = nullptr;

    const int tid = threadIdx.x;
    const int lane = tid & 63, wave = tid >> 6;
    const int wm = wave / NWN, wn = wave % NWN;
    // loading: instruction j of a wave fills rows j*8*NW + wave*8 .. +7; lane -> row lane/8, slot lane%8
    const int load_row = wave * 8 + (lane >> 3);
    const int load_piece = (lane & 7) ^ (lane >> 3) ^ (wave & 1);          // lane%8 ^ swz(row)
    unsigned off_x[LX], off_w[LW];
#pragma unroll
    for (int j = 0; j < LX; ++j)
        off_x[j] = (unsigned)min(m0 + j * 8 * NW + load_row, M - 1) * (unsigned)K_all + load_piece * 8;
#pragma unroll
    for (int j = 0; j < LW; ++j)
        off_w[j] = (unsigned)min(n0 + j * 8 * NW + load_row, N - 1) * (unsigned)K_all + load_piece * 8;
    auto load_step = [&](bf16_t* stage, int kt) __attribute__((always_inline)) {
        const bf16_t* xk = X + (size_t)kt * DM_BK;
        const bf16_t* wk = W + (size_t)kt * DM_BK;
        if (STAGES == 4) {
            const unsigned to = __builtin_amdgcn_readfirstlane(
                (unsigned)(size_t)(__attribute__((address_space(3))) bf16_t*)stage + wave * 8 * DM_BK * 2);
#pragma unroll
            for (int j = 0; j < LX; ++j) load_to_lds_uncounted(xk + off_x[j], to + j * 8 * NW * DM_BK * 2);
#pragma unroll
            for (int j = 0; j < LW; ++j) load_to_lds_uncounted(wk + off_w[j], to + (BM + j * 8 * NW) * DM_BK * 2);
            return;
        }
#pragma unroll
        for (int j = 0; j < LX; ++j) load_to_lds(xk + off_x[j], stage + (j * 8 * NW + wave * 8) * DM_BK);
#pragma unroll
        for (int j = 0; j < LW; ++j) load_to_lds(wk + off_w[j], stage + (BM + j * 8 * NW + wave * 8) * DM_BK);
    };
    // fragments: lane holds row lane%32, K-half lane/32 of a 32x16 piece; sub-step ks is pieces 2ks, 2ks+1
    const int frag_row = lane & 31;
    const int swz = (frag_row & 7) ^ ((frag_row >> 3) & 1);
    const int a_base = (wm * WM + frag_row) * DM_BK + (((lane >> 5) ^ swz) << 3);
    const int b_base = (BM + wn * WN + frag_row) * DM_BK + (((lane >> 5) ^ swz) << 3);
    f32x16 acc[TMI][TN];
#pragma unroll
    for (int i = 0; i < TMI; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;
    auto read = [&](const bf16_t* stage, int ks, Frag8 (&fa)[TMI], Frag8 (&fb)[TN]) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < TMI; ++i)
            fa[i].u = *reinterpret_cast<const uint4*>(&stage[(a_base ^ (ks << 4)) + i * 32 * DM_BK]);
#pragma unroll
        for (int j = 0; j < TN; ++j)
            fb[j].u = *reinterpret_cast<const uint4*>(&stage[(b_base ^ (ks << 4)) + j * 32 * DM_BK]);
    };
    auto multiply = [&](const Frag8 (&fa)[TMI], const Frag8 (&fb)[TN]) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < TMI; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j)
                acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[i].v, fb[j].v, acc[i][j], 0, 0, 0);
    };
    const int nk = K / DM_BK;
    Frag8 fa0[TMI], fb0[TN], fa1[TMI], fb1[TN];
    // K-step kt from `cur`: on entry set 0 holds its first sub-step and the loads of step kt+1
    // into `next` are in flight (and with four stages those of kt+2 and kt+3); on exit set 0 holds
    // the first sub-step of kt+1 and the loads of kt+STAGES into `cur` are in flight. `after`: how many steps
    // follow, as far as it matters (the last ones ask for nothing: with the last step loaded again and again a block
    // of 16 steps on four stages moved a quarter more than it needs)
    auto k_step = [&](bf16_t* cur, bf16_t* next, int kt, auto after) __attribute__((always_inline)) {
        constexpr int AFTER = decltype(after)::value;
        // (the scheduling barriers keep each sub-step's reads and products where they are written:
        // left alone, the compiler sinks the loads of the next step to just before the wait for them)
        read(cur, 1, fa1, fb1);
        multiply(fa0, fb0);
        __builtin_amdgcn_sched_barrier(0);
        read(cur, 2, fa0, fb0);
        multiply(fa1, fb1);
        __builtin_amdgcn_sched_barrier(0);
        read(cur, 3, fa1, fb1);
        multiply(fa0, fb0);
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (AFTER == 0) {
            multiply(fa1, fb1);
            return;
        }
        // this wave's part of `next` has landed and `cur` is read; after the barrier, so for every wave
        if (STAGES == 4) {             // the loads of the steps after `next` stay in flight: a bare barrier
            constexpr int BEYOND = AFTER - 1 < 2 ? (AFTER > 0 ? AFTER - 1 : 0) : 2;
            asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(BEYOND * (LX + LW)) : "memory");
            __builtin_amdgcn_s_barrier();
        } else {
            __syncthreads();
        }
        read(next, 0, fa0, fb0);
        if constexpr (AFTER >= STAGES) load_step(cur, kt + STAGES);
        multiply(fa1, fb1);
        if constexpr (AFTER >= STAGES) {
#pragma unroll
            for (int q = 0; q < TMI * TN; ++q) {        // one product, (one fragment read,) one load or two
                __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                if (q < TMI + TN) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
                if (q < LX + LW - TMI * TN)
                    __builtin_amdgcn_sched_group_barrier(0x020, 2, 0);
                else if (q < LX + LW)
                    __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);
            }
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    constexpr std::integral_constant<int, STAGES> many{};
    if constexpr (STAGES == 4) {
        load_step(stage0, 0);
        load_step(stage1, 1);
        load_step(stage2, 2);
        load_step(stage3, 3);
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"(3 * (LX + LW)) : "memory");
        __builtin_amdgcn_s_barrier();
        read(stage0, 0, fa0, fb0);
        int kt = 0;
        for (; kt + 4 < nk; kt += 4) {                 // K-steps in fours: one loop, one way round it
            k_step(stage0, stage1, kt, many);
            k_step(stage1, stage2, kt + 1, many);
            k_step(stage2, stage3, kt + 2, many);
            k_step(stage3, stage0, kt + 3, many);
        }
        k_step(stage0, stage1, kt, std::integral_constant<int, 3>{});
        k_step(stage1, stage2, kt + 1, std::integral_constant<int, 2>{});
        k_step(stage2, stage3, kt + 2, std::integral_constant<int, 1>{});
        k_step(stage3, stage0, kt + 3, std::integral_constant<int, 0>{});
    } else {
        load_step(stage0, 0);
        __syncthreads();
        load_step(stage1, 1);
        read(stage0, 0, fa0, fb0);
        int kt = 0;
        for (; kt + 2 < nk; kt += 2) {                 // an even number of K-steps: one loop, one way round it
            k_step(stage0, stage1, kt, many);
            k_step(stage1, stage0, kt + 1, many);
        }
        k_step(stage0, stage1, kt, std::integral_constant<int, 1>{});
        k_step(stage1, stage0, kt + 1, std::integral_constant<int, 0>{});
    }
    // The tile leaves from the accumulators, as the matrix pipe left them: a lane has one column (a weight row), lane % 32 of a
    // 32x32 product, of 16 rows, so a store of 64 lanes is two rows of 128 bytes, and the stores of a tile go out one after the
    // other without waiting for anything. Through LDS, 32 rows at a time and 16 bytes a lane as it was before, the waves wrote,
    // waited and read back in turn. Measured with the last steps' loads left out, us before and now: 8,192 rows of 6,144 by 2,048
    // 201 and 178, gate and up of 16,384 by 2,048 469 and 458; 2,048 rows 57.4 and 51.0, 124 and 121, of 2,048 by 2,048 added
    // 27.5 and 24.0, by 8,192 76.4 and 74.9; 520 rows of 6,144 by 2,048 24.0 and 21.4, of 2,048 by 2,048 in two slices 13.3 and 10.9.
    // Of a tile that is cut, every product that lies whole inside goes the same way, and only those on the edge value by value: all
    // value by value 198 rows of 220 by 256 added took 15.0 us, now 5.9, 5,292 of 6,656 by 768 added 167 and 81, 1,881 of 512 by 256
    // 7.7 and 5.0.
    const int l32 = lane & 31, m_lane = m0 + wm * WM + 4 * (lane >> 5), n_lane = n0 + wn * WN + l32;
    const int m_wave = __builtin_amdgcn_readfirstlane(m0 + wm * WM), n_wave = __builtin_amdgcn_readfirstlane(n0 + wn * WN);
    const bool swiglu = epilogue == EPI_SWIGLU;
    const bool adds = epilogue == EPI_ADD;             // (float32 out; the launcher sees to it)
    const bool inside = m0 + BM <= M && n0 + BN <= N;
    constexpr bool FLOAT = std::is_same<TOut, float>::value;
    float bn[TN];
#pragma unroll
    for (int j = 0; j < TN; ++j) bn[j] = bias && n_lane + j * 32 < N ? bias[n_lane + j * 32] : 0.f;
#pragma unroll
    for (int j = 0; j < TN; ++j) asm volatile("" : "+v"(bn[j]));     // waited for here: a store under a condition would wait for it, and for the store before
    if (swiglu) {
        // Gates and ups are neighbouring lanes: of two rows the even lane takes the first one's pair and the odd lane the
        // second's. In bfloat16 two such results of neighbouring columns go on to one lane, of two rows and the next two again.
        const int out_n = N / 2;
        const bool odd = lane & 1, upper = lane & 2;
        const bool fits = !FLOAT && out_n % 2 == 0 && ((uintptr_t)Y & 3) == 0;
        auto gated = [&](const f32x16& a, float b, int r) __attribute__((always_inline)) {       // row r + odd, column l32 / 2
            const float first = a[r] + b, second = a[r + 1] + b;
            const float other = lane_xor<1>(odd ? first : second);
            return gated_mul_fast(epilogue, odd ? other : first, odd ? second : other);
        };
#pragma unroll
        for (int i = 0; i < TMI; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j) {
                const int col = (n0 + wn * WN + j * 32) / 2;
                const bool pairs = fits && (inside || (m_wave + i * 32 + 32 <= M && n_wave + j * 32 + 32 <= N));
#pragma unroll
                for (int r = 0; r < 16; r += 4) {
                    const float lo = gated(acc[i][j], bn[j], r), hi = gated(acc[i][j], bn[j], r + 2);
                    const int m = m_lane + i * 32 + (r >> 2) * 8 + odd;
                    if (pairs) {
                        const float other = lane_xor<2>(upper ? lo : hi);
                        *reinterpret_cast<uint32_t*>(Y + (size_t)(m + (upper ? 2 : 0)) * out_n + col + (l32 >> 2) * 2) =
                            upper ? f32x2_to_bf16x2(other, hi) : f32x2_to_bf16x2(lo, other);
                    } else if (col + (l32 >> 1) < out_n) {
                        if (m < M) store_f32<TOut>(Y, (size_t)m * out_n + col + (l32 >> 1), lo);
                        if (m + 2 < M) store_f32<TOut>(Y, (size_t)(m + 2) * out_n + col + (l32 >> 1), hi);
                    }
                }
            }
        return;
    }
    if constexpr (FLOAT) {
#pragma unroll
        for (int i = 0; i < TMI; ++i) {
            float* dst = Y + (size_t)(m_lane + i * 32) * N + n_lane;
            if (inside) {
                // what the output holds (the epilogue that adds): the rows of a product asked for together
                float held[TN][16];
                if (adds) {
#pragma unroll
                    for (int j = 0; j < TN; ++j)
#pragma unroll
                        for (int r = 0; r < 16; ++r) held[j][r] = dst[(size_t)((r >> 2) * 8 + (r & 3)) * N + j * 32];
                }
#pragma unroll
                for (int r = 0; r < 16; ++r)
#pragma unroll
                    for (int j = 0; j < TN; ++j) {
                        const float v = acc[i][j][r] + bn[j];
                        dst[(size_t)((r >> 2) * 8 + (r & 3)) * N + j * 32] = adds ? held[j][r] + v : v;
                    }
                continue;
            }
#pragma unroll
            for (int j = 0; j < TN; ++j) {
                const int m_first = m_wave + i * 32, n_first = n_wave + j * 32;
                if (m_first >= M || n_first >= N) continue;
                float held[16];
                if (m_first + 32 <= M && n_first + 32 <= N) {
                    if (adds) {
#pragma unroll
                        for (int r = 0; r < 16; ++r) held[r] = dst[(size_t)((r >> 2) * 8 + (r & 3)) * N + j * 32];
                    }
#pragma unroll
                    for (int r = 0; r < 16; ++r) {
                        const float v = acc[i][j][r] + bn[j];
                        dst[(size_t)((r >> 2) * 8 + (r & 3)) * N + j * 32] = adds ? held[r] + v : v;
                    }
                    continue;
                }
                const int left = n_lane + j * 32 < N ? M - (m_lane + i * 32) : 0;      // rows of this lane's column, four of every eight
                if (adds) {                            // (a row outside asks for the first activations: no load under a branch)
#pragma unroll
                    for (int r = 0; r < 16; ++r) {
                        const int row = (r >> 2) * 8 + (r & 3);
                        held[r] = *(row < left ? dst + (size_t)row * N + j * 32 : reinterpret_cast<const float*>(X));
                    }
#pragma unroll
                    for (int r = 0; r < 16; ++r) asm volatile("" : "+v"(held[r]));     // (waited for together, as the bias)
                }
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    const int row = (r >> 2) * 8 + (r & 3);
                    const float v = acc[i][j][r] + bn[j];
                    if (row < left) dst[(size_t)row * N + j * 32] = adds ? held[r] + v : v;
                }
            }
        }
    } else {
        const bool odd = lane & 1, fits = N % 2 == 0 && ((uintptr_t)Y & 3) == 0;
#pragma unroll
        for (int i = 0; i < TMI; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j) {
                const bool pairs = fits && (inside || (m_wave + i * 32 + 32 <= M && n_wave + j * 32 + 32 <= N));
#pragma unroll
                for (int r = 0; r < 16; r += 2) {
                    const float first = acc[i][j][r] + bn[j], second = acc[i][j][r + 1] + bn[j];
                    const int m = m_lane + i * 32 + (r >> 2) * 8 + (r & 3), n = n_lane + j * 32;
                    if (pairs) {                       // (two neighbouring columns of the first row in the even lane, of the second in the odd)
                        const float other = lane_xor<1>(odd ? first : second);
                        *reinterpret_cast<uint32_t*>(Y + (size_t)(m + odd) * N + n - odd) =
                            odd ? f32x2_to_bf16x2(other, second) : f32x2_to_bf16x2(first, other);
                    } else if (n < N) {
                        if (m < M) store_f32<TOut>(Y, (size_t)m * N + n, first);
                        if (m + 1 < M) store_f32<TOut>(Y, (size_t)(m + 1) * N + n, second);
                    }
                }
            }
    }
}

static bool dma_tile_takes(int m, int n, int k) {
    // the operands' offsets are kept in 32 bits
    return k % (2 * DM_BK) == 0 && (long long)m * k < (1LL << 31) && (long long)n * k < (1LL << 31);
}

// Which tile (bm = 256, 192 or 128 activation rows, tn = 4, 3, 2, 1 for 256, 192, 128, 64 weight rows; 192 with
// bm 256 only, 64 with bm 128 only, bm 192 with 256 only), on how many stages, and how many slices of K suit a product of many rows; tn = 0:
// none (a K the kernel does not take). A model of the time, fitted to this machine:
//   - a K-step of 64 takes a block alone on its CU `few` us with few CUs busy and `all` with all 256 (clocks, L2), in
//     between in proportion (the tables below; 192 activation rows suit portions a little over a power of two, a prompt's beside
//     the tokens of other requests);
//   - a tile of 128 rows by 64 weight rows on four waves and four stages makes twice the blocks of the 128x128 tile: with at most
//     128 rows out of a weight that is streamed once, where a block's share of the weights is what bounds such a product, and
//     wherever the larger tiles leave CUs idle (520 rows of 3,072 by 2,048 13.7 us against 16.2);
//   - two blocks fit a CU where their stages take 80 KB or less each (the 128x128 tile on two
//     stages); a step of both then takes `both`, and with two on some CUs only, in between;
//   - the 128x128 tile can instead keep four stages (one block a CU, three steps' loads in flight),
//     which pays where the tiles are one round of the CUs or less;
//   - with one or two tiles down the rows (a decode batch of 65 to 256 rows) every block meets its
//     weights first, and cold: a step then takes 0.55 us at least on two stages and 0.36 on four;
//   - a block's beginning and end take 4.3 us + 0.116 us per MFMA of a SIMD in a K-step
//     (bm * bn / 1024 of them; measured when tiles left through LDS, and kept: the figures for the tiles are fitted beside it);
//   - blocks run in rounds of what fits the chip at once; the operands have to come from memory
//     once (5.5 TB/s) and the results have to go there (7.6 TB/s); a slice beyond the first costs
//     its consumer one more pass over rows x width of float32 (5 TB/s).
// `fixed_slices` > 0: the caller has decided. Then the tile is chosen by what the kernel takes now (240 products of 129 to 6,000 rows,
// two thirds of them over K of 4,224 to 12,800, every tile measured: 0.14 % above the fastest on average and 8 % at most; with
// figures fitted up to K of 4,608 the long ones were 2.8 % above it and 22 % at most, as two 128x128 tiles a CU were held to be
// slower than they are: 641 rows of 8,192 by 9,088 166 us on 128x256, 135 on 128x128). Else the slices are, by the figures they were always
// chosen with: a count once chosen stays, as fewer slices are further from 64 bits (151 rows of 69,516 by 3,584 in two 2.5e-7 and in one
// 3.7e-7), and what a tile is does not change a sum.
struct DmaPlan {
    int bm, tn, slices, stages;
};
struct DmaStep {
    double few, all;
};
struct DmaRates {
    DmaStep t256x256, t256x192, t256x128, t192x256, t128x256, t128x128, t128x128_four, t128x64_four;
    double both;
};
static const DmaRates dma_rates_slices = {{1.03, 1.58}, {0.89, 1.30}, {0.66, 1.08}, {0.95, 1.25}, {0.70, 1.08}, {0.46, 0.78}, {0.33, 0.53},
                                          {0.35, 0.50}, 1.09};
static const DmaRates dma_rates_tile = {{1.06, 1.63}, {0.89, 1.30}, {0.49, 1.13}, {0.96, 1.29}, {0.62, 1.08}, {0.46, 0.81}, {0.37, 0.58},
                                        {0.35, 0.48}, 1.05};
static DmaPlan dma_plan(int m, int n, int k, int fixed_slices) {
    DmaPlan best{0, 0, fixed_slices > 0 ? fixed_slices : 1, 2};
    if (m <= 64 || !dma_tile_takes(m, n, k)) return best;
    const DmaRates& rates = fixed_slices > 0 ? dma_rates_tile : dma_rates_slices;
    double best_cost = 0.0;
    for (int slices : {1, 2, 3, 4, 6, 8}) {            // (3 and 6: a K of 27 or 9 times 256 has no other cut)
        if (fixed_slices > 0 && slices != fixed_slices) continue;
        if (k % (128 * slices) != 0 || (slices > 1 && k / slices < 512)) continue;
        for (int bm = 256; bm >= 128; bm -= 64) {
            const int tiles_m = (m + bm - 1) / bm;
            for (int tn = 4; tn >= 1; --tn) {
                if (tn == 3 && bm != 256) continue;
                if (tn == 1 && bm != 128) continue;
                // (192 rows: the tile is chosen among all, the slices never were)
                if (bm == 192 && (tn != 4 || fixed_slices <= 0 || m <= 128 || k / slices < 256)) continue;
                const int bn = 64 * tn;
                for (int stages = 2; stages <= 4; stages += 2) {
                    // four stages: the 128x128 tile and the 128x64 one (which runs on four only), K-steps in fours
                    if (stages == 4 && (bm != 128 || tn > 2 || (k / slices) % (4 * DM_BK) != 0)) continue;
                    if (stages == 2 && tn == 1) continue;
                    const long long blocks = (long long)tiles_m * ((n + bn - 1) / bn) * slices;
                    const int at_once = 256 * ((bm + bn) * DM_BK * 2 * stages <= 80 * 1024 ? 2 : 1);
                    const long long rounds = (blocks + at_once - 1) / at_once;
                    const long long per_round = (blocks + rounds - 1) / rounds;
                    const double cus = (double)std::min<long long>(256, per_round);
                    const DmaStep& a_step = bm == 192 ? rates.t192x256 : bm == 128 && tn == 1 ? rates.t128x64_four
                                          : bm == 128 && tn == 2 ? (stages == 4 ? rates.t128x128_four : rates.t128x128)
                                          : bm == 128 ? rates.t128x256 : tn == 2 ? rates.t256x128 : tn == 3 ? rates.t256x192 : rates.t256x256;
                    double step = per_round > 256 ? a_step.all + (rates.both - a_step.all) * (per_round - 256) / 256.0    // some CUs, or all, with two
                                                  : a_step.few + (a_step.all - a_step.few) * cus / 256.0;
                    if (tiles_m <= 2) step = std::max(step, stages == 4 ? 0.36 : 0.55);
                    // one tile down the rows: a block streams its weight rows alone, 128 bytes of each a
                    // step, and one CU draws about 28 GB/s of cold weights (0.60 us a step measured on the
                    // 128x128 tile at 128 rows, where the figures above would have it at 0.43)
                    if (tiles_m == 1) step = std::max(step, bn * 128.0 / 28e3);
                    const double ends = 4.3 + 0.116 * (bm * bn / 1024.0);
                    const double from_memory = ((double)m + n) * k * 2.0 / 5.5e6;
                    const double cost = std::max(rounds * (k / slices / DM_BK * step + ends), from_memory + ends) +
                                        (double)slices * m * n * 4.0 / 7.6e6 + (slices - 1) * ((double)m * n * 4.0 / 5e6);
                    if (best.tn == 0 || cost < best_cost) {
                        best = DmaPlan{bm, tn, slices, stages};
                        best_cost = cost;
                    }
                }
            }
        }
    }
    return best;
}

// `slices` must leave every slice a multiple of 128 of K (dma_tile_takes(m, n, k / slices) and k % slices == 0).
// bm: 256, 192 or 128 activation rows to a tile; tn: 4, 3 (bm 256 only), 2 or 1 (bm 128 only) for 256, 192, 128 or 64 weight rows.
template <typename TOut>
static int launch_dma(const bf16_t* x, const bf16_t* w, const float* bias, TOut* y, int m, int n, int k, Epilogue epilogue,
                      int bm, int tn, int slices, hipStream_t s, int stages = 2) {
    const int tiles_m = (m + bm - 1) / bm, tiles_n = (n + 64 * tn - 1) / (64 * tn);
    const long long total = (long long)tiles_m * tiles_n;
    const dim3 grid((unsigned)(((total + N_XCD - 1) / N_XCD) * N_XCD), (unsigned)slices);
#define DMA_GO(TMI, TN, NWN)                                                                                         \
    k_gemm_bf16_dma<TOut, TMI, TN, NWN><<<grid, 128 * NWN, 0, s>>>(x, w, bias, y, m, n, k, k / slices, tiles_m,     \
                                                                   tiles_n, epilogue)
    if (bm == 128 && tn == 1 && stages == 4)   // 64 wide: four waves of 64 rows by 32
        k_gemm_bf16_dma<TOut, 2, 1, 2, 2, 4><<<grid, 256, 0, s>>>(x, w, bias, y, m, n, k, k / slices, tiles_m, tiles_n, epilogue);
    else if (bm == 128 && tn == 1)
        k_gemm_bf16_dma<TOut, 2, 1, 2, 2, 2><<<grid, 256, 0, s>>>(x, w, bias, y, m, n, k, k / slices, tiles_m, tiles_n, epilogue);
    else if (bm == 128 && tn == 4)
        DMA_GO(2, 2, 4);
    else if (bm == 128 && stages == 4)
        k_gemm_bf16_dma<TOut, 2, 1, 4, 2, 4><<<grid, 512, 0, s>>>(x, w, bias, y, m, n, k, k / slices, tiles_m, tiles_n, epilogue);
    else if (bm == 128)
        DMA_GO(2, 1, 4);
    else if (bm == 192)   // 256 wide: eight waves of 96 rows by 64
        DMA_GO(3, 2, 4);
    else if (tn == 4)     // 256 wide: eight waves
        DMA_GO(4, 2, 4);
    else if (tn == 3)     // 192 wide: eight waves of 64 rows by 96
        k_gemm_bf16_dma<TOut, 2, 3, 2, 4><<<grid, 512, 0, s>>>(x, w, bias, y, m, n, k, k / slices, tiles_m, tiles_n, epilogue);
    else                  // 128 wide: eight waves
        DMA_GO(4, 1, 4);
#undef DMA_GO
    return launch_status();
}

// ------------------------------------------------------------------ conv input projection + gated conv, single tokens
// For a decode step's rows (one token each, at most 16): the projection to [B | C | x] and the
// gated short convolution that consumes it in one launch. A block takes 8 channels: its first
// MFMA tile holds the B rows of those channels (tile rows 0..7) and their x rows (8..15), its
// second the C rows (0..7; its other lanes ask for nothing).
// K is split over the waves in chunks of 128, all of whose loads go out at once (CH chunks a wave and
// round, as the products of decode_rows.hip have them), and the partial sums meet in LDS in wave
// order; then 32 lanes of wave 0 each own one token and four channels: u = B * x, the taps
// oldest first exactly as the conv kernels sum them, the C gate, and the shift of the state
// (a lane owns its channels' history, so nothing races). With HIST > 0 the history, the taps
// and the biases are asked for before the walk along K, so they are there when it ends. Measured: 8 rows
// of 2,048 9.3 -> 8.5 us, one row of 1,024 6.2 -> 5.4 (a chunk ahead of the one that is multiplied before).
// With ssq_in, X is the residual stream times a norm's weight, not yet scaled: the partial sums of
// squares of its rows [n_parts, 16] give each row's scale, which multiplies B, C and x at the end (rows.h).
template <typename TOut, int CH, int HIST>
__global__ __launch_bounds__(512) void k_in_proj_conv_decode(
    const bf16_t* __restrict__ X, const float* __restrict__ ssq_in, int n_parts, float eps,
    const bf16_t* __restrict__ W, const float* __restrict__ in_bias,
    const float* __restrict__ conv_w, const float* __restrict__ conv_b, float* __restrict__ state,
    const int32_t* __restrict__ slot, TOut* __restrict__ out, int M, int E, int K, int taps) {
    __shared__ float4 red[8][2][64];
    __shared__ __attribute__((aligned(16))) float norm_part[8 * 16];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), waves = blockDim.x >> 6;
    const int r16 = lane & 15, g = lane >> 4;
    const int c0 = blockIdx.x * 8;
    const bf16_t* wrow0 = W + (size_t)(r16 < 8 ? c0 + r16 : 2 * E + c0 + (r16 - 8)) * K;
    const bf16_t* wrow1 = W + (size_t)(E + c0 + (r16 & 7)) * K;
    const bf16_t* xrow = X + (size_t)min(r16, M - 1) * K;
    const int n_chunks = (K + 127) / 128;
    const int history = HIST > 0 ? HIST : taps - 1;
    // the lanes that finish the block: token r16, channels cb .. cb+3. Where a token's state lies is asked for before all
    // else and its state after the weights: who waits for the one to ask for the other waits with the weights on their way.
    const bool finisher = wave == 0 && g < 2 && r16 < M;
    const int cb = c0 + 4 * (g & 1);
    const int my_slot = finisher ? slot[r16] : 0;
    __builtin_amdgcn_sched_barrier(0);
    Frag8 w0[CH][4], w1[CH][4], x[CH][4];
    auto ask = [&](int first) __attribute__((always_inline)) {
        int k[CH][4];
#pragma unroll
        for (int j = 0; j < CH; ++j)
#pragma unroll
            for (int s2 = 0; s2 < 4; ++s2) k[j][s2] = min(min(first + j * waves, n_chunks - 1) * 128 + s2 * 32 + g * 8, K - 8);
#pragma unroll
        for (int j = 0; j < CH; ++j)
#pragma unroll
            for (int s2 = 0; s2 < 4; ++s2) x[j][s2].u = *reinterpret_cast<const uint4*>(xrow + k[j][s2]);
#pragma unroll
        for (int j = 0; j < CH; ++j)
#pragma unroll
            for (int s2 = 0; s2 < 4; ++s2) {
                w0[j][s2].u = *reinterpret_cast<const uint4*>(wrow0 + k[j][s2]);
                w1[j][s2].u = make_uint4(0u, 0u, 0u, 0u);
                if (r16 < 8) w1[j][s2].u = *reinterpret_cast<const uint4*>(wrow1 + k[j][s2]);
            }
        __builtin_amdgcn_sched_barrier(0);
    };
    // (the rows' sums of squares before the weights: they are added up while those are on their way)
    RowsSsq early;
    if (ssq_in) rows_ssq_ask(early, ssq_in, n_parts, 0);
    __builtin_amdgcn_sched_barrier(0);
    ask(wave);
    if (ssq_in) rows_ssq_share(norm_part, early, ssq_in, n_parts);
    float* st = state + (size_t)my_slot * history * E;
    constexpr int HN = HIST > 0 ? HIST : 1;
    float hist[HN][4], tap[HN + 1][4], bias_b[4], bias_c[4], bias_x[4], bias_conv[4];
    if (HIST > 0 && finisher) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
#pragma unroll
            for (int k = 0; k <= HIST; ++k) tap[k][i] = conv_w[(size_t)(cb + i) * (HIST + 1) + k];
            bias_b[i] = in_bias ? in_bias[cb + i] : 0.f;
            bias_c[i] = in_bias ? in_bias[E + cb + i] : 0.f;
            bias_x[i] = in_bias ? in_bias[2 * E + cb + i] : 0.f;
            bias_conv[i] = conv_b ? conv_b[cb + i] : 0.f;
#pragma unroll
            for (int k = 0; k < HIST; ++k) hist[k][i] = st[(size_t)k * E + cb + i];
        }
    }
    f32x4 acc0 = {0.f, 0.f, 0.f, 0.f}, acc1 = {0.f, 0.f, 0.f, 0.f};
    for (int first = wave; first < n_chunks;) {
#pragma unroll
        for (int j = 0; j < CH; ++j) {
            if (first + j * waves >= n_chunks) continue;
#pragma unroll
            for (int s2 = 0; s2 < 4; ++s2) {             // (what lies beyond K counts as zeros: activations too, which may be infinite)
                const bool beyond = (first + j * waves) * 128 + s2 * 32 + g * 8 >= K;
                x[j][s2].u = zero_if(beyond, x[j][s2].u);
                w0[j][s2].u = zero_if(beyond, w0[j][s2].u);
                w1[j][s2].u = zero_if(beyond, w1[j][s2].u);
                acc0 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w0[j][s2].v, x[j][s2].v, acc0, 0, 0, 0);
                acc1 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w1[j][s2].v, x[j][s2].v, acc1, 0, 0, 0);
            }
        }
        first += waves * CH;
        if (first < n_chunks) ask(first);
    }
    red[wave][0][lane] = make_float4(acc0[0], acc0[1], acc0[2], acc0[3]);
    red[wave][1][lane] = make_float4(acc1[0], acc1[1], acc1[2], acc1[3]);
    __syncthreads();
    if (!finisher) return;
    const float scale = ssq_in ? rows_scale(norm_part, r16, K, eps) : 1.f;
    // D layout: lane holds column lane%16 (a token), tile rows 4*(lane/16) + i: B and C of channel
    // cb + i sit in this lane's entries, x of the same channel 8 tile rows further: lane + 32
    float b[4], c[4], xc[4];
    {
        float4 sb[8], sx[8], sc[8];
#pragma unroll
        for (int q = 0; q < 8; ++q) {
            const int w = min(q, waves - 1);
            sb[q] = red[w][0][lane], sx[q] = red[w][0][lane + 32], sc[q] = red[w][1][lane];
        }
        float4 tb = sb[0], tx = sx[0], tc = sc[0];
#pragma unroll
        for (int q = 1; q < 8; ++q)
            if (q < waves) {
                tb.x += sb[q].x, tb.y += sb[q].y, tb.z += sb[q].z, tb.w += sb[q].w;
                tx.x += sx[q].x, tx.y += sx[q].y, tx.z += sx[q].z, tx.w += sx[q].w;
                tc.x += sc[q].x, tc.y += sc[q].y, tc.z += sc[q].z, tc.w += sc[q].w;
            }
        b[0] = tb.x, b[1] = tb.y, b[2] = tb.z, b[3] = tb.w;
        xc[0] = tx.x, xc[1] = tx.y, xc[2] = tx.z, xc[3] = tx.w;
        c[0] = tc.x, c[1] = tc.y, c[2] = tc.z, c[3] = tc.w;
    }
    if (ssq_in) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            b[i] = __fmul_rn(b[i], scale);
            xc[i] = __fmul_rn(xc[i], scale);
            c[i] = __fmul_rn(c[i], scale);
        }
    }
    float y[4];
    if (HIST > 0) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const float u = (b[i] + bias_b[i]) * (xc[i] + bias_x[i]);
            float a = 0.f;
#pragma unroll
            for (int k = 0; k < HIST; ++k) {
                a = fmaf(tap[k][i], hist[k][i], a);
                st[(size_t)k * E + cb + i] = k + 1 < HIST ? hist[k + 1][i] : u;
            }
            a = fmaf(tap[HIST][i], u, a);
            a += bias_conv[i];
            y[i] = (c[i] + bias_c[i]) * a;
        }
    } else {
        for (int i = 0; i < 4; ++i) {
            const int ch = cb + i;
            const float bv = b[i] + (in_bias ? in_bias[ch] : 0.f);
            const float cv = c[i] + (in_bias ? in_bias[E + ch] : 0.f);
            const float xv = xc[i] + (in_bias ? in_bias[2 * E + ch] : 0.f);
            const float u = bv * xv;
            float a = 0.f;
            float prev = st[ch];                                  // oldest
            for (int k = 0; k < history; ++k) {
                a = fmaf(conv_w[(size_t)ch * taps + k], prev, a);
                const float next = (k + 1 < history) ? st[(size_t)(k + 1) * E + ch] : u;
                st[(size_t)k * E + ch] = next;
                prev = next;
            }
            a = fmaf(conv_w[(size_t)ch * taps + history], u, a);
            a += conv_b ? conv_b[ch] : 0.f;
            y[i] = cv * a;
        }
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) store_f32<TOut>(out, (size_t)r16 * E + cb + i, y[i]);
}

template <typename TOut>
static void launch_in_proj_conv(const bf16_t* x, const float* ssq_in, int n_parts, float eps, const bf16_t* w,
                                const float* in_bias, const float* conv_w, const float* conv_b, float* state,
                                const int32_t* slot, TOut* out, int m, int e, int k, int taps, hipStream_t s) {
    const unsigned blocks = (unsigned)(e / 8);
    // (eight waves from eight chunks on, though some have a chunk less than others: the sums' order of before, and nearer to
    // 64 bits than fewer longer ones)
    const int chunks = (k + 127) / 128, waves = std::min(chunks, 8);
#define CONV_GO(CH, HIST)                                                                                              \
    k_in_proj_conv_decode<TOut, CH, HIST><<<blocks, waves * 64, 0, s>>>(x, ssq_in, n_parts, eps, w, in_bias, conv_w, conv_b, \
                                                                   state, slot, out, m, e, k, taps)
#define CONV_HIST(CH)                                                                                                  \
    do {                                                                                                             \
        switch (taps - 1) {                                                                                          \
            case 1: CONV_GO(CH, 1); break;                                                                             \
            case 2: CONV_GO(CH, 2); break;                                                                             \
            case 3: CONV_GO(CH, 3); break;                                                                             \
            default: CONV_GO(CH, 0);                                                                                   \
        }                                                                                                            \
    } while (0)
    if (chunks <= 8) CONV_HIST(1);
    else CONV_HIST(2);
#undef CONV_HIST
#undef CONV_GO
}

// x [m, k] bfloat16 (m <= 16 single tokens), w [3 e, k] bfloat16, conv_w [e, taps], state
// [n_slots, taps-1, e], slot [m] (distinct): out [m, e] = the gated conv's output, state shifted.
// ssq_in [n_parts, 16] (or null) and eps: x is the residual stream times a norm's weight, each row
// still to be scaled by rsqrt(sum of its partial sums of squares / k + eps), which the launch does.
extern "C" int imparo_in_proj_conv_decode_normed(const void* x, const float* ssq_in, int n_parts, float eps,
                                                 const void* w, const float* in_bias, const float* conv_w,
                                                 const float* conv_b, float* state, const int32_t* slot, void* out,
                                                 int out_dtype, int m, int e, int k, int taps, int n_slots,
                                                 imparo_stream stream) {
    if (!x || !w || !conv_w || !state || !slot || !out) return IMPARO_BAD_ARGUMENT;
    if (ssq_in && (n_parts <= 0 || !(eps > 0.f))) return IMPARO_BAD_ARGUMENT;
    if (m < 0 || m > 16 || e <= 0 || e % 8 != 0 || k <= 0 || k % 8 != 0 || taps < 2 || taps > 64 || n_slots <= 0)
        return IMPARO_BAD_ARGUMENT;
    if (((uintptr_t)x & 15) || ((uintptr_t)w & 15)) return IMPARO_BAD_ARGUMENT;
    if (out_dtype != IMPARO_F32 && out_dtype != IMPARO_BF16) return IMPARO_BAD_ARGUMENT;
    if (m == 0) return IMPARO_OK;
    hipStream_t s = (hipStream_t)stream;
    const bf16_t* xb = (const bf16_t*)x;
    const bf16_t* wb = (const bf16_t*)w;
    if (out_dtype == IMPARO_F32)
        launch_in_proj_conv<float>(xb, ssq_in, n_parts, eps, wb, in_bias, conv_w, conv_b, state, slot, (float*)out, m, e, k, taps, s);
    else
        launch_in_proj_conv<bf16_t>(xb, ssq_in, n_parts, eps, wb, in_bias, conv_w, conv_b, state, slot, (bf16_t*)out, m, e, k, taps, s);
    return launch_status();
}

extern "C" int imparo_in_proj_conv_decode(const void* x, const void* w, const float* in_bias, const float* conv_w,
                                          const float* conv_b, float* state, const int32_t* slot, void* out,
                                          int out_dtype, int m, int e, int k, int taps, int n_slots,
                                          imparo_stream stream) {
    return imparo_in_proj_conv_decode_normed(x, nullptr, 0, 0.f, w, in_bias, conv_w, conv_b, state, slot, out, out_dtype,
                                             m, e, k, taps, n_slots, stream);
}


// The waves a block of the shared-activation kernel, for products of 17 to 64 rows with a K that is no multiple of 128. Measured with cold weights (they never
// stay in cache between decode steps): four from about 12k weight rows on, two below.
static int stream_waves(int n) { return n >= 12288 ? 4 : 2; }

// A slice's length is rounded up to the kernel's step along K; with a ragged K that can leave the
// last slices empty. The consumer adds every slice it was promised: fewer slices then, all of
// them non-empty.
static int whole_slices(int slices, int k, int step) {
    while (slices > 1) {
        const int k_per = ((k + slices - 1) / slices + step - 1) / step * step;
        if ((k + k_per - 1) / k_per == slices) break;
        slices /= 2;
    }
    return slices;
}

// Into how many slices of K a product may be cut when its consumer adds the slices. A weight
// with few rows gives too few blocks to keep the memory system busy otherwise (one CU draws
// about 50 GB/s at best, so it takes all of them): the measured optimum, with cold weights,
// is about 256 blocks, with at least 512 of K per slice and at most 8 slices.
extern "C" int imparo_gemm_slices(int m, int n, int k, int dtype) {
    if (dtype != IMPARO_BF16) return 1;
    if (m > 64) {
        const DmaPlan plan = dma_plan(m, n, k, 0);
        if (plan.tn) return plan.slices;
        // many rows: with about one tile of 128x128 per CU or fewer, a block has a CU to itself and
        // nothing hides its waits; slices of K (at least 1024 each, at most 4) multiply the blocks
        const long long tiles = (long long)((m + BG_BM - 1) / BG_BM) * ((n + BG_BN - 1) / BG_BN);
        int slices = 1;
        while (slices < 4 && tiles * slices * 2 <= 512 && k / (slices * 2) >= 1024) slices *= 2;
        return whole_slices(slices, k, BG_BK);
    }
    // (weight rows a block that the count goes by, those of the kernels it was measured with. The kernels of now take 16 to 64 as
    // the slices and the CUs have it, so that 2,048 by 8,192 in four slices are 256 blocks of 32 and 1,024 by 4,608 in eight 512 of 16;
    // the counts stay, as fewer slices are further from 64 bits)
    const int rows_per_block = n >= 12288 ? 64 : m > 16 || k >= 4096 ? 32 : 16;
    const int blocks = (n + rows_per_block - 1) / rows_per_block;
    int slices = 1;
    while (slices < 8 && blocks * slices * 2 <= 256 && k / (slices * 2) >= 512) slices *= 2;
    return whole_slices(slices, k, 128);
}

// Whether imparo_gemm takes the epilogue that adds the product to what Y holds (float32 out, K in one
// piece) for this shape: where the tile kernel with loads straight into LDS runs it.
extern "C" int imparo_gemm_adds(int m, int n, int k, int dtype) {
    return dtype == IMPARO_BF16 && m > 64 && dma_plan(m, n, k, 1).tn != 0;
}


// ------------------------------------------------------------------ bfloat16, some rows (17..64), any K
// (K a multiple of 128: some_rows.hip)
// A block of ST_WAVES waves takes 16 weight rows per wave and up to 16*MT
// activation rows, and walks its part of K in chunks of 128. The activation
// chunk is staged in LDS once per block and shared by the waves (with more
// than 16 rows every wave fetching its own activations costs several times the
// weight traffic); weights go from memory straight into the MFMA operand
// registers. Loads run three chunks ahead of the products: four register sets
// in rotation, the activation part of a set goes to LDS one step before its
// chunk is multiplied. With slices (gridDim.y > 1) block (x, y) sums K range
// [y * k_per, (y+1) * k_per) into Y + y * M * N and the consumer adds the slices.
#define ST_BK 128
#define ST_LD (ST_BK + 8)   // LDS row stride in elements: 272 bytes, 16 rows of 16-byte reads on distinct banks

template <int XP>
struct StreamSet {
    Frag8 w[4];       // this wave's weight rows, chunk columns s*32 + g*8
    uint4 x[XP];      // this thread's pieces of the activation chunk
};

template <typename TOut, int MT, int ST_WAVES>
__global__ __launch_bounds__(ST_WAVES * 64) void k_gemm_bf16_stream(
    const bf16_t* __restrict__ X, const bf16_t* __restrict__ W, const float* __restrict__ bias,
    TOut* __restrict__ Y, int M, int N, int K_all, int k_per, Epilogue epilogue) {
    __shared__ __attribute__((aligned(16))) bf16_t xs[2][MT * 16 * ST_LD];
    const int tid = threadIdx.x;
    const int lane = tid & 63, wave = tid >> 6;
    const int r16 = lane & 15, g = lane >> 4;
    const int n0 = blockIdx.x * (ST_WAVES * 16) + wave * 16;
    const int k_lo = blockIdx.y * k_per;
    const int K = min(K_all, k_lo + k_per) - k_lo;       // this block's part of K, re-based to 0
    X += k_lo;
    W += k_lo;
    Y += (size_t)blockIdx.y * M * N;
    if (blockIdx.y > 0) bias = nullptr;                  // the bias belongs to one slice only
    const bf16_t* wrow = W + (size_t)min(n0 + r16, N - 1) * K_all;

    // the activation chunk: MT*16 rows x 16 pieces of 16 bytes, XP pieces per thread
    constexpr int PIECES = MT * 16 * (ST_BK / 8);
    constexpr int XP = (PIECES + ST_WAVES * 64 - 1) / (ST_WAVES * 64);
    const bf16_t* xsrc[XP];
    int xdst[XP], xkc[XP];
#pragma unroll
    for (int j = 0; j < XP; ++j) {
        const int p = min(tid + j * ST_WAVES * 64, PIECES - 1);
        const int row = p / (ST_BK / 8);
        xkc[j] = (p % (ST_BK / 8)) * 8;
        xsrc[j] = X + (size_t)min(row, M - 1) * K_all;
        xdst[j] = row * ST_LD + xkc[j];
    }
    const int nk = (K + ST_BK - 1) / ST_BK;
    // The walk along K is free of branches: a load under a branch, or a step under one, makes
    // the compiler wait for every load in flight at the next use of any. So every load is
    // issued unconditionally from an address clamped into the row, what a chunk reads at or
    // beyond K is zeroed before use, and the number of steps is rounded up to the four
    // register sets (a chunk past the end reads the last one again and counts as zeros).
    // Blocks start their walk at different chunks and wrap around: rows are a power of two
    // apart in memory, so blocks in step would ask the same few cache channels for the same
    // activation chunk at the same time.
    const int rot = (blockIdx.x + blockIdx.y) % nk;
    auto chunk_of = [&](int kt) {                        // kt >= nk: past the end
        const int c = kt + rot;
        return kt >= nk ? kt : (c >= nk ? c - nk : c);
    };
    auto fetch = [&](int kt, StreamSet<XP>& f) {
        const int k0 = min(chunk_of(kt), nk - 1) * ST_BK;
#pragma unroll
        for (int s2 = 0; s2 < 4; ++s2)
            f.w[s2].u = *reinterpret_cast<const uint4*>(wrow + min(k0 + s2 * 32 + g * 8, K - 8));
#pragma unroll
        for (int j = 0; j < XP; ++j) f.x[j] = *reinterpret_cast<const uint4*>(xsrc[j] + min(k0 + xkc[j], K - 8));
    };
    // (What an activation chunk holds at or beyond K is real data read again from inside the row; only
    // the weights there are zeroed, in `compute`: one select per weight value instead of one more per
    // activation value, which with 64 rows were a third of the kernel's vector instructions.)
    auto stash = [&](int buf, const StreamSet<XP>& f) {
#pragma unroll
        for (int j = 0; j < XP; ++j)     // threads beyond the last piece repeat it: same value, same place
            *reinterpret_cast<uint4*>(&xs[buf][xdst[j]]) = f.x[j];
    };
    f32x4 acc[MT];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) acc[mt] = f32x4{0.f, 0.f, 0.f, 0.f};
    // The activation fragments of K-sub-step s2+1 are read from LDS while the products of
    // sub-step s2 run: a block may be alone on its CU, with nothing else to hide the LDS latency.
    auto read_x = [&](int buf, int s2, Frag8 (&xf)[MT]) {
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
            xf[mt].u = *reinterpret_cast<const uint4*>(&xs[buf][(mt * 16 + r16) * ST_LD + s2 * 32 + g * 8]);
    };
    auto multiply = [&](const Frag8& wf, const Frag8 (&xf)[MT]) {
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
            acc[mt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf.v, xf[mt].v, acc[mt], 0, 0, 0);
    };
    auto compute = [&](int kt, int buf, const StreamSet<XP>& f) {
        const int k0 = chunk_of(kt) * ST_BK + g * 8;
        Frag8 xa[MT], xb[MT], wf;
        read_x(buf, 0, xa);
        read_x(buf, 1, xb);
        __builtin_amdgcn_sched_barrier(0);
        wf.u = zero_if(k0 >= K, f.w[0].u);
        multiply(wf, xa);
        read_x(buf, 2, xa);
        __builtin_amdgcn_sched_barrier(0);
        wf.u = zero_if(k0 + 32 >= K, f.w[1].u);
        multiply(wf, xb);
        read_x(buf, 3, xb);
        __builtin_amdgcn_sched_barrier(0);
        wf.u = zero_if(k0 + 64 >= K, f.w[2].u);
        multiply(wf, xa);
        __builtin_amdgcn_sched_barrier(0);
        wf.u = zero_if(k0 + 96 >= K, f.w[3].u);
        multiply(wf, xb);
    };
    // chunk i: the next chunk's activations go from their registers to LDS, the set that
    // chunk i-1 used takes the loads of chunk i+3, then chunk i is multiplied
    auto step = [&](int i, const StreamSet<XP>& cur, const StreamSet<XP>& next, StreamSet<XP>& refill) {
        const int buf = i & 1;
        stash(buf ^ 1, next);
        fetch(i + 3, refill);
        compute(i, buf, cur);
        __syncthreads();
    };
    StreamSet<XP> s0, s1, s2, s3;
    fetch(0, s0);
    fetch(1, s1);
    fetch(2, s2);
    stash(0, s0);
    __syncthreads();
    for (int kt = 0; kt < nk; kt += 4) {
        step(kt, s0, s1, s3);
        step(kt + 1, s1, s2, s0);
        step(kt + 2, s2, s3, s1);
        step(kt + 3, s3, s0, s2);
    }
    // D layout of the 16x16 tile: lane holds column lane%16 (an activation row), rows 4*(lane/16)+i (weight rows)
    const int nq = n0 + g * 4;
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
        const int m = mt * 16 + r16;
        if (m >= M) continue;
        float v[4];
#pragma unroll
        for (int i = 0; i < 4; ++i)
            v[i] = acc[mt][i] + ((bias && nq + i < N) ? bias[nq + i] : 0.f);
        if (epilogue == EPI_SWIGLU) {
#pragma unroll
            for (int i = 0; i < 4; i += 2)
                if (nq + i + 1 < N) store_f32<TOut>(Y, (size_t)m * (N / 2) + (nq + i) / 2, gated_mul_fast(epilogue, v[i], v[i + 1]));
            continue;
        }
#pragma unroll
        for (int i = 0; i < 4; ++i)
            if (nq + i < N) store_f32<TOut>(Y, (size_t)m * N + nq + i, v[i]);
    }
}

template <typename TOut, int MT>
static void launch_stream(const bf16_t* x, const bf16_t* w, const float* bias, TOut* y, int m, int n, int k,
                          Epilogue epilogue, int nw, int slices, hipStream_t s) {
    const int k_per = ((k + slices - 1) / slices + ST_BK - 1) / ST_BK * ST_BK;
    dim3 grid((unsigned)((n + nw * 16 - 1) / (nw * 16)), (unsigned)((k + k_per - 1) / k_per));
    if (nw == 8)
        k_gemm_bf16_stream<TOut, MT, 8><<<grid, 8 * 64, 0, s>>>(x, w, bias, y, m, n, k, k_per, epilogue);
    else if (nw == 4)
        k_gemm_bf16_stream<TOut, MT, 4><<<grid, 4 * 64, 0, s>>>(x, w, bias, y, m, n, k, k_per, epilogue);
    else
        k_gemm_bf16_stream<TOut, MT, 2><<<grid, 2 * 64, 0, s>>>(x, w, bias, y, m, n, k, k_per, epilogue);
}

// With a K that the kernel with loads straight into LDS does not take: the 256x256 tile with register
// staging (one block per CU) pays once its tiles keep most of the chip's 256 CUs busy: measured, from
// about 160 tiles on (192 tiles: +15% over 128x128; 96 tiles: -30%).
static bool big_tile_pays(int m, int n, int k) {
    (void)k;
    return (long long)((m + 255) / 256) * ((n + 255) / 256) >= 160;
}

template <typename TOut>
static int launch_bf16(const bf16_t* x, const bf16_t* w, const float* bias, TOut* y, int m, int n, int k, Epilogue epilogue,
                       int force, int slices, hipStream_t s) {
    // `force` (for measurements): 2/4/8 = shared activations with that many waves
    // 452: the 128 by 128 tile on four stages, at any number of rows
    if (force == 452 && k % slices == 0 && (k / slices) % (4 * DM_BK) == 0 && dma_tile_takes(m, n, k))
        return launch_dma<TOut>(x, w, bias, y, m, n, k, epilogue, 128, 2, slices, s, 4);
    if (m <= ROWS_MAX && force == 0)
        return imparo_few_rows(x, w, bias, y, std::is_same<TOut, float>::value ? IMPARO_F32 : IMPARO_BF16, m, n, k, epilogue, slices,
                               nullptr, 0, 0.f, s);
    // Up to 64 rows the kernel of some_rows.hip, and up to 128 where it takes few weight rows a block: with 64 the tile of 128 by
    // 64 draws the same bytes a CU with less to do about them (128 rows of 16,384 by 2,048 gated 20.0 us, 20.8 there; 96 rows 18.9
    // and 19.3, 65 rows 17.5 and 18.9; 79 rows of 60,418 by 128 8.6 and 21.5, 93 of 49,664 by 1,024 gated 26.8 and 39.1). But that
    // tile's four stages take K-steps in fours: where K does not come in fours, up to 96 rows and in one round of the CUs this kernel is the
    // faster one again (72 rows of 12,288 by 9,344 gated 68.7 us, 125.5 on the tile; 78 of 9,090 by 3,456 27.2 and 47.1, 71 of
    // 9,216 by 640 8.9 and 11.8; in two rounds 70 of 17,920 by 2,688 40.1 and 39.2; 73 of 9,216 by 128 5.7 and 4.4).
    // 616, 632, 664: this kernel with 16, 32 and 64 weight rows a block
    if (imparo_some_rows_takes(m, n, k) && (force == 0 || force == 616 || force == 632 || force == 664)) {
        const int tile = force ? force - 600 : imparo_some_rows_tile(m, n, slices), k_slice = k / slices;
        const bool odd_steps = k_slice % (4 * DM_BK) != 0 && k_slice > 2 * DM_BK && (long long)((n + 63) / 64) * slices <= 256;
        if (force || m <= 64 || tile <= 32 || (m <= 96 && odd_steps))
            return imparo_some_rows(x, w, bias, y, std::is_same<TOut, float>::value ? IMPARO_F32 : IMPARO_BF16, m, n, k, epilogue,
                                    slices, tile, s);
    }
    if (m <= 64) {
        const int nw = force == 2 || force == 4 || force == 8 ? force : stream_waves(n);
        if (m <= 32)
            launch_stream<TOut, 2>(x, w, bias, y, m, n, k, epilogue, nw, slices, s);
        else
            launch_stream<TOut, 4>(x, w, bias, y, m, n, k, epilogue, nw, slices, s);
    } else {
        // by shape: the tile kernel with loads straight into LDS where it takes the K, as its plan says;
        // `force` (for measurements) 256: the 256x256 tile with register staging
        if (force == 0) {
            const DmaPlan plan = dma_plan(m, n, k, slices);
            if (plan.tn)
                return launch_dma<TOut>(x, w, bias, y, m, n, k, epilogue, plan.bm, plan.tn, slices, s, plan.stages);
        }
        if (slices == 1 && (force == 256 || (force == 0 && big_tile_pays(m, n, k))))
            return launch_big<TOut, 2, 4, 4, 2>(x, w, bias, y, m, n, k, epilogue, s);
        // 258: the tile that loads straight into LDS, 256 wide; 262, 263: 128 and 192 wide
        if ((force == 258 || force == 262 || force == 263) && k % slices == 0 && dma_tile_takes(m, n, k / slices) &&
            dma_tile_takes(m, n, k))
            return launch_dma<TOut>(x, w, bias, y, m, n, k, epilogue, 256, force == 258 ? 4 : force - 260, slices, s);
        // 558: 192 activation rows to a tile, 256 wide
        if (force == 558 && k % slices == 0 && dma_tile_takes(m, n, k / slices) && dma_tile_takes(m, n, k))
            return launch_dma<TOut>(x, w, bias, y, m, n, k, epilogue, 192, 4, slices, s);
        // 358, 352: 128 activation rows to a tile, 256 and 128 wide
        if ((force == 358 || force == 352) && k % slices == 0 && dma_tile_takes(m, n, k / slices) && dma_tile_takes(m, n, k))
            return launch_dma<TOut>(x, w, bias, y, m, n, k, epilogue, 128, force == 358 ? 4 : 2, slices, s);
        // 351, 451: 128 activation rows by 64 weight rows, on two stages and on four
        if ((force == 351 || force == 451) && k % slices == 0 && dma_tile_takes(m, n, k / slices) && dma_tile_takes(m, n, k) &&
            (force == 351 || (k / slices) % (4 * DM_BK) == 0))
            return launch_dma<TOut>(x, w, bias, y, m, n, k, epilogue, 128, 1, slices, s, force == 451 ? 4 : 2);
        const int tiles_m = (m + BG_BM - 1) / BG_BM, tiles_n = (n + BG_BN - 1) / BG_BN;
        const long long total = (long long)tiles_m * tiles_n;
        if (total > 0x7fffff00LL) return IMPARO_BAD_ARGUMENT;
        const unsigned blocks = (unsigned)(((total + N_XCD - 1) / N_XCD) * N_XCD);
        const int k_per = ((k + slices - 1) / slices + BG_BK - 1) / BG_BK * BG_BK;
        dim3 grid(blocks, (unsigned)((k + k_per - 1) / k_per));
        k_gemm_bf16_tile<TOut><<<grid, 256, 0, s>>>(x, w, bias, y, m, n, k, tiles_m, tiles_n, epilogue, k_per);
    }
    return launch_status();
}


// `variant` 0 lets the library choose the kernel. The others are for measurements and tests only, so
// that each kernel can be met at any shape: 2, 4 or 8 the shared-activation kernel with that many waves (up to 64 rows), 256 the 256x256 tile with register staging, 258 / 263 / 262 the tile
// with loads straight into LDS at 256 rows by 256 / 192 / 128, 358 / 352 the same at 128 rows by
// 256 / 128, 558 at 192 rows by 256, 616 / 632 / 664 the kernel of 17 to 128 rows with 16 / 32 / 64 weight rows a block, 452 the 128 by 128 tile on four stages, 351 / 451 the 128 by 64 tile on two / four stages;
// with a variant, any number of K slices is taken.
static int gemm_variant(const void* x, const void* w, const float* bias, void* y, int dtype, int out_dtype,
                        int m, int n, int k, Epilogue epilogue, int slices, int variant, imparo_stream stream) {
    if (!x || !w || !y || m < 0 || n <= 0 || k <= 0) return IMPARO_BAD_ARGUMENT;
    if (slices < 1 || variant == 1) return IMPARO_BAD_ARGUMENT;      // (1: a kernel that is no more)
    // slices: only what imparo_gemm_slices allows, float32 out, no epilogue that is not linear
    const int slices_ok = imparo_gemm_slices(m, n, k, dtype);
    if (slices > 1 && ((slices != slices_ok && variant == 0) || out_dtype != IMPARO_F32 || epilogue != EPI_NONE))
        return IMPARO_BAD_ARGUMENT;
    if (epilogue != EPI_NONE && epilogue != EPI_SWIGLU && epilogue != EPI_ADD) return IMPARO_BAD_ARGUMENT;
    if (epilogue == EPI_SWIGLU && (n % 2 != 0)) return IMPARO_BAD_ARGUMENT;
    // adding into Y: the tile kernel that loads straight into LDS only, chosen by the library, K in one piece
    if (epilogue == EPI_ADD && (variant != 0 || slices != 1 || out_dtype != IMPARO_F32 || !imparo_gemm_adds(m, n, k, dtype)))
        return IMPARO_BAD_ARGUMENT;
    if (m == 0) return IMPARO_OK;
    hipStream_t s = (hipStream_t)stream;
    if (dtype == IMPARO_F32) {
        if (out_dtype == IMPARO_F32)
            return launch_f32<float>((const float*)x, (const float*)w, bias, (float*)y, m, n, k, epilogue, s);
        if (out_dtype == IMPARO_BF16)
            return launch_f32<bf16_t>((const float*)x, (const float*)w, bias, (bf16_t*)y, m, n, k, epilogue, s);
        return IMPARO_BAD_ARGUMENT;
    }
    if (dtype != IMPARO_BF16) return IMPARO_BAD_ARGUMENT;
    // 16-byte loads along K: rows must start 16-byte aligned
    if (k % 8 != 0 || ((uintptr_t)x & 15) || ((uintptr_t)w & 15)) return IMPARO_BAD_ARGUMENT;
    if (out_dtype == IMPARO_F32)
        return launch_bf16<float>((const bf16_t*)x, (const bf16_t*)w, bias, (float*)y, m, n, k, epilogue,
                                  variant, slices, s);
    if (out_dtype == IMPARO_BF16)
        return launch_bf16<bf16_t>((const bf16_t*)x, (const bf16_t*)w, bias, (bf16_t*)y, m, n, k, epilogue,
                                   variant, slices, s);
    return IMPARO_BAD_ARGUMENT;
}

extern "C" int imparo_gemm(const void* x, const void* w, const float* bias, void* y, int dtype, int out_dtype,
                           int m, int n, int k, int epilogue, int slices, imparo_stream stream) {
    return gemm_variant(x, w, bias, y, dtype, out_dtype, m, n, k, epilogue, slices, 0, stream);
}

extern "C" int imparo_gemm_gated(const void* x, const void* w, const float* bias, void* y, int dtype, int out_dtype,
                                 int m, int n, int k, float scale, float limit, float alpha, imparo_stream stream) {
    if (!(limit >= 0.f) || alpha != alpha) return IMPARO_BAD_ARGUMENT;
    return gemm_variant(x, w, bias, y, dtype, out_dtype, m, n, k, Epilogue(EPI_SWIGLU, scale, limit, limit > 0.f ? alpha : 1.0f), 1,
                        0, stream);
}

extern "C" int imparo_gemm_variant(const void* x, const void* w, const float* bias, void* y, int dtype, int out_dtype,
                                   int m, int n, int k, int epilogue, int slices, int variant, imparo_stream stream) {
    return gemm_variant(x, w, bias, y, dtype, out_dtype, m, n, k, epilogue, slices, variant, stream);
}

// Asks the runtime about one kernel of this file, which makes it load the file's code onto the
// current device (it loads a file's kernels when one of them is first used; a stream under capture
// cannot do that).
int imparo_load_code_gemm() {
    hipFuncAttributes attributes;
    return hipFuncGetAttributes(&attributes, reinterpret_cast<const void*>(&k_gemm_f32_rows<float>)) == hipSuccess ? IMPARO_OK
                                                                                              : IMPARO_LAUNCH_FAILED;
}
