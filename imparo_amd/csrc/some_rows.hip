// Products of 17 to 128 rows, bfloat16: Y[m, n] = X[m, k] . W[n, k]^T with float32 accumulation, K a multiple of 128.
//
// What bounds them is a CU's way to memory: a block draws its weight rows once, cold, and every activation row beside them,
// and a CU takes in about 40 to 60 GB/s of the two together, whatever waits behind it. So a block has the weight rows
// that make weights plus activations a CU fewest (64, 32 or 16), and the two ways are kept apart, so that neither waits for the other:
//   - weights go from memory into the operand registers of the four (or eight) waves that multiply, four chunks of 128 k ahead;
//     a wave has a quarter of each chunk's k and 16 or 32 weight rows;
//   - activations go straight into a ring of four chunks in LDS, brought by one or two waves that do nothing else. Loads are
//     counted in the order they were sent: a wave that sent both would wait for its far weights with every near activation.
// One bare barrier a chunk hands a chunk over and its place back. The quarters of K meet in LDS at the end, in one order
// whatever the shape, and rows leave in whole vectors.
// Measured with cold weights, 64 rows (the kernel that staged activations through registers, now for other K only): 16,384 by
// 2,048 gated 17.4 us (19.1), 6,144 by 2,048 10.2 (12.7), 3,072 by 2,048 8.0 (12.1), 2,048 by 2,048 in four slices 4.7 (6.5), 2,048
// by 8,192 in four 11.3 (13.5), 9,216 by 1,024 gated 9.3 (13.2).
#include "common.h"
#include "api.h"
#include "rows.h"

#include <type_traits>

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

#define SR_BK 128        // k of a chunk: 32 of each of the four quarters
#define SR_STAGES 4      // chunks of activations in LDS
#define SR_AHEAD 4       // chunks of weights in registers

union SomeFrag {
    uint4 u;
    bf16x8 v;
};

// MT: tiles of 16 activation rows; RT: of 16 weight rows a wave; NN: groups of four waves, each group with its own weight rows
template <typename TOut, int MT, int RT, int NN>
struct SomeRows {
    static constexpr int LOADERS = MT > 4 ? 2 : 1, COMPUTE = NN * 4, THREADS = (COMPUTE + LOADERS) * 64;
    static constexpr int BM = MT * 16, BN = NN * RT * 16;
    static constexpr int PER = BM / 4 / LOADERS;             // load instructions a loader and chunk, four rows each
    static constexpr int STAGE = BM * SR_BK;
    static constexpr int LD = BN + 4;                        // floats from row to row where the quarters meet
    static constexpr int RING_BYTES = SR_STAGES * STAGE * 2, PART_BYTES = 4 * BM * LD * 4;
    static constexpr int LDS = RING_BYTES > PART_BYTES ? RING_BYTES : PART_BYTES;
    static_assert((SR_STAGES - 1) * PER <= 63 && LDS <= 160 * 1024, "loads a wave can count, and LDS");
};

template <typename TOut, int MT, int RT, int NN>
__global__ __launch_bounds__((SomeRows<TOut, MT, RT, NN>::THREADS)) void k_some_rows(
    const bf16_t* __restrict__ X, const bf16_t* __restrict__ W, const float* __restrict__ bias, TOut* __restrict__ Y, int M, int N,
    int K_all, int k_per, int slices, Epilogue epilogue) {
    using S = SomeRows<TOut, MT, RT, NN>;
    extern __shared__ __attribute__((aligned(1024))) bf16_t ring[];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    // the slices of a tile are neighbours: with 2, 4 or 8 of them an XCD meets the activations of one slice or few
    const int slice = blockIdx.x % slices, tile = blockIdx.x / slices, n0 = tile * S::BN;
    const int k_lo = slice * k_per, nc = (min(K_all, k_lo + k_per) - k_lo) / SR_BK;
    // blocks start their walk at different chunks: rows are a power of two apart, so blocks in step would ask the same few
    // channels of a cache for the same chunk
    const int rot = tile % nc;
    auto chunk_at = [&](int c) __attribute__((always_inline)) { return (c + rot >= nc ? c + rot - nc : c + rot) * SR_BK; };
    X += k_lo;
    W += (size_t)n0 * K_all + k_lo;
    const int r16 = lane & 15, g = lane >> 4;
    f32x4 acc[RT][MT];
    if (wave >= S::COMPUTE) {
        const int first = (wave - S::COMPUTE) * S::PER;
        const unsigned lds = (unsigned)(size_t)(__attribute__((address_space(3))) bf16_t*)ring + first * 1024;
        // lane -> row lane / 16 of an instruction's four, place lane % 16, where the row's piece place ^ (row % 16) of 8 k lies: the
        // 16 rows that are read together fall on distinct banks
        unsigned off[S::PER];
#pragma unroll
        for (int j = 0; j < S::PER; ++j) {
            const int row = (first + j) * 4 + (lane >> 4);
            off[j] = ((unsigned)min(row, M - 1) * (unsigned)K_all + (((lane & 15) ^ (row & 15)) << 3)) * 2u;
        }
        auto load = [&](int stage, int c) __attribute__((always_inline)) {
            const float* base = reinterpret_cast<const float*>(X + chunk_at(c));
#pragma unroll
            for (int j = 0; j < S::PER; ++j)
                load_to_lds_uncounted(base, off[j], __builtin_amdgcn_readfirstlane(lds + stage * S::STAGE * 2 + j * 1024));
        };
        for (int c = 0; c < min(SR_STAGES - 1, nc); ++c) load(c, c);
        int stage = 0;
        for (int c = 0; c < nc; ++c) {
            static_assert(SR_STAGES == 4, "the chunks that may be on their way beyond c: two, one or none");
            if (c + 2 < nc)
                asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 * S::PER) : "memory");
            else if (c + 1 < nc)
                asm volatile("s_waitcnt vmcnt(%0)" ::"n"(S::PER) : "memory");
            else
                asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            __builtin_amdgcn_s_barrier();                    // chunk c is there, chunk c - 1 is read
            if (c + SR_STAGES - 1 < nc) load((stage + SR_STAGES - 1) % SR_STAGES, c + SR_STAGES - 1);
            stage = (stage + 1) % SR_STAGES;
        }
    } else {
        const int quarter = wave & 3, group = wave >> 2;
#pragma unroll
        for (int r = 0; r < RT; ++r)
#pragma unroll
            for (int mt = 0; mt < MT; ++mt) acc[r][mt] = f32x4{0.f, 0.f, 0.f, 0.f};
        unsigned off[RT];
#pragma unroll
        for (int r = 0; r < RT; ++r)
            off[r] = ((unsigned)min((group * RT + r) * 16 + r16, N - 1 - n0) * (unsigned)K_all + quarter * 32 + g * 8) * 2u;
        SomeFrag w[SR_AHEAD][RT];
        auto fetch = [&](int c, SomeFrag (&f)[RT]) __attribute__((always_inline)) {
            const char* base = reinterpret_cast<const char*>(W + chunk_at(min(c, nc - 1)));      // (past the end: the last chunk again)
#pragma unroll
            for (int r = 0; r < RT; ++r) f[r].u = *reinterpret_cast<const uint4*>(base + off[r]);
            __builtin_amdgcn_sched_barrier(0);               // (loads stay in the order they are used and where they are written)
        };
#pragma unroll
        for (int i = 0; i < SR_AHEAD; ++i) fetch(i, w[i]);
        const bf16_t* xs = ring + r16 * SR_BK + (((quarter * 4 + g) ^ r16) << 3);
        int stage = 0;
        auto use = [&](const SomeFrag (&f)[RT]) __attribute__((always_inline)) {
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");       // the chunk before is read
            __builtin_amdgcn_s_barrier();
            asm volatile("" ::: "memory");
            SomeFrag x[MT];
#pragma unroll
            for (int mt = 0; mt < MT; ++mt) x[mt].u = *reinterpret_cast<const uint4*>(xs + stage * S::STAGE + mt * 16 * SR_BK);
#pragma unroll
            for (int mt = 0; mt < MT; ++mt)
#pragma unroll
                for (int r = 0; r < RT; ++r)
                    acc[r][mt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(f[r].v, x[mt].v, acc[r][mt], 0, 0, 0);
            stage = (stage + 1) % SR_STAGES;
        };
        int c = 0;
        for (; c + SR_AHEAD < nc; c += SR_AHEAD) {
#pragma unroll
            for (int i = 0; i < SR_AHEAD; ++i) {
                use(w[i]);
                fetch(c + SR_AHEAD + i, w[i]);
            }
        }
#pragma unroll
        for (int i = 0; i < SR_AHEAD; ++i) {
            if (c + i < nc) use(w[i]);
            __builtin_amdgcn_sched_barrier(0);
        }
    }
    __syncthreads();                                         // the ring is read, and nothing is on its way into it
    float* part = reinterpret_cast<float*>(ring);
    if (wave < S::COMPUTE) {
        // a lane holds activation row r16 of each tile and four neighbouring weight rows
        const int quarter = wave & 3, group = wave >> 2;
#pragma unroll
        for (int r = 0; r < RT; ++r)
#pragma unroll
            for (int mt = 0; mt < MT; ++mt)
                *reinterpret_cast<f32x4*>(&part[(quarter * S::BM + mt * 16 + r16) * S::LD + (group * RT + r) * 16 + g * 4]) = acc[r][mt];
    }
    __syncthreads();
    Y += (size_t)slice * M * N;
    const bool biased = bias && slice == 0, swiglu = epilogue == EPI_SWIGLU, adds = epilogue == EPI_ADD;   // (adds: float32 out)
    const int out_n = swiglu ? N / 2 : N;
    constexpr int LANES = S::BN / 4;                         // of a row
    for (int q = tid; q < S::BM * LANES; q += S::THREADS) {
        const int m = q / LANES, col = (q % LANES) * 4, n = n0 + col;
        if (m >= M || n >= N) continue;
        f32x4 p[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) p[i] = *reinterpret_cast<const f32x4*>(&part[(i * S::BM + m) * S::LD + col]);
        float v[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) v[i] = ((p[0][i] + p[1][i]) + (p[2][i] + p[3][i])) + (biased && n + i < N ? bias[n + i] : 0.f);
        TOut* dst = Y + (size_t)m * out_n + (swiglu ? n / 2 : n);
        if (swiglu) {
            const float a = gated_mul_fast(epilogue, v[0], v[1]), b = gated_mul_fast(epilogue, v[2], v[3]);
            if (n + 4 <= N && !((uintptr_t)dst % (2 * sizeof(TOut)))) {
                if constexpr (std::is_same<TOut, float>::value)
                    *reinterpret_cast<float2*>(dst) = make_float2(a, b);
                else
                    *reinterpret_cast<uint32_t*>(dst) = f32x2_to_bf16x2(a, b);
            } else {
                store_f32<TOut>(dst, 0, a);                  // (N is even, so n + 1 is inside)
                if (n + 3 < N) store_f32<TOut>(dst, 1, b);
            }
        } else if (n + 4 <= N && (std::is_same<TOut, float>::value || !((uintptr_t)dst % 8))) {
            if constexpr (std::is_same<TOut, float>::value) {
                f32x4_any o = {v[0], v[1], v[2], v[3]};
                if (adds) o = *reinterpret_cast<const f32x4_any*>(dst) + o;
                *reinterpret_cast<f32x4_any*>(dst) = o;
            } else {
                *reinterpret_cast<uint2*>(dst) = make_uint2(f32x2_to_bf16x2(v[0], v[1]), f32x2_to_bf16x2(v[2], v[3]));
            }
        } else {
#pragma unroll
            for (int i = 0; i < 4; ++i)
                if (n + i < N) store_f32<TOut>(dst, i, adds ? load_f32<TOut>(dst, i) + v[i] : v[i]);
        }
    }
}

template <typename TOut, int MT, int RT, int NN>
static int launch_some(const bf16_t* x, const bf16_t* w, const float* bias, TOut* y, int m, int n, int k, const Epilogue& epilogue,
                       int slices, hipStream_t s) {
    using S = SomeRows<TOut, MT, RT, NN>;
    static bool configured = false;
    if (!configured) {
        if (hipFuncSetAttribute((const void*)k_some_rows<TOut, MT, RT, NN>, hipFuncAttributeMaxDynamicSharedMemorySize, S::LDS) !=
            hipSuccess)
            return IMPARO_LAUNCH_FAILED;
        configured = true;
    }
    const int k_per = ((k + slices - 1) / slices + SR_BK - 1) / SR_BK * SR_BK;
    slices = (k + k_per - 1) / k_per;
    const long long blocks = ((long long)n + S::BN - 1) / S::BN * slices;
    if (blocks * S::THREADS >= (1LL << 32)) return IMPARO_BAD_ARGUMENT;
    k_some_rows<TOut, MT, RT, NN><<<(unsigned)blocks, S::THREADS, S::LDS, s>>>(x, w, bias, y, m, n, k, k_per, slices, epilogue);
    return launch_status();
}

template <typename TOut>
static int launch_some_rows(const bf16_t* x, const bf16_t* w, const float* bias, TOut* y, int m, int n, int k, const Epilogue& epilogue,
                            int slices, int bn, hipStream_t s) {
#define SOME_ROWS(MT)                                                                                   \
    if (m <= MT * 16) {                                                                                 \
        if (bn == 64) return launch_some<TOut, MT, 2, 2>(x, w, bias, y, m, n, k, epilogue, slices, s);  \
        if (bn == 32) return launch_some<TOut, MT, 1, 2>(x, w, bias, y, m, n, k, epilogue, slices, s);  \
        return launch_some<TOut, MT, 1, 1>(x, w, bias, y, m, n, k, epilogue, slices, s);                \
    }
    SOME_ROWS(2)
    SOME_ROWS(3)
    SOME_ROWS(4)
    SOME_ROWS(6)
    SOME_ROWS(8)
#undef SOME_ROWS
    return IMPARO_BAD_ARGUMENT;
}

bool imparo_some_rows_takes(int m, int n, int k) {
    // offsets inside a block's weight rows and the activation rows are kept in 32 bits, bytes; a launch holds fewer than
    // 2^32 threads
    return m > 16 && m <= SOME_ROWS_MAX && k % SR_BK == 0 && k < (1 << 23) && n < (1 << 25);
}

// What the fullest CU draws, weights and activations: the fewest weight rows a block whose blocks are still one round of the CUs, else 64
// (but for a few shapes of more than 64 rows in three or six slices, where 32 take no more rounds than 64 do).
int imparo_some_rows_tile(int m, int n, int slices) {
    const int rows = (m <= 64 ? (m + 15) / 16 : (m + 31) / 32 * 2) * 16;
    int best = 0;
    long long best_cost = 0;
    for (int bn = 64; bn >= 16; bn /= 2) {
        const long long blocks = ((long long)n + bn - 1) / bn * slices, cost = (blocks + 255) / 256 * (bn + rows);
        if (!best || cost < best_cost) best = bn, best_cost = cost;
    }
    return best;
}

int imparo_some_rows(const bf16_t* x, const bf16_t* w, const float* bias, void* y, int out_dtype, int m, int n, int k,
                     const Epilogue& epilogue, int slices, int tile, hipStream_t s) {
    if (out_dtype == IMPARO_F32) return launch_some_rows<float>(x, w, bias, (float*)y, m, n, k, epilogue, slices, tile, s);
    return launch_some_rows<bf16_t>(x, w, bias, (bf16_t*)y, m, n, k, epilogue, slices, tile, s);
}

int imparo_load_code_some_rows() {
    hipFuncAttributes attributes;
    return hipFuncGetAttributes(&attributes, reinterpret_cast<const void*>(&k_some_rows<float, 2, 1, 1>)) == hipSuccess
               ? IMPARO_OK
               : IMPARO_LAUNCH_FAILED;
}
