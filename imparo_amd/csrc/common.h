// Shared device helpers for the gfx950 kernels: storage types, bf16
// conversion, wave64 reductions, and the error codes the C entry points return.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#define IMPARO_OK 0
#define IMPARO_BAD_ARGUMENT 1
#define IMPARO_LAUNCH_FAILED 2
#define IMPARO_SCRATCH_TOO_SMALL 3

// dtype codes shared with the Python side
#define IMPARO_F32 0
#define IMPARO_BF16 1

#define WAVE 64

typedef uint16_t bf16_t;   // raw bfloat16 bits

__device__ __forceinline__ float bf16_to_f32(bf16_t v) {
    return __uint_as_float(((uint32_t)v) << 16);
}

// round to nearest even; NaN stays NaN (gfx950 converts in hardware, two values per instruction)
__device__ __forceinline__ bf16_t f32_to_bf16(float f) {
    const __bf16 b = (__bf16)f;
    return *reinterpret_cast<const bf16_t*>(&b);
}

// two values in one register, `lo` in the low half
__device__ __forceinline__ uint32_t f32x2_to_bf16x2(float lo, float hi) {
    typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
    const bf16x2_t b = {(__bf16)lo, (__bf16)hi};
    return *reinterpret_cast<const uint32_t*>(&b);
}

template <typename T> __device__ __forceinline__ float load_f32(const T* p, size_t i);
template <> __device__ __forceinline__ float load_f32<float>(const float* p, size_t i) { return p[i]; }
template <> __device__ __forceinline__ float load_f32<bf16_t>(const bf16_t* p, size_t i) { return bf16_to_f32(p[i]); }

template <typename T> __device__ __forceinline__ void store_f32(T* p, size_t i, float v);
template <> __device__ __forceinline__ void store_f32<float>(float* p, size_t i, float v) { p[i] = v; }
template <> __device__ __forceinline__ void store_f32<bf16_t>(bf16_t* p, size_t i, float v) { p[i] = f32_to_bf16(v); }

// Sums and maxima over a wave, the same in every lane: lanes 32 apart first, then 16, 8, 4, 2, 1. On lane swaps and
// moves inside rows of 16, which take a few cycles where a shuffle through LDS takes about a hundred: after a step all
// lanes that far apart agree, so "rotated by n" stands for "n apart" (and a sum of two is the same either way round).
// All 64 lanes must be active: no call where lanes have left or taken another branch.
#define WAVE_STEPS(v, OP)                                                                                              \
    do {                                                                                                               \
        auto halves = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);          \
        v = OP(__uint_as_float(halves[0]), __uint_as_float(halves[1]));                                                \
        halves = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);               \
        v = OP(__uint_as_float(halves[0]), __uint_as_float(halves[1]));                                                \
        v = OP(v, rotated_in_row<8>(v));                                                                               \
        v = OP(v, rotated_in_row<4>(v));                                                                               \
        v = OP(v, rotated_in_row<2>(v));                                                                               \
        v = OP(v, rotated_in_row<1>(v));                                                                               \
    } while (0)

template <int N>
__device__ __forceinline__ float rotated_in_row(float v) {
    return __uint_as_float(__builtin_amdgcn_update_dpp(0, __float_as_uint(v), 0x120 + N, 0xf, 0xf, false));   // row_ror:N
}
__device__ __forceinline__ float plain_sum(float a, float b) { return a + b; }

__device__ __forceinline__ float wave_sum(float v) {
    WAVE_STEPS(v, plain_sum);
    return v;
}

__device__ __forceinline__ float wave_max(float v) {
    WAVE_STEPS(v, fmaxf);
    return v;
}

// What the lane N apart (lane ^ N) holds, on moves inside rows of 16 and lane swaps: a few cycles each, where a shuffle is a trip
// through LDS. Both lanes must be active (for 16 and 32 the whole wave).
template <int N>
__device__ __forceinline__ uint32_t lane_xor_bits(uint32_t v) {
    static_assert(N == 1 || N == 2 || N == 4 || N == 8 || N == 16 || N == 32, "a power of two inside a wave");
    if constexpr (N == 1) return __builtin_amdgcn_update_dpp(0, v, 0xB1, 0xf, 0xf, false);           // quad_perm:[1,0,3,2]
    if constexpr (N == 2) return __builtin_amdgcn_update_dpp(0, v, 0x4E, 0xf, 0xf, false);           // quad_perm:[2,3,0,1]
    if constexpr (N == 4) {                                                                          // row_shl:4 into quads 0 and 2,
        const uint32_t up = __builtin_amdgcn_update_dpp(v, v, 0x104, 0xf, 0x5, false);               // row_shr:4 into quads 1 and 3
        return __builtin_amdgcn_update_dpp(up, v, 0x114, 0xf, 0xA, false);
    }
    if constexpr (N == 8) return __builtin_amdgcn_update_dpp(0, v, 0x128, 0xf, 0xf, false);          // row_ror:8
    if constexpr (N == 16) {
        const auto r = __builtin_amdgcn_permlane16_swap(v, v, false, false);
        return threadIdx.x & 16 ? r[0] : r[1];
    }
    const auto r = __builtin_amdgcn_permlane32_swap(v, v, false, false);
    return threadIdx.x & 32 ? r[0] : r[1];
}
template <int N> __device__ __forceinline__ float lane_xor(float v) { return __uint_as_float(lane_xor_bits<N>(__float_as_uint(v))); }
template <int N> __device__ __forceinline__ int lane_xor(int v) { return (int)lane_xor_bits<N>((uint32_t)v); }

// Sums and maxima over the lanes 16 and then 32 apart (all 64 lanes active); a sum of two is the same either way round
__device__ __forceinline__ float sum_16_32(float v) {
    auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    v = __uint_as_float(r[0]) + __uint_as_float(r[1]);
    r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}
__device__ __forceinline__ float sum_32_16(float v) {      // (32 and then 16 apart)
    auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    v = __uint_as_float(r[0]) + __uint_as_float(r[1]);
    r = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}
__device__ __forceinline__ float max_16_32(float v) {
    auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    v = fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
    r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
// The sum over LANES neighbouring lanes (a power of two), the nearest first (1, 2, 4, ... apart): after a step all lanes that near
// agree, so a mirrored quad or half row stands for the one 4 or 8 apart
template <int LANES>
__device__ __forceinline__ float sum_near_first(float v) {
    if constexpr (LANES > 1) v += lane_xor<1>(v);
    if constexpr (LANES > 2) v += lane_xor<2>(v);
    if constexpr (LANES > 4) v += __uint_as_float(__builtin_amdgcn_update_dpp(0, __float_as_uint(v), 0x141, 0xf, 0xf, false));   // row_half_mirror
    if constexpr (LANES > 8) v += __uint_as_float(__builtin_amdgcn_update_dpp(0, __float_as_uint(v), 0x140, 0xf, 0xf, false));   // row_mirror
    if constexpr (LANES > 16) v += lane_xor<16>(v);
    if constexpr (LANES > 32) v += lane_xor<32>(v);
    return v;
}

// Sum over a block of up to 1024 threads in whole waves; every thread gets the result.
// `scratch` holds at least 16 floats of LDS. The order of the additions
// depends only on the block size, never on the data.
__device__ __forceinline__ float block_sum(float v, float* scratch) {
    v = wave_sum(v);
    const int lane = threadIdx.x & (WAVE - 1);
    const int wave = threadIdx.x / WAVE;
    const int n_waves = (blockDim.x + WAVE - 1) / WAVE;
    __syncthreads();
    if (lane == 0) scratch[wave] = v;
    __syncthreads();
    float total = 0.f;
    for (int i = 0; i < n_waves; ++i) total += scratch[i];
    return total;
}

// ---- what every kernel that norms and rotates a head shares, so that all of them round alike
// The angle is position * inv_freq, the product taken in float64 and rounded to float32; its sine and
// cosine to float32 accuracy. Angles reach 1e5 and more, where a float32 library routine reduces the
// argument with a long integer product (thousands of cycles in which a whole block waits for its table,
// and the routine's code for that case weighs on the small angles too). So everything is done here, in
// float64: the multiple of pi/2 comes off (two constants carry pi/2 to 107 bits; the product with a count
// below 2^17 is exact enough by far), and what is left, at most pi/4, goes into the two power series, cut
// where the next term is below 2e-9 (sine, after x^9) and 2e-10 (cosine, after x^10).
__device__ __forceinline__ void rotation_of(int pos, float inv_freq, float& sn, float& cs) {
    const float theta = (float)((double)pos * (double)inv_freq);
    const double t = (double)theta;
    const double k = rint(t * 0.63661977236758134308);
    double r = fma(-k, 1.57079632679489655800, t);
    r = fma(-k, 6.12323399573676603587e-17, r);
    const double z = r * r;
    double s = fma(z, 1.0 / 362880.0, -1.0 / 5040.0);
    s = fma(z, s, 1.0 / 120.0);
    s = fma(z, s, -1.0 / 6.0);
    s = fma(z * r, s, r);
    double c = fma(z, -1.0 / 3628800.0, 1.0 / 40320.0);
    c = fma(z, c, -1.0 / 720.0);
    c = fma(z, c, 1.0 / 24.0);
    c = fma(z, c, -0.5);
    c = fma(z, c, 1.0);
    const int quarter = (int)((long long)k & 3);
    const float sf = (float)s, cf = (float)c;
    sn = (quarter & 1) ? cf : sf;
    cs = (quarter & 1) ? sf : cf;
    if (quarter == 1 || quarter == 2) cs = -cs;
    if (quarter >= 2) sn = -sn;
}
// The first position a query at `pos` sees. window > 0: the last `window` positions up to its own; window < 0:
// the positions of its own chunk, chunks of -window positions counted from position 0; 0: every position
// before it. Never decreases with pos, which is all the attention kernels ask of it.
__device__ __forceinline__ int first_seen(int pos, int window) {
    return window > 0 ? max(0, pos + 1 - window) : window < 0 ? pos - pos % (-window) : 0;
}
__device__ __forceinline__ float head_norm_scale(float sum_squares, int head_dim, float eps) {
    return 1.0f / sqrtf(sum_squares / (float)head_dim + eps);
}

// 16 bytes a lane from memory straight into LDS, lane after lane from `dst_wave_uniform` on
__device__ __forceinline__ void load_to_lds(const bf16_t* src, bf16_t* dst_wave_uniform) {
    __builtin_amdgcn_global_load_lds((const void __attribute__((address_space(1)))*)src,
                                     (void __attribute__((address_space(3)))*)dst_wave_uniform, 16, 0, 0);
}

// The same load written out, for kernels that keep the loads of several K-steps in flight. The compiler
// answers a fragment read from LDS that follows any load into LDS it knows of with a wait for every load
// (it counts such a load as one that may come back out of order), which empties the pipeline; a load it
// does not know of it does not wait for, and the kernel waits itself, by count. `lds_byte` is the same
// for the whole wave.
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
__device__ __forceinline__ void load_to_lds_uncounted(const bf16_t* src, unsigned lds_byte) {
    asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off"
                 :
                 : "v"(src), "s"(lds_byte)
                 : "memory", "m0");
}
// The same from a uniform base and a byte offset a lane
__device__ __forceinline__ void load_to_lds_uncounted(const float* base, unsigned byte_offset, unsigned lds_byte) {
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1"
                 :
                 : "v"(byte_offset), "s"(base), "s"(lds_byte)
                 : "memory", "m0");
}
#pragma clang diagnostic pop

// Orders LDS traffic between the lanes of one wave: what any lane wrote before
// is visible to every lane after.
__device__ __forceinline__ void wave_lds_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// One per file of kernels: loads that file's code onto the current device (imparo_load_code calls them all).
int imparo_load_code_attention();
int imparo_load_code_attention_mfma();
int imparo_load_code_decay_scan();
int imparo_load_code_decode_rows();
int imparo_load_code_diff_attention();
int imparo_load_code_elementwise();
int imparo_load_code_gated_ops();
int imparo_load_code_gemm();
int imparo_load_code_hgrn2();
int imparo_load_code_latent_attention();
int imparo_load_code_moe();
int imparo_load_code_rope_cache();
int imparo_load_code_row_ops();
int imparo_load_code_sampling();
int imparo_load_code_selective_scan();
int imparo_load_code_some_rows();
int imparo_load_code_streams();

static inline int launch_status() {
    return hipGetLastError() == hipSuccess ? IMPARO_OK : IMPARO_LAUNCH_FAILED;
}
