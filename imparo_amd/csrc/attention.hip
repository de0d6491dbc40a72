// Causal grouped-query attention over the paged cache.
//
// k_attention_wave: one wave per (token, head). Keys are walked in chunks of 64
// aligned at absolute multiples of 64, one key per lane for the scores, one
// output dimension per lane for the weighted sum, online softmax in float32.
// The order of every sum depends only on the query's position, so the result
// does not depend on how a prompt was cut or what else is in the batch.
#include <type_traits>
#include "common.h"
#include "api.h"

#define ATT_MAX_HEAD_DIM 576
#define ATT_WAVES 4

template <typename T> struct Vec16;
template <> struct Vec16<float> { static constexpr int N = 4; };
template <> struct Vec16<bf16_t> { static constexpr int N = 8; };

template <typename T>
__device__ __forceinline__ float dot_row(const float* __restrict__ q, const T* __restrict__ k, int head_dim);

template <>
__device__ __forceinline__ float dot_row<float>(const float* __restrict__ q, const float* __restrict__ k, int head_dim) {
    float s = 0.f;
    for (int i = 0; i < head_dim; i += 4) {
        const float4 kv = *reinterpret_cast<const float4*>(k + i);
        s += q[i] * kv.x;
        s += q[i + 1] * kv.y;
        s += q[i + 2] * kv.z;
        s += q[i + 3] * kv.w;
    }
    return s;
}

template <>
__device__ __forceinline__ float dot_row<bf16_t>(const float* __restrict__ q, const bf16_t* __restrict__ k, int head_dim) {
    float s = 0.f;
    for (int i = 0; i < head_dim; i += 8) {
        const uint4 kv = *reinterpret_cast<const uint4*>(k + i);
        const uint32_t w[4] = {kv.x, kv.y, kv.z, kv.w};
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            s += q[i + 2 * j] * __uint_as_float(w[j] << 16);
            s += q[i + 2 * j + 1] * __uint_as_float(w[j] & 0xffff0000u);
        }
    }
    return s;
}

// a head size that is no multiple of a 16-byte vector: element by element, in the same order
template <typename T>
__device__ __forceinline__ float dot_row_any(const float* __restrict__ q, const T* __restrict__ k, int head_dim) {
    float s = 0.f;
    for (int i = 0; i < head_dim; ++i) s += q[i] * load_f32<T>(k, i);
    return s;
}

template <typename T>
__global__ void k_attention_wave(const T* __restrict__ q, const T* __restrict__ k_cache, const T* __restrict__ v_cache,
                                 T* __restrict__ out, const int32_t* __restrict__ positions,
                                 const int32_t* __restrict__ row_of_token, const int32_t* __restrict__ block_table,
                                 int table_stride, int page_size, int n_tokens, int heads, int kv_heads, int head_dim,
                                 int value_dim, int out_ld, int n_pages, float scale, int window, int v_transposed,
                                 int v_ld, const ImparoAttentionRule rule) {
    __shared__ float q_rows[ATT_WAVES][ATT_MAX_HEAD_DIM];
    __shared__ float probs[ATT_WAVES][WAVE];
    __shared__ long long v_off[ATT_WAVES][WAVE];
    const int lane = threadIdx.x & (WAVE - 1);
    const int wave = threadIdx.x / WAVE;
    const long long id = (long long)blockIdx.x * ATT_WAVES + wave;
    if (id >= (long long)n_tokens * heads) return;
    const int t = (int)(id / heads);
    const int h = (int)(id - (long long)t * heads);
    const int kvh = h / (heads / kv_heads);
    const int pos = positions[t];
    const int lo = first_seen(pos, window);
    const int32_t* table = block_table + (size_t)row_of_token[t] * table_stride;

    float* qr = q_rows[wave];
    const T* qsrc = q + ((size_t)t * heads + h) * head_dim;
    for (int i = lane; i < head_dim; i += WAVE) qr[i] = load_f32<T>(qsrc, i);
    wave_lds_sync();

    constexpr int DPL = ATT_MAX_HEAD_DIM / WAVE;
    float acc[DPL];
#pragma unroll
    for (int j = 0; j < DPL; ++j) acc[j] = 0.f;
    float m = -INFINITY, l = 0.f;

    // the first positions that stay visible come first, then the window: chunks between the two are skipped
    const int lo_chunk = (lo / WAVE) * WAVE;
    const int keep = rule.keep_first;
    for (int c = keep > 0 ? 0 : lo_chunk; c <= pos; c = (c + WAVE >= keep && c + WAVE < lo_chunk) ? lo_chunk : c + WAVE) {
        const int p = c + lane;
        const bool valid = p <= pos && (p >= lo || p < keep);
        float s = -INFINITY;
        long long off = -1;
        if (valid) {
            const int page = table[p / page_size];
            if (page >= 0 && page < n_pages) {
                off = (((long long)page * kv_heads + kvh) * page_size + (p % page_size)) * head_dim;
                s = (head_dim % Vec16<T>::N == 0 ? dot_row<T>(qr, k_cache + off, head_dim)
                                                 : dot_row_any<T>(qr, k_cache + off, head_dim)) * scale;
                if (rule.softcap > 0.f) s = rule.softcap * tanhf(s / rule.softcap);
                // from here on `off` is where the key's value row starts
                off = v_transposed ? ((long long)page * kv_heads + kvh) * page_size * value_dim + (p % page_size)
                                   : (((long long)page * kv_heads + kvh) * page_size + (p % page_size)) * v_ld;
            }
        }
        const float m_new = fmaxf(m, wave_max(s));
        const float pe = (off >= 0) ? expf(s - m_new) : 0.f;
        const float corr = (m == -INFINITY) ? 0.f : expf(m - m_new);
        l = l * corr + wave_sum(pe);
        m = m_new;
        probs[wave][lane] = pe;
        v_off[wave][lane] = off;
        wave_lds_sync();
        const int n_keys = min(WAVE, pos - c + 1);
#pragma unroll
        for (int j = 0; j < DPL; ++j) acc[j] *= corr;
        for (int kk = 0; kk < n_keys; ++kk) {
            const long long vo = v_off[wave][kk];
            if (vo < 0) continue;           // uniform over the wave
            const float pk = probs[wave][kk];
            const T* vrow = v_cache + vo;
#pragma unroll
            for (int j = 0; j < DPL; ++j) {
                const int d = lane + j * WAVE;
                if (d < value_dim) acc[j] += pk * load_f32<T>(vrow, v_transposed ? (size_t)d * page_size : (size_t)d);
            }
        }
        wave_lds_sync();
    }
    float inv = l > 0.f ? 1.0f / l : 0.f;
    if (rule.sink) {                        // one more term of the denominator, without a key or a value
        const float sink = rule.sink[h], top = fmaxf(m, sink);
        const float w = (m == -INFINITY) ? 0.f : expf(m - top);
        inv = w / fmaf(l, w, expf(sink - top));
    }
    inv *= rule.out_scale;
    if (rule.gate) inv *= 1.0f / (1.0f + expf(-rule.gate[(size_t)t * rule.gate_ld + h]));
    T* dst = out + (size_t)t * out_ld + (size_t)h * value_dim;
#pragma unroll
    for (int j = 0; j < DPL; ++j) {
        const int d = lane + j * WAVE;
        if (d < value_dim) store_f32<T>(dst, d, acc[j] * inv);
    }
    // a row wider than its heads (filled up for a product that walks it in steps of 8) ends in zeros
    if (h == heads - 1)
        for (int d = value_dim + lane; d < out_ld - h * value_dim; d += WAVE) store_f32<T>(dst, d, 0.f);
}

// The same walk for float32 heads of HD numbers whose values lie in rows as the keys do (every LFM2 checkpoint in
// the float32 engine): the same chunks and the same order of every sum, so the same bits. What bounds a wave is its
// chain of trips to the caches, so they are few and overlap: a lane keeps its key's row in registers, asked for a
// chunk ahead; value rows come 32 at a time (16 of 128 numbers), their places and weights from lane registers, no load under a branch.
// Measured, two decoded tokens at 340 keys, 16 heads of 64: 30 us where the general kernel takes 200; two prompts of
// 333 tokens: 120 us where it takes 270.
// ONE: the block table has room for 64 keys at most, so one chunk holds them all: nothing is asked for ahead, no row without a
// key, value rows eight at a time, a third of the registers. (Many short prompts fill the chip and are bound by what they ask
// for: 64 of 30 tokens, 16 heads of 64, 76 us in the loop, 38 here, 73 in the general kernel.)
template <int HD, bool ONE>
__global__ __launch_bounds__(ATT_WAVES * WAVE) void k_attention_wave_f32(
    const float* __restrict__ q, const float* __restrict__ k_cache, const float* __restrict__ v_cache, float* __restrict__ out,
    const int32_t* __restrict__ positions, const int32_t* __restrict__ row_of_token, const int32_t* __restrict__ block_table,
    int table_stride, int page_size, int n_tokens, int heads, int kv_heads, int out_ld, int n_pages, float scale, int window,
    const ImparoAttentionRule rule) {
    __shared__ __attribute__((aligned(16))) float q_rows[ATT_WAVES][HD];
    constexpr int DPL = HD / WAVE, AHEAD = 32 / DPL;
    const int lane = threadIdx.x & (WAVE - 1);
    const int wave = threadIdx.x / WAVE;
    const long long id = (long long)blockIdx.x * ATT_WAVES + wave;
    if (id >= (long long)n_tokens * heads) return;
    const int t = (int)(id / heads);
    const int h = (int)(id - (long long)t * heads);
    const int kvh = h / (heads / kv_heads);
    const int pos = positions[t];
    const int lo = first_seen(pos, window);
    const int32_t* table = block_table + (size_t)row_of_token[t] * table_stride;
    float* qr = q_rows[wave];
#pragma unroll
    for (int j = 0; j < DPL; ++j) qr[lane + j * WAVE] = q[((size_t)t * heads + h) * HD + lane + j * WAVE];
    wave_lds_sync();

    const int lo_chunk = (lo / WAVE) * WAVE;
    const int keep = rule.keep_first;
    auto next_of = [&](int c) { return (c + WAVE >= keep && c + WAVE < lo_chunk) ? lo_chunk : c + WAVE; };
    // which row of the caches holds this lane's key of chunk c, -1: none (a token at a position below 0 has no keys, and its
    // place in the table is read all the same)
    auto row_of = [&](int c) __attribute__((always_inline)) {
        const int p = c + lane;
        const bool valid = p <= pos && (p >= lo || p < keep);
        const int page = table[max(min(p, pos), 0) / page_size];
        return valid && page >= 0 && page < n_pages ? (page * kv_heads + kvh) * page_size + p % page_size : -1;
    };
    float4 key[HD / 4];
    auto ask = [&](int row) __attribute__((always_inline)) {
        const float4* src = reinterpret_cast<const float4*>(k_cache + (size_t)max(row, 0) * HD);
#pragma unroll
        for (int i = 0; i < HD / 4; ++i) key[i] = src[i];
    };
    float acc[DPL];
#pragma unroll
    for (int j = 0; j < DPL; ++j) acc[j] = 0.f;
    float m = -INFINITY, l = 0.f;
    int c = keep > 0 ? 0 : lo_chunk;
    if constexpr (ONE) {
        const int row = row_of(c);
        if (row >= 0) ask(row);
        float s = 0.f;
#pragma unroll
        for (int i = 0; i < HD / 4; ++i) {
            const float4 qv = *reinterpret_cast<const float4*>(&qr[4 * i]);
            s = fmaf(qv.x, key[i].x, s);
            s = fmaf(qv.y, key[i].y, s);
            s = fmaf(qv.z, key[i].z, s);
            s = fmaf(qv.w, key[i].w, s);
        }
        s *= scale;
        if (rule.softcap > 0.f) s = rule.softcap * tanhf(s / rule.softcap);
        if (row < 0) s = -INFINITY;
        m = fmaxf(m, wave_max(s));
        const float pe = row >= 0 ? expf(s - m) : 0.f;
        l = wave_sum(pe);
        for (int k0 = 0; k0 <= pos - c; k0 += 8) {
            float v[8][DPL], w[8];
            int at[8];
#pragma unroll
            for (int kk = 0; kk < 8; ++kk) {
                at[kk] = __builtin_amdgcn_readlane(row, k0 + kk);
                w[kk] = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(pe), k0 + kk));
#pragma unroll
                for (int j = 0; j < DPL; ++j) v[kk][j] = v_cache[(size_t)max(at[kk], 0) * HD + lane + j * WAVE];
            }
#pragma unroll
            for (int kk = 0; kk < 8; ++kk)
#pragma unroll
                for (int j = 0; j < DPL; ++j) acc[j] = at[kk] >= 0 ? fmaf(w[kk], v[kk][j], acc[j]) : acc[j];
        }
    } else {
        int row = row_of(c), row_next = row_of(min(next_of(c), pos));      // (places are looked up two chunks ahead of their rows)
        ask(row);
        while (c <= pos) {
            float s = 0.f;
#pragma unroll
            for (int i = 0; i < HD / 4; ++i) {
                const float4 qv = *reinterpret_cast<const float4*>(&qr[4 * i]);
                s = fmaf(qv.x, key[i].x, s);
                s = fmaf(qv.y, key[i].y, s);
                s = fmaf(qv.z, key[i].z, s);
                s = fmaf(qv.w, key[i].w, s);
            }
            s *= scale;
            if (rule.softcap > 0.f) s = rule.softcap * tanhf(s / rule.softcap);
            if (row < 0) s = -INFINITY;
            const int c_next = next_of(c);
            ask(row_next);
            const int row_after = row_of(min(next_of(c_next), pos));       // (past the end: nobody looks at it)
            const float m_new = fmaxf(m, wave_max(s));
            const float pe = row >= 0 ? expf(s - m_new) : 0.f;
            const float corr = (m == -INFINITY) ? 0.f : expf(m - m_new);
            l = fmaf(l, corr, wave_sum(pe));
            m = m_new;
            const int n_keys = min(WAVE, pos - c + 1);
#pragma unroll
            for (int j = 0; j < DPL; ++j) acc[j] *= corr;
            for (int k0 = 0; k0 < n_keys; k0 += AHEAD) {
                float v[AHEAD][DPL], w[AHEAD];
                int at[AHEAD];
#pragma unroll
                for (int kk = 0; kk < AHEAD; ++kk) {
                    at[kk] = __builtin_amdgcn_readlane(row, k0 + kk);
                    w[kk] = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(pe), k0 + kk));
#pragma unroll
                    for (int j = 0; j < DPL; ++j) v[kk][j] = v_cache[(size_t)max(at[kk], 0) * HD + lane + j * WAVE];
                }
#pragma unroll
                for (int kk = 0; kk < AHEAD; ++kk)
#pragma unroll
                    for (int j = 0; j < DPL; ++j) acc[j] = at[kk] >= 0 ? fmaf(w[kk], v[kk][j], acc[j]) : acc[j];
            }
            c = c_next;
            row = row_next;
            row_next = row_after;
        }
    }
    float inv = l > 0.f ? 1.0f / l : 0.f;
    if (rule.sink) {                        // one more term of the denominator, without a key or a value
        const float sink = rule.sink[h], top = fmaxf(m, sink);
        const float w = (m == -INFINITY) ? 0.f : expf(m - top);
        inv = w / fmaf(l, w, expf(sink - top));
    }
    inv *= rule.out_scale;
    if (rule.gate) inv *= 1.0f / (1.0f + expf(-rule.gate[(size_t)t * rule.gate_ld + h]));
    float* dst = out + (size_t)t * out_ld + (size_t)h * HD;
#pragma unroll
    for (int j = 0; j < DPL; ++j) dst[lane + j * WAVE] = acc[j] * inv;
    if (h == heads - 1)
        for (int d = HD + lane; d < out_ld - h * HD; d += WAVE) dst[d] = 0.f;
}

// The same again for few tokens (a decode step): one wave's walk leaves the chip idle behind its chain of trips, 5 us a chunk. Of
// what a walk does only three things are a chain: the running maximum, which is the maximum of all chunks before whatever
// order it is taken in; the denominator, one multiply-add a chunk; and the weighted sum, one multiply-add a key. So a block has all
// heads of one kv head of a token, its waves take chunks side by side (scores, their maximum, then the weights under the
// maximum so far), the values wait in LDS, and a wave a head adds them up in the order of the keys: the same bits. Two tokens
// over 340 keys, 16 heads of 64 by 8, 27.4 -> 11.3 us, over 4,000 288 -> 85, of 128 50 -> 20 and 557 -> 163, 32 tokens over 340 keys 29.8 ->
// 16.4; over 40 keys 7.1 -> 6.1. What is left is a CU's way to memory, about 1 us for the keys and values of a chunk. Two float32
// requests of 333 tokens, 8 decoded, 15.35 -> 14.48 ms.
template <int HD> struct SplitF32 {
    static constexpr int WAVES = HD == 64 ? 8 : 4;           // chunks at once, whose rows, keys and then values, fill 136 KB of LDS
    static constexpr int LD = HD + 4;                        // floats from row to row there: lanes that read a row each meet no bank twice
};
template <int HD, int GMAX>
__global__ __launch_bounds__(SplitF32<HD>::WAVES * WAVE, 1) void k_attention_split_f32(
    const float* __restrict__ q, const float* __restrict__ k_cache, const float* __restrict__ v_cache, float* __restrict__ out,
    const int32_t* __restrict__ positions, const int32_t* __restrict__ row_of_token, const int32_t* __restrict__ block_table,
    int table_stride, int page_size, int heads, int kv_heads, int out_ld, int n_pages, float scale, int window,
    const ImparoAttentionRule rule) {
    typedef float f32x4 __attribute__((ext_vector_type(4)));    // (arrays of the header's float4 end up in memory here)
    constexpr int W = SplitF32<HD>::WAVES, LD = SplitF32<HD>::LD, DPL = HD / WAVE;
    constexpr int PIECES = HD / 4;                           // of a row, and of a lane's share of a chunk
    extern __shared__ __attribute__((aligned(16))) float values[];       // [W][64][LD]
    __shared__ __attribute__((aligned(16))) float q_rows[GMAX][HD];
    __shared__ __attribute__((aligned(16))) float weights[GMAX][W][WAVE];
    __shared__ float top_of[GMAX][W], sum_of[GMAX][W], corr_of[GMAX][W];
    __shared__ unsigned long long rows_of[W];                // which keys of a chunk there are
    const int lane = threadIdx.x & (WAVE - 1), wave = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
    const int t = blockIdx.x / kv_heads, kvh = blockIdx.x - t * kv_heads, G = heads / kv_heads;
    const int pos = positions[t];
    const int lo = first_seen(pos, window), keep = rule.keep_first;
    const int32_t* table = block_table + (size_t)row_of_token[t] * table_stride;
    // chunk i of the walk starts at 64 i, or behind the first positions that stay at 64 i + gap
    const int keep_end = (keep + WAVE - 1) / WAVE * WAVE, gap = max(0, lo / WAVE * WAVE - keep_end);
    const int chunks = pos < 0 ? 0 : (pos - gap) / WAVE + 1;
    auto start_of = [&](int i) { return i * WAVE < keep_end ? i * WAVE : i * WAVE + gap; };
    for (int i = threadIdx.x; i < G * HD; i += W * WAVE) q_rows[i / HD][i % HD] = q[((size_t)t * heads + kvh * G) * HD + i];
    float m[GMAX], l = 0.f, acc[DPL];                        // m of every head in every wave; l and acc of the head that a wave adds up
#pragma unroll
    for (int g = 0; g < GMAX; ++g) m[g] = -INFINITY;
#pragma unroll
    for (int j = 0; j < DPL; ++j) acc[j] = 0.f;
    // A round: W chunks, one a wave. A walk of one chunk (`alone_as`) has nothing for the other waves but its heads: one a wave, each with
    // the chunk's keys and values of its own, of those the sixteens of rows that hold keys (what LDS has in place of the others is not
    // looked at). Launch behind launch, a block a head | so, 16 heads by 4 of 128: 5 keys 6.0 | 6.1 us, 40 keys 9.1 | 7.7, 32 by 8 of 64
    // 5.4 | 4.8, 7.3 | 5.6 (16 by 4 with the whole chunk asked for 8.8 over 5 keys). As branches in the code of the other rounds this cost those 0.3 to 0.7 us.
    auto round = [&](auto alone_as, int first) __attribute__((always_inline)) {
        constexpr bool alone = decltype(alone_as)::value;
        const int slot = alone ? 0 : wave;                   // the chunk of this round that the wave makes
        const bool busy = alone ? wave < G : first + wave < chunks;      // (the last round: a wave may have none)
        constexpr int QUARTER = PIECES / 4;
        const int first_row = keep > 0 ? 0 : lo - start_of(0), rows_end = pos + 1 - start_of(0);
        auto wanted = [&](int i) { return i / QUARTER * 16 < rows_end && i / QUARTER * 16 + 16 > first_row; };
        f32x4 key[PIECES], v[PIECES];
        bool there = false;
        if (busy) {
        const int p = start_of(first + slot) + lane;
        const int page = table[min(p, pos) / page_size];
        there = p <= pos && (p >= lo || p < keep) && page >= 0 && page < n_pages;
        const int row = there ? (page * kv_heads + kvh) * page_size + p % page_size : 0;
        // 64 lanes ask for 1,024 bytes of neighbouring rows: a row a lane, each instruction would meet 64 lines
        unsigned at[PIECES];                                 // (a pool holds up to 2^32 numbers)
#pragma unroll
        for (int i = 0; i < PIECES; ++i) {
            const unsigned piece = i * WAVE + lane;
            at[i] = (unsigned)__shfl(row, piece / PIECES) * HD + piece % PIECES * 4;
        }
#pragma unroll
        for (int i = 0; i < PIECES; i += QUARTER)
            if (!alone || wanted(i))
#pragma unroll
                for (int j = i; j < i + QUARTER; ++j) key[j] = *reinterpret_cast<const f32x4*>(k_cache + (size_t)at[j]);
#pragma unroll
        for (int i = 0; i < PIECES; i += QUARTER)
            if (!alone || wanted(i))
#pragma unroll
                for (int j = i; j < i + QUARTER; ++j) v[j] = *reinterpret_cast<const f32x4*>(v_cache + (size_t)at[j]);
        }
        float* rows_lds = values + (size_t)wave * WAVE * LD;
        auto put = [&](const f32x4 (&piece)[PIECES]) __attribute__((always_inline)) {
#pragma unroll
            for (int i = 0; i < PIECES; i += QUARTER)
                if (!alone || wanted(i))
#pragma unroll
                    for (int j = i; j < i + QUARTER; ++j)
                        *reinterpret_cast<f32x4*>(rows_lds + (j * WAVE + lane) / PIECES * LD + lane % PIECES * 4) = piece[j];
        };
        __syncthreads();                                     // (queries are there; the values before are read)
        float s[GMAX];
#pragma unroll
        for (int g = 0; g < GMAX; ++g) s[g] = 0.f;
        if (busy) {
        put(key);
        wave_lds_sync();
#pragma unroll
        for (int i = 0; i < PIECES; ++i) key[i] = *reinterpret_cast<const f32x4*>(rows_lds + lane * LD + 4 * i);
        wave_lds_sync();
        put(v);
        auto score = [&](float& sum, int g, int i) __attribute__((always_inline)) {
            const f32x4 qv = *reinterpret_cast<const f32x4*>(&q_rows[g][4 * i]);
            sum = fmaf(qv.x, key[i].x, sum);
            sum = fmaf(qv.y, key[i].y, sum);
            sum = fmaf(qv.z, key[i].z, sum);
            sum = fmaf(qv.w, key[i].w, sum);
        };
        if constexpr (alone) {
            float mine = 0.f;
#pragma unroll
            for (int i = 0; i < PIECES; ++i) score(mine, wave, i);
#pragma unroll
            for (int g = 0; g < GMAX; ++g) s[g] = mine;
        } else {
#pragma unroll
            for (int i = 0; i < PIECES; ++i)
#pragma unroll
                for (int g = 0; g < GMAX; ++g)
                    if (g < G) score(s[g], g, i);
        }
        }
        const unsigned long long keys = __ballot(there);
#pragma unroll
        for (int g = 0; g < GMAX; ++g) {
            if (g >= G || (alone && g != wave)) continue;
            s[g] *= scale;
            if (rule.softcap > 0.f) s[g] = rule.softcap * tanhf(s[g] / rule.softcap);
            if (!there) s[g] = -INFINITY;
            const float top = wave_max(s[g]);
            if (lane == 0) top_of[g][slot] = top;          // (of no keys: -inf)
        }
        if (lane == 0) rows_of[wave] = keys;
        __syncthreads();
#pragma unroll
        for (int g = 0; g < GMAX; ++g) {
            if (g >= G || (alone && g != wave)) continue;
            float before = m[g], all = m[g];
#pragma unroll
            for (int w = 0; w < W; ++w) {
                const float top = top_of[g][alone ? 0 : w];
                before = w < slot ? fmaxf(before, top) : before;
                all = fmaxf(all, top);
            }
            const float m_new = fmaxf(before, top_of[g][slot]);
            const float pe = there ? expf(s[g] - m_new) : 0.f;
            const float corr = (before == -INFINITY) ? 0.f : expf(before - m_new);
            const float sum = wave_sum(pe);
            weights[g][slot][lane] = pe;
            if (lane == 0) sum_of[g][slot] = sum, corr_of[g][slot] = corr;
            m[g] = all;
        }
        __syncthreads();
        if (wave < G) {
            for (int w = 0; w < min(W, chunks - first); ++w) {
                const float corr = corr_of[wave][w];
                l = fmaf(l, corr, sum_of[wave][w]);
#pragma unroll
                for (int j = 0; j < DPL; ++j) acc[j] *= corr;
                const int from = alone ? wave : w;
                const unsigned long long have = rows_of[from];
                const float* vw = values + (size_t)from * WAVE * LD + lane;
                const float* pw = weights[wave][w];
                // (sixteen keys ahead of the chain)
                constexpr int N = 16;
                float vn[N][DPL], pn[N];
                auto ask = [&](int k) __attribute__((always_inline)) {
#pragma unroll
                    for (int i = 0; i < N; i += 4) {
                        const f32x4 p4 = *reinterpret_cast<const f32x4*>(pw + k + i);
#pragma unroll
                        for (int n = 0; n < 4; ++n) pn[i + n] = p4[n];
                    }
#pragma unroll
                    for (int i = 0; i < N; ++i)
#pragma unroll
                        for (int j = 0; j < DPL; ++j) vn[i][j] = vw[(k + i) * LD + j * WAVE];
                };
                ask(0);
#pragma unroll
                for (int k = 0; k < WAVE; k += N) {
                    float vk[N][DPL], pk[N];
#pragma unroll
                    for (int i = 0; i < N; ++i) {
                        pk[i] = pn[i];
#pragma unroll
                        for (int j = 0; j < DPL; ++j) vk[i][j] = vn[i][j];
                    }
                    if (k + N < WAVE) ask(k + N);
                    const unsigned some = (unsigned)(have >> k) & ((1u << N) - 1);
                    if (some == (1u << N) - 1) {
#pragma unroll
                        for (int i = 0; i < N; ++i)
#pragma unroll
                            for (int j = 0; j < DPL; ++j) acc[j] = fmaf(pk[i], vk[i][j], acc[j]);
                    } else if (some) {
#pragma unroll
                        for (int i = 0; i < N; ++i)
#pragma unroll
                            for (int j = 0; j < DPL; ++j) {
                                const float to = fmaf(pk[i], vk[i][j], acc[j]);
                                acc[j] = some >> i & 1 ? to : acc[j];
                            }
                    }
                }
            }
        }
    };
    if (chunks == 1)
        round(std::true_type{}, 0);
    else
        for (int first = 0; first < chunks; first += W) round(std::false_type{}, first);
    if (wave >= G) return;
    const int h = kvh * G + wave;
    float inv = l > 0.f ? 1.0f / l : 0.f;
    if (rule.sink) {                        // one more term of the denominator, without a key or a value
        float mine = m[0];
#pragma unroll
        for (int g = 1; g < GMAX; ++g) mine = g == wave ? m[g] : mine;
        const float sink = rule.sink[h], top = fmaxf(mine, sink);
        const float w = (mine == -INFINITY) ? 0.f : expf(mine - top);
        inv = w / fmaf(l, w, expf(sink - top));
    }
    inv *= rule.out_scale;
    if (rule.gate) inv *= 1.0f / (1.0f + expf(-rule.gate[(size_t)t * rule.gate_ld + h]));
    float* dst = out + (size_t)t * out_ld + (size_t)h * HD;
#pragma unroll
    for (int j = 0; j < DPL; ++j) dst[lane + j * WAVE] = acc[j] * inv;
    if (h == heads - 1)
        for (int d = HD + lane; d < out_ld - h * HD; d += WAVE) dst[d] = 0.f;
}

template <int HD, int GMAX>
static int launch_split_f32(const float* q, const float* k_cache, const float* v_cache, float* out, const int32_t* positions,
                            const int32_t* row_of_token, const int32_t* block_table, int table_stride, int page_size, int n_tokens,
                            int heads, int kv_heads, int out_ld, int n_pages, float scale, int window, const ImparoAttentionRule& r,
                            hipStream_t s) {
    constexpr int W = SplitF32<HD>::WAVES, LDS = W * WAVE * SplitF32<HD>::LD * 4;
    if (hipFuncSetAttribute((const void*)k_attention_split_f32<HD, GMAX>, hipFuncAttributeMaxDynamicSharedMemorySize, LDS) != hipSuccess)
        return IMPARO_LAUNCH_FAILED;
    k_attention_split_f32<HD, GMAX><<<n_tokens * kv_heads, W * WAVE, LDS, s>>>(q, k_cache, v_cache, out, positions, row_of_token,
        block_table, table_stride, page_size, heads, kv_heads, out_ld, n_pages, scale, window, r);
    return launch_status();
}

static int check_attention_args(const void* q, const void* k_cache, const void* v_cache, void* out,
                                const int32_t* positions, const int32_t* row_of_token, const int32_t* block_table,
                                int table_stride, int page_size, int n_tokens, int heads, int kv_heads, int head_dim,
                                int n_pages, int window) {
    if (!q || !k_cache || !v_cache || !out || !positions || !row_of_token || !block_table) return IMPARO_BAD_ARGUMENT;
    if (n_tokens < 0 || heads <= 0 || kv_heads <= 0 || heads % kv_heads != 0) return IMPARO_BAD_ARGUMENT;
    if (head_dim <= 0 || head_dim > ATT_MAX_HEAD_DIM) return IMPARO_BAD_ARGUMENT;
    if (page_size <= 0 || table_stride <= 0 || n_pages <= 0) return IMPARO_BAD_ARGUMENT;
    return IMPARO_OK;
}

// Whether few float32 tokens take k_attention_split_f32: heads of 64 or 128, at most four a kv head, as long as each token's kv head has
// a CU of its own. Few keys of a window or a chunk that lie in two runs of 64 are two runs' reads there, for all heads of a wave, and with
// three or four heads a kv head a block a head is the faster way: us, a block a head | so, one token, a window of 20, 16 heads by 4 of 128
// over 130 keys 11.4 | 14.2, 32 by 8 of 64 over 1,100 8.8 | 9.7. As times of a block a head at worst, 16 by 4 of 128: windows of 40 1.20, of 56
// 1.14, of 64 1.11, of 72 1.04, of 96 0.81, chunks of 20 1.31 and of 100 1.24; 32 by 8 of 64: 1.08, 1.04, 1.02, 1.01, 0.82, 1.13 and 1.09; 12 by
// 4 of 128: a window of 8 1.35, of 40 1.03; up to two heads a kv head 0.95 for all. Chunks that start with a run of 64 have few keys in one run only.
extern "C" int imparo_attention_f32_split_pays(int n_tokens, int heads, int kv_heads, int head_dim, int window, int keep_first) {
    if (heads < 1 || kv_heads < 1 || heads % kv_heads || (head_dim != 64 && head_dim != 128)) return 0;
    const int G = heads / kv_heads;
    if (G > 4 || (long long)n_tokens * kv_heads > 256) return 0;
    if (window == 0 || keep_first > 0 || G <= 2) return 1;
    if (G == 3) return head_dim == 64 || window >= 32 || window <= -32;
    return window > 0 ? window >= 80 : window <= -128 || window % WAVE == 0;
}

// Keys of head_dim and values of value_dim a head: q [tokens, heads, head_dim], the value cache
// [pages, kv_heads, page, value_dim] (or transposed inside the page), out [tokens, out_ld] with out_ld >=
// heads * value_dim; what lies beyond the heads in a row is written as zeros.
static int attention_wave(const void* q, const void* k_cache, const void* v_cache, void* out, int dtype,
                          const int32_t* positions, const int32_t* row_of_token,
                          const int32_t* block_table, int table_stride, int page_size,
                          int n_tokens, int heads, int kv_heads, int head_dim, int value_dim, int out_ld,
                          int n_pages, float scale, int window, int v_transposed, int v_ld, imparo_stream stream,
                          const ImparoAttentionRule* rule = nullptr) {
    const int bad = check_attention_args(q, k_cache, v_cache, out, positions, row_of_token, block_table, table_stride,
                                         page_size, n_tokens, heads, kv_heads, head_dim, n_pages, window);
    if (bad) return bad;
    if (value_dim <= 0 || value_dim > ATT_MAX_HEAD_DIM || out_ld < heads * value_dim) return IMPARO_BAD_ARGUMENT;
    if (v_ld < value_dim || (v_transposed && v_ld != value_dim)) return IMPARO_BAD_ARGUMENT;
    const ImparoAttentionRule r = rule ? *rule : ImparoAttentionRule{0, 0.f, nullptr, 1.0f, nullptr, 0};
    if (imparo_attention_rule_bad(r, window)) return IMPARO_BAD_ARGUMENT;
    if (n_tokens == 0) return IMPARO_OK;
    const long long total = (long long)n_tokens * heads;
    const unsigned blocks = (unsigned)((total + ATT_WAVES - 1) / ATT_WAVES);
    hipStream_t s = (hipStream_t)stream;
    // heads of 64 or 128 whose values lie as the keys do, rows 16 bytes aligned and counted in 32 bits
    const bool plain = dtype == IMPARO_F32 && head_dim == value_dim && v_ld == head_dim && !v_transposed &&
                       !((uintptr_t)k_cache & 15) && (long long)n_pages * kv_heads * page_size < (1LL << 31);
#define WAVE_F32_GO(HD, ONE)                                                                                            \
    k_attention_wave_f32<HD, ONE><<<blocks, ATT_WAVES * WAVE, 0, s>>>(                                                  \
        (const float*)q, (const float*)k_cache, (const float*)v_cache, (float*)out, positions, row_of_token, block_table, \
        table_stride, page_size, n_tokens, heads, kv_heads, out_ld, n_pages, scale, window, r)
    // One chunk where the table has no room for more keys. Otherwise, where the waves are many and not bound by their trips, the
    // general kernel: for windows of less than a chunk (1,000 tokens, 64 heads of 64, 20 keys: 222 us in the loop, 206 there),
    // and with heads of 128, whose registers leave a SIMD one wave where it has four, for any window (64 heads, 128 keys: 1,292
    // and 1,146) and short contexts (4 prompts of 100 tokens, 64 heads 251 and 216; one of 333 537 and 554).
    const long long room = (long long)table_stride * page_size;
    const bool one = room <= WAVE, few = total <= 4096;
    // Few tokens: a block of several waves for a token's kv head (k_attention_split_f32).
    const int G = heads / kv_heads;
    if (plain && !one && imparo_attention_f32_split_pays(n_tokens, heads, kv_heads, head_dim, window, r.keep_first) && !((uintptr_t)v_cache & 15) &&
        (long long)n_pages * kv_heads * page_size * head_dim < (1LL << 32)) {
#define SPLIT_F32(HD, GMAX)                                                                                             \
    return launch_split_f32<HD, GMAX>((const float*)q, (const float*)k_cache, (const float*)v_cache, (float*)out, positions, row_of_token, \
                                      block_table, table_stride, page_size, n_tokens, heads, kv_heads, out_ld, n_pages, scale, window, r, s)
        if (head_dim == 64 && G <= 2) SPLIT_F32(64, 2);
        if (head_dim == 64) SPLIT_F32(64, 4);
        if (G <= 2) SPLIT_F32(128, 2);
        SPLIT_F32(128, 4);
#undef SPLIT_F32
    }
    if (plain && head_dim == 64 && one)
        WAVE_F32_GO(64, true);
    else if (plain && head_dim == 64 && (few || window <= 0 || window >= WAVE))
        WAVE_F32_GO(64, false);
    else if (plain && head_dim == 128 && one)
        WAVE_F32_GO(128, true);
    else if (plain && head_dim == 128 && (few || (window <= 0 && room >= 320)))
        WAVE_F32_GO(128, false);
#undef WAVE_F32_GO
    else if (dtype == IMPARO_F32)
        k_attention_wave<float><<<blocks, ATT_WAVES * WAVE, 0, s>>>(
            (const float*)q, (const float*)k_cache, (const float*)v_cache, (float*)out, positions, row_of_token,
            block_table, table_stride, page_size, n_tokens, heads, kv_heads, head_dim, value_dim, out_ld, n_pages, scale, window, v_transposed,
            v_ld, r);
    else if (dtype == IMPARO_BF16)
        k_attention_wave<bf16_t><<<blocks, ATT_WAVES * WAVE, 0, s>>>(
            (const bf16_t*)q, (const bf16_t*)k_cache, (const bf16_t*)v_cache, (bf16_t*)out, positions, row_of_token,
            block_table, table_stride, page_size, n_tokens, heads, kv_heads, head_dim, value_dim, out_ld, n_pages, scale, window,
            v_transposed, v_ld, r);
    else
        return IMPARO_BAD_ARGUMENT;
    return launch_status();
}

extern "C" int imparo_attention_dv(const void* q, const void* k_cache, const void* v_cache, void* out, int dtype,
                                const int32_t* positions, const int32_t* row_of_token,
                                const int32_t* block_table, int table_stride, int page_size,
                                int n_tokens, int heads, int kv_heads, int head_dim, int value_dim, int out_ld,
                                int n_pages, float scale, int window, int v_transposed, imparo_stream stream) {
    return attention_wave(q, k_cache, v_cache, out, dtype, positions, row_of_token, block_table, table_stride, page_size,
                          n_tokens, heads, kv_heads, head_dim, value_dim, out_ld, n_pages, scale, window, v_transposed,
                          value_dim, stream);
}

extern "C" int imparo_attention_ruled(const void* q, const void* k_cache, const void* v_cache, void* out, int dtype,
                                      const int32_t* positions, const int32_t* row_of_token, const int32_t* block_table,
                                      int table_stride, int page_size, int n_tokens, int heads, int kv_heads, int head_dim,
                                      int value_dim, int out_ld, int n_pages, float scale, int window, int v_transposed,
                                      const ImparoAttentionRule* rule, imparo_stream stream) {
    return attention_wave(q, k_cache, v_cache, out, dtype, positions, row_of_token, block_table, table_stride, page_size,
                          n_tokens, heads, kv_heads, head_dim, value_dim, out_ld, n_pages, scale, window, v_transposed,
                          value_dim, stream, rule);
}

// Attention over a cached latent: every head reads the same rows [pages, page, row_dim]; a key is a whole
// row, its value the row's first value_dim numbers (queries carry their side of the keys' up-projection,
// the values' up-projection follows the weighted sum). out [tokens, heads * value_dim].
extern "C" int imparo_attention_latent(const void* q, const void* rows_cache, void* out, int dtype,
                                       const int32_t* positions, const int32_t* row_of_token,
                                       const int32_t* block_table, int table_stride, int page_size, int n_tokens,
                                       int heads, int row_dim, int value_dim, int n_pages, float scale, int window,
                                       imparo_stream stream) {
    if (value_dim > row_dim) return IMPARO_BAD_ARGUMENT;
    return attention_wave(q, rows_cache, rows_cache, out, dtype, positions, row_of_token, block_table, table_stride,
                          page_size, n_tokens, heads, 1, row_dim, value_dim, heads * value_dim, n_pages, scale, window, 0,
                          row_dim, stream);
}

extern "C" int imparo_attention(const void* q, const void* k_cache, const void* v_cache, void* out, int dtype,
                                const int32_t* positions, const int32_t* row_of_token,
                                const int32_t* block_table, int table_stride, int page_size,
                                int n_tokens, int heads, int kv_heads, int head_dim, int n_pages,
                                float scale, int window, int v_transposed, imparo_stream stream) {
    if (head_dim % 16 != 0) return IMPARO_BAD_ARGUMENT;
    return imparo_attention_dv(q, k_cache, v_cache, out, dtype, positions, row_of_token, block_table, table_stride,
                               page_size, n_tokens, heads, kv_heads, head_dim, head_dim, heads * head_dim, n_pages, scale,
                               window, v_transposed, stream);
}

// Asks the runtime about one kernel of this file, which makes it load the file's code onto the
// current device (it loads a file's kernels when one of them is first used; a stream under capture
// cannot do that).
int imparo_load_code_attention() {
    hipFuncAttributes attributes;
    return hipFuncGetAttributes(&attributes, reinterpret_cast<const void*>(&k_attention_wave<float>)) == hipSuccess ? IMPARO_OK
                                                                                              : IMPARO_LAUNCH_FAILED;
}
