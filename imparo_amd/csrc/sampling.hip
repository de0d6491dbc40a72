// Picking the next token from float32 logits: argmax (smallest index at the
// maximum, NaN never wins) and temperature sampling by inverse CDF.
#include "common.h"
#include "api.h"
#include <limits.h>

struct Best {
    float v;
    int i;
};

__device__ __forceinline__ Best better(Best a, Best b) {
    return (b.v > a.v || (b.v == a.v && b.i < a.i)) ? b : a;
}

__device__ __forceinline__ Best block_best(Best b, Best* scratch) {
    b = better(b, Best{lane_xor<32>(b.v), lane_xor<32>(b.i)});
    b = better(b, Best{lane_xor<16>(b.v), lane_xor<16>(b.i)});
    b = better(b, Best{lane_xor<8>(b.v), lane_xor<8>(b.i)});
    b = better(b, Best{lane_xor<4>(b.v), lane_xor<4>(b.i)});
    b = better(b, Best{lane_xor<2>(b.v), lane_xor<2>(b.i)});
    b = better(b, Best{lane_xor<1>(b.v), lane_xor<1>(b.i)});
    const int lane = threadIdx.x & (WAVE - 1), wave = threadIdx.x / WAVE;
    const int n_waves = (blockDim.x + WAVE - 1) / WAVE;
    __syncthreads();
    if (lane == 0) scratch[wave] = b;
    __syncthreads();
    Best r = scratch[0];
    for (int w = 1; w < n_waves; ++w) r = better(r, scratch[w]);
    return r;
}

__device__ __forceinline__ Best row_best(const float* __restrict__ row, int vocab, Best* scratch) {
    Best b;
    b.v = -INFINITY;
    b.i = INT_MAX;
    if ((vocab & 3) == 0 && (((uintptr_t)row) & 15) == 0) {
        // The maximum first, four values a load and sixteen loads in flight (a row of 65,536 on 1,024 threads is one trip
        // to memory; no load sits under a branch: past the end the row's last piece is read again, which changes no
        // maximum), then its smallest index by the threads that met it, from the run of loads they met it in: a comparison
        // and a choice of index for every value were a third of the time (one row of 65,536 9.0 us, so 6.2).
        const float4* row4 = reinterpret_cast<const float4*>(row);
        const int n4 = vocab >> 2;
        if (n4 <= (int)blockDim.x) {
            // one load a thread: the maximum and its index together, one meeting of the block (a row of 1,000 in two 3.8 us)
            const float4 v = row4[min((int)threadIdx.x, n4 - 1)];
            const float vs[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
            for (int j = 0; j < 4; ++j)
                if ((int)threadIdx.x < n4 && (vs[j] > b.v || (vs[j] == b.v && 4 * (int)threadIdx.x + j < b.i))) {
                    b.v = vs[j];
                    b.i = 4 * (int)threadIdx.x + j;
                }
            b = block_best(b, scratch);
            if (b.i == INT_MAX) b.i = 0;   // every value was NaN
            return b;
        }
        constexpr int DEEP = 16;
        float m = -INFINITY;
        int met = 0;
        for (int first = threadIdx.x; first < n4; first += DEEP * (int)blockDim.x) {
            float4 v[DEEP];
#pragma unroll
            for (int k = 0; k < DEEP; ++k) v[k] = row4[min(first + k * (int)blockDim.x, n4 - 1)];
            float mm = -INFINITY;
#pragma unroll
            for (int k = 0; k < DEEP; ++k) mm = fmaxf(mm, fmaxf(fmaxf(v[k].x, v[k].y), fmaxf(v[k].z, v[k].w)));
            if (mm > m) {
                m = mm;
                met = first;
            }
        }
        float top = wave_max(m);
        const int n_waves = (blockDim.x + WAVE - 1) / WAVE;
        if ((threadIdx.x & (WAVE - 1)) == 0) scratch[threadIdx.x / WAVE].v = top;
        __syncthreads();
        float tops[16];
#pragma unroll
        for (int w = 0; w < 16; ++w) tops[w] = scratch[min(w, n_waves - 1)].v;
#pragma unroll
        for (int w = 0; w < 16; ++w) top = fmaxf(top, tops[w]);
        if (top > -INFINITY) {                       // (nothing but -inf and NaN: value by value below)
            if (m == top) {
                float4 v[DEEP];
#pragma unroll
                for (int k = 0; k < DEEP; ++k) v[k] = row4[min(met + k * (int)blockDim.x, n4 - 1)];
#pragma unroll
                for (int k = DEEP - 1; k >= 0; --k) {
                    const int i = min(met + k * (int)blockDim.x, n4 - 1);
                    const float vs[4] = {v[k].x, v[k].y, v[k].z, v[k].w};
#pragma unroll
                    for (int j = 3; j >= 0; --j)
                        if (vs[j] == top) b.i = 4 * i + j;
                }
                b.v = top;
            }
            return block_best(b, scratch);
        }
    }
    for (int i = threadIdx.x; i < vocab; i += blockDim.x) {
        const float v = row[i];
        if (v > b.v || (v == b.v && i < b.i)) {
            b.v = v;
            b.i = i;
        }
    }
    b = block_best(b, scratch);
    if (b.i == INT_MAX) b.i = 0;   // every value was NaN
    return b;
}

__global__ void k_argmax_rows(const float* __restrict__ logits, int32_t* __restrict__ out, int vocab) {
    __shared__ Best scratch[16];
    const Best b = row_best(logits + (size_t)blockIdx.x * vocab, vocab, scratch);
    if (threadIdx.x == 0) out[blockIdx.x] = b.i;
}

extern "C" int imparo_argmax_rows(const float* logits, int32_t* out, int n_rows, int vocab, imparo_stream stream) {
    if (!logits || !out || n_rows < 0 || vocab <= 0) return IMPARO_BAD_ARGUMENT;
    if (n_rows == 0) return IMPARO_OK;
    const int threads = vocab >= 16384 ? 1024 : 256;
    k_argmax_rows<<<n_rows, threads, 0, (hipStream_t)stream>>>(logits, out, vocab);
    return launch_status();
}

// Each thread owns one contiguous piece of the row. Piece sums are scanned in
// thread order, the piece holding u * total is walked element by element: the
// pick is the first index whose running sum exceeds the target.
// The sums' order is part of the result (two machines that draw the same number pick the same token), so the scan
// over the pieces and the walk inside one stay chains of additions; what a chain adds is fetched ahead of it, sixteen
// values a time, and all that is no addition (exponentials, comparisons) is done by the whole block. Measured, 64
// rows of 65,536 logits: 153 us with both chains reading LDS and memory value by value, 38 us so (28 us for rows of 16,384).
#define SAMPLE_THREADS 1024
__global__ __launch_bounds__(SAMPLE_THREADS) void k_sample_rows(
    const float* __restrict__ logits, const float* __restrict__ temperature, const float* __restrict__ uniform,
    int32_t* __restrict__ out, int vocab) {
    __shared__ Best scratch[16];
    __shared__ __attribute__((aligned(16))) float sums[SAMPLE_THREADS], before[SAMPLE_THREADS];
    __shared__ int first_past, last_positive, found;
    __shared__ float cum_shared, target_shared;
    const float* row = logits + (size_t)blockIdx.x * vocab;
    const Best top = row_best(row, vocab, scratch);
    const float temp = temperature[blockIdx.x];
    if (!(temp > 0.f)) {
        if (threadIdx.x == 0) out[blockIdx.x] = top.i;
        return;
    }
    const float inv_t = 1.0f / temp;
    const int tid = threadIdx.x, threads = blockDim.x;         // (a multiple of 16)
    const int piece = (vocab + threads - 1) / threads;
    const int begin = min(vocab, tid * piece), end = min(vocab, begin + piece);
    float local = 0.f;
    int i = begin;
    if (piece % 16 == 0 && (((uintptr_t)row) & 15) == 0) {     // whole vectors, sixteen values in flight
        for (; i + 16 <= end; i += 16) {
            float4 v[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) v[j] = *reinterpret_cast<const float4*>(row + i + 4 * j);
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const float x[4] = {v[j].x, v[j].y, v[j].z, v[j].w};
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    const float e = expf((x[k] - top.v) * inv_t);
                    if (e == e) local += e;   // a NaN logit has probability zero
                }
            }
        }
    }
    for (; i < end; ++i) {
        const float e = expf((row[i] - top.v) * inv_t);
        if (e == e) local += e;
    }
    sums[tid] = local;
    if (tid == 0) {
        first_past = INT_MAX;
        last_positive = 0;
        found = -1;
    }
    __syncthreads();
    if (tid == 0) {                                            // what lies before each piece, and the total
        float total = 0.f;
        float4 next[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) next[j] = *reinterpret_cast<const float4*>(&sums[4 * j]);
        for (int t = 0; t < threads; t += 16) {
            float4 now[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                now[j] = next[j];
                next[j] = *reinterpret_cast<const float4*>(&sums[min(t + 16, threads - 16) + 4 * j]);
            }
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                float4 b;
                b.x = total, total += now[j].x;
                b.y = total, total += now[j].y;
                b.z = total, total += now[j].z;
                b.w = total, total += now[j].w;
                *reinterpret_cast<float4*>(&before[t + 4 * j]) = b;
            }
        }
        target_shared = uniform[blockIdx.x] * total;
    }
    __syncthreads();
    const float target = target_shared;
    if (local > 0.f) {
        if (before[tid] + local > target) atomicMin(&first_past, tid);
        atomicMax(&last_positive, tid);
    }
    __syncthreads();
    const int owner = first_past != INT_MAX ? first_past : last_positive;   // (rounding can push the target past the total)
    if (tid == 0) cum_shared = before[owner];
    const int own_begin = min(vocab, owner * piece), own_end = min(vocab, own_begin + piece);
    int last = top.i;
    for (int at = own_begin; at < own_end; at += threads) {
        __syncthreads();
        sums[tid] = at + tid < own_end ? expf((row[at + tid] - top.v) * inv_t) : 0.f;
        __syncthreads();
        if (tid == 0) {
            float cum = cum_shared;
            int pick = -1;
            const int n = min(threads, own_end - at);
            for (int t = 0; t < n && pick < 0; t += 16) {
                float4 v[4];
#pragma unroll
                for (int j = 0; j < 4; ++j) v[j] = *reinterpret_cast<const float4*>(&sums[t + 4 * j]);
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const float e[4] = {v[j].x, v[j].y, v[j].z, v[j].w};
#pragma unroll
                    for (int k = 0; k < 4; ++k) {
                        const bool on = e[k] > 0.f && pick < 0;
                        if (on) last = at + t + 4 * j + k;
                        cum = on ? cum + e[k] : cum;
                        if (on && cum > target) pick = last;
                    }
                }
            }
            cum_shared = cum;
            found = pick;
        }
        __syncthreads();
        if (found >= 0) break;
    }
    if (tid == 0) out[blockIdx.x] = found >= 0 ? found : last;
}

extern "C" int imparo_sample_rows(const float* logits, const float* temperature, const float* uniform, int32_t* out,
                                  int n_rows, int vocab, imparo_stream stream) {
    if (!logits || !temperature || !uniform || !out || n_rows < 0 || vocab <= 0) return IMPARO_BAD_ARGUMENT;
    if (n_rows == 0) return IMPARO_OK;
    const int threads = vocab >= 16384 ? SAMPLE_THREADS : 256;
    k_sample_rows<<<n_rows, threads, 0, (hipStream_t)stream>>>(logits, temperature, uniform, out, vocab);
    return launch_status();
}

// The hash of the sources this library was built from (given by the build), so that a
// library older than its sources is noticed when it is loaded.
#ifndef IMPARO_SOURCE_HASH
#define IMPARO_SOURCE_HASH "unknown"
#endif
extern "C" const char* imparo_hip_source_hash() { return IMPARO_SOURCE_HASH; }

// Asks the runtime about one kernel of this file, which makes it load the file's code onto the
// current device (it loads a file's kernels when one of them is first used; a stream under capture
// cannot do that).
int imparo_load_code_sampling() {
    hipFuncAttributes attributes;
    return hipFuncGetAttributes(&attributes, reinterpret_cast<const void*>(&k_argmax_rows)) == hipSuccess ? IMPARO_OK
                                                                                              : IMPARO_LAUNCH_FAILED;
}
