// Recurrences with a matrix of state a head and one decay a head and token:
//   S <- a S + k v^T,                 o = S^T q                  (a linear attention with decay)
//   S <- a S;  u = b (v - S^T k);  S <- S + k u^T,  o = S^T q    (the gated delta rule)
//   the same with S <- diag(g) S, one decay a state row          (the gated delta rule, decays a channel)
// S [dim, vdim] float32 per request and head, carried from token to token. The decay a is a constant of
// the head, or exp(-rate_h softplus(raw + bias_h)) of a projected number (the step; the values may be
// multiplied by that step, as a state-space layer does, and the head's result may take D_h x on top). b is
// the sigmoid of a projected number. Heads may share queries and keys in groups of neighbours (q_div, k_div
// heads read one). Decays, steps, gates, the state and every sum are float32 whatever the engine's dtype.
//
// A block takes one request's segment, one head and a run of value columns. A thread keeps a slice of one
// column of S in registers: KS neighbouring lanes share a column, so that the sums over dim (the delta
// rule's S^T k, every o) end with a few exchanges inside a wave. The tokens' q, k, v and scalars come
// through LDS eight tokens at a time. Every sum runs in an order that dim alone decides.
//
// A long segment of the first form is walked in three launches, its chunks side by side (the recurrence
// is linear in S with a scalar factor: after a chunk S = (product of the chunk's a) S_before + what the chunk
// makes of a zero state). The delta rule's transition is a matrix (a (I - b k k^T)): its long segments take the
// form in chunks further down (a triangle solved a chunk, then the chunks in order), short ones this walk.
//
// Beside it: what such mixers do to a head before the walk (unit length, rotation, a factor) and to the
// heads behind it (a gate and a norm in groups of the row).
#include "common.h"
#include "api.h"

#define DS_KPT 16             // entries of a column a thread keeps at most
#define DS_TOKENS 8           // tokens staged in LDS at once
#define DS_MAX_THREADS 256
#define DS_MAX_DIM 512

__device__ __forceinline__ float ds_sigmoid(float z) { return 1.0f / (1.0f + expf(-z)); }
__device__ __forceinline__ float ds_silu(float z) { return z / (1.0f + expf(-z)); }
__device__ __forceinline__ float ds_softplus(float z) { return z > 20.0f ? z : log1pf(expf(z)); }

__device__ __forceinline__ float ds_gate(float z, int act) { return act ? ds_sigmoid(z) : ds_silu(z); }

struct DecayScanArgs {
    const float* q; int q_ld, q_off, q_div;      // head h reads q head h / q_div
    const float* k; int k_ld, k_off, k_div;
    const float* v; int v_ld, v_off;
    const float* decay_const;                    // [heads], or null: the decay comes from `step`
    const float* step; int step_ld, step_off;    // raw steps [tokens, heads]
    const float* step_bias;                      // [heads]
    const float* rate;                           // [heads]: a = exp(-rate softplus(raw + bias))
    int v_times_step;                            // v <- softplus(raw + bias) v
    const float* beta; int beta_ld, beta_off;    // raw [tokens, heads], the delta rule's only
    const float* skip;                           // [heads] or null: o += skip_h v (v as it came)
    float* state;                                // [slots, heads, dim, vdim]
    const int32_t* seg_start; const int32_t* seg_len; const int32_t* slot;
    float* out;                                  // [tokens, heads * vdim]
    int heads, dim, vdim, kpt;
    int chunk_tokens, max_chunks;
    float* chunk_state;                          // [rows * max_chunks, heads, dim, vdim]
    float* chunk_decay;                          // [rows * max_chunks, heads]
    int silu_in;                                 // q, k, v go through SiLU when they are read (token by token only)
};

// MODE 0: a segment from its request's state to its end. With chunks (blockIdx.x = row * max_chunks + chunk):
// MODE 1: a chunk that is not the segment's last, from a zero state: its end state goes to chunk_state, the
// product of its decays to chunk_decay, no results; MODE 2: a chunk from the state chunk_state holds for it,
// with results; the last chunk writes the request's state.
// V4: a thread's slice is whole 16-byte pieces, read as such. CHAN: step and step_bias hold heads x dim numbers, a
// decay for every state row.
template <int KS, int MODE, bool DELTA, bool V4, bool CHAN = false>
__global__ __launch_bounds__(DS_MAX_THREADS) void k_decay_scan(const DecayScanArgs A) {
    __shared__ __attribute__((aligned(16))) float sq[DS_TOKENS][DS_MAX_DIM], sk[DS_TOKENS][DS_MAX_DIM];
    __shared__ __attribute__((aligned(16))) float sg[CHAN ? DS_TOKENS : 1][CHAN ? DS_MAX_DIM : 4];
    __shared__ float sv[DS_TOKENS][DS_MAX_THREADS];
    __shared__ float sa[DS_TOKENS], sb[DS_TOKENS], sdt[DS_TOKENS];
    const int VB = blockDim.x / KS;                      // value columns of a block
    const int r = MODE == 0 ? blockIdx.x : blockIdx.x / A.max_chunks;
    const int chunk = MODE == 0 ? 0 : blockIdx.x - r * A.max_chunks;
    const int h = blockIdx.y, v0 = blockIdx.z * VB;
    const int tid = threadIdx.x, ks = tid % KS, vl = tid / KS;
    const int v = v0 + vl;
    const int heads = A.heads, dim = A.dim, vdim = A.vdim, kpt = A.kpt;
    const bool live = v < vdim;
    const int n_all = A.seg_len[r];
    const int n_chunks = MODE == 0 ? 1 : (n_all + A.chunk_tokens - 1) / A.chunk_tokens;
    if (MODE == 1 && chunk >= n_chunks - 1) return;      // (the whole block)
    if (MODE == 2 && chunk >= n_chunks) return;
    const int first = A.seg_start[r] + (MODE == 0 ? 0 : chunk * A.chunk_tokens);
    const int n = MODE == 0 ? n_all : min(A.chunk_tokens, n_all - chunk * A.chunk_tokens);
    const int dkp = KS * kpt;                            // dim, filled up to whole slices
    const int qh = h / A.q_div, kh = h / A.k_div;
    float* S_at = A.state + (((size_t)A.slot[r] * heads + h) * dim) * vdim;
    float* C_at = MODE == 0 ? nullptr : A.chunk_state + (((size_t)blockIdx.x * heads + h) * dim) * vdim;
    float S[DS_KPT];
    float decay_all = 1.f;
#pragma unroll
    for (int j = 0; j < DS_KPT; ++j) {
        const int k = ks * kpt + j;
        if constexpr (MODE == 1)
            S[j] = 0.f;
        else
            S[j] = (j < kpt && k < dim && live) ? (MODE == 0 ? S_at : C_at)[(size_t)k * vdim + v] : 0.f;
    }
    const float skip = A.skip ? A.skip[h] : 0.f;
    for (int t0 = 0; t0 < n; t0 += DS_TOKENS) {
        const int nt = min(DS_TOKENS, n - t0);
        __syncthreads();                                 // the last batch has been read
        for (int i = tid; i < nt * dkp; i += blockDim.x) {
            const int tok = i / dkp, k = i - tok * dkp;
            const size_t t = (size_t)(first + t0 + tok);
            float qv = k < dim ? A.q[t * A.q_ld + A.q_off + qh * dim + k] : 0.f;     // beyond dim: a state that stays zero
            float kv = k < dim ? A.k[t * A.k_ld + A.k_off + kh * dim + k] : 0.f;
            if (!DELTA && A.silu_in) qv = ds_silu(qv), kv = ds_silu(kv);
            sq[tok][k] = qv;
            sk[tok][k] = kv;
            if constexpr (CHAN) {
                const int kc = min(k, dim - 1);
                sg[tok][k] = expf(-A.rate[h] * ds_softplus(A.step[t * A.step_ld + A.step_off + h * dim + kc] +
                                                           A.step_bias[h * dim + kc]));
            }
        }
        for (int i = tid; i < nt * VB; i += blockDim.x) {
            const int tok = i / VB, c = i - tok * VB;
            float vv = (v0 + c) < vdim ? A.v[(size_t)(first + t0 + tok) * A.v_ld + A.v_off + h * vdim + v0 + c] : 0.f;
            if (!DELTA && A.silu_in) vv = ds_silu(vv);
            sv[tok][c] = vv;
        }
        if (tid < nt) {
            const size_t t = (size_t)(first + t0 + tid);
            float a, dt = 1.f;
            if constexpr (CHAN) {
                a = 1.f;
            } else if (A.decay_const) {
                a = A.decay_const[h];
            } else {
                dt = ds_softplus(A.step[t * A.step_ld + A.step_off + h] + A.step_bias[h]);
                a = expf(-A.rate[h] * dt);
            }
            sa[tid] = a;
            sdt[tid] = A.v_times_step ? dt : 1.f;
            sb[tid] = DELTA ? ds_sigmoid(A.beta[t * A.beta_ld + A.beta_off + h]) : 1.f;
        }
        __syncthreads();
        for (int tok = 0; tok < nt; ++tok) {
            const float a = sa[tok];
            const float raw = sv[tok][vl];
            float val = raw * sdt[tok];
            float acc = 0.f;
            float kk[DS_KPT], qq[DS_KPT];
            if constexpr (V4) {
#pragma unroll
                for (int j = 0; j < DS_KPT; j += 4)
                    if (j < kpt) {
                        const float4 k4 = *reinterpret_cast<const float4*>(&sk[tok][ks * kpt + j]);
                        const float4 q4 = *reinterpret_cast<const float4*>(&sq[tok][ks * kpt + j]);
                        kk[j] = k4.x, kk[j + 1] = k4.y, kk[j + 2] = k4.z, kk[j + 3] = k4.w;
                        qq[j] = q4.x, qq[j + 1] = q4.y, qq[j + 2] = q4.z, qq[j + 3] = q4.w;
                    }
            } else {
#pragma unroll
                for (int j = 0; j < DS_KPT; ++j)
                    if (j < kpt) {
                        kk[j] = sk[tok][ks * kpt + j];
                        qq[j] = sq[tok][ks * kpt + j];
                    }
            }
            if constexpr (DELTA) {
                float seen = 0.f;
                float gg[CHAN ? DS_KPT : 1];
                if constexpr (CHAN) {
#pragma unroll
                    for (int j = 0; j < DS_KPT; j += V4 ? 4 : 1)
                        if (j < kpt) {
                            if constexpr (V4) {
                                const float4 g4 = *reinterpret_cast<const float4*>(&sg[tok][ks * kpt + j]);
                                gg[j] = g4.x, gg[j + 1] = g4.y, gg[j + 2] = g4.z, gg[j + 3] = g4.w;
                            } else {
                                gg[j] = sg[tok][ks * kpt + j];
                            }
                        }
                }
#pragma unroll
                for (int j = 0; j < DS_KPT; ++j)
                    if (j < kpt) {
                        S[j] *= CHAN ? gg[CHAN ? j : 0] : a;
                        seen = fmaf(S[j], kk[j], seen);
                    }
                seen = sum_near_first<KS>(seen);
                val = sb[tok] * (val - seen);
#pragma unroll
                for (int j = 0; j < DS_KPT; ++j)
                    if (j < kpt) {
                        S[j] = fmaf(kk[j], val, S[j]);
                        acc = fmaf(S[j], qq[j], acc);
                    }
            } else {
#pragma unroll
                for (int j = 0; j < DS_KPT; ++j)
                    if (j < kpt) {
                        S[j] = fmaf(kk[j], val, a * S[j]);
                        if constexpr (MODE != 1) acc = fmaf(S[j], qq[j], acc);
                    }
                if constexpr (MODE == 1) decay_all *= a;
            }
            if (MODE != 1) {
                acc = sum_near_first<KS>(acc);
                if (ks == 0 && live)
                    A.out[(size_t)(first + t0 + tok) * heads * vdim + (size_t)h * vdim + v] = fmaf(skip, raw, acc);
            }
        }
    }
    if (MODE == 2 && chunk != n_chunks - 1) return;
    float* end_at = MODE == 1 ? C_at : S_at;
#pragma unroll
    for (int j = 0; j < DS_KPT; ++j) {
        const int k = ks * kpt + j;
        if (j < kpt && k < dim && live) end_at[(size_t)k * vdim + v] = S[j];
    }
    if (MODE == 1 && tid == 0 && blockIdx.z == 0) A.chunk_decay[(size_t)blockIdx.x * heads + h] = decay_all;
}

// One thread a state entry: the request's state walks over the chunks' ends; chunk_state[chunk] turns from
// "what the chunk makes of a zero state" into "the state the chunk starts from".
__global__ void k_decay_carry(float* __restrict__ chunk_state, const float* __restrict__ chunk_decay,
                              const float* __restrict__ state, const int32_t* __restrict__ seg_len,
                              const int32_t* __restrict__ slot, int n_rows, int heads, int dim, int vdim,
                              int chunk_tokens, int max_chunks) {
    const long long per_head = (long long)dim * vdim, per_row = per_head * heads;
    const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n_rows * per_row) return;
    const int r = (int)(i / per_row);
    const long long e = i - r * per_row;
    const int h = (int)(e / per_head);
    const int n_chunks = (seg_len[r] + chunk_tokens - 1) / chunk_tokens;
    float S = state[(size_t)slot[r] * per_row + e];
    for (int c = 0; c < n_chunks; ++c) {
        float* at = chunk_state + ((size_t)r * max_chunks + c) * per_row + e;
        const bool more = c < n_chunks - 1;
        const float made = more ? *at : 0.f;
        *at = S;
        if (more) S = fmaf(chunk_decay[((size_t)r * max_chunks + c) * heads + h], S, made);
    }
}

// ---------------------------------------------------------------- the delta rule in chunks
// Inside a chunk of DC tokens that starts from the state S0, with g_t the product of the decays from the
// chunk's start up to token t:
//   u_t = b_t (v_t - g_t S0^T k_t - sum_{j<t} (g_t / g_j) (k_t . k_j) u_j)        (I + L) U = diag(b) (V - P),
//   o_t = g_t S0^T q_t + sum_{j<=t} (g_t / g_j) (q_t . k_j) u_j                     O = Qs + M U,
//   S_end = g_last S0 + sum_j (g_last / g_j) k_j u_j^T.
// A first launch makes, for every chunk of every segment and head side by side, T = (I + L)^-1 diag(b) (a lower
// triangle, by forward substitution, a column a thread), M and the logarithms of g (sums of -rate * step, so
// that every ratio is the exponential of a difference and at most one). A second launch walks a segment's
// chunks in order: five small products a chunk on the matrix cores, every sum in an order the sizes alone decide. Tokens past a segment's
// end count as k = q = 0, b = 0 and a decay of one: they change nothing.
#define DC 32                 // tokens a chunk
#define DMAXK 128             // state rows a head at most, in this form

// PLAIN: the recurrence without the delta rule's correction (b = 1, no triangle): M, log g and the steps only.
// With a decay a state row (CHANNEL) the ratios are numbers of a state row too and stand inside the dot products:
//   L_tj = b_t sum_i k_ti k_ji g_ti / g_ji,  M_tj = sum_i q_ti k_ji g_ti / g_ji,
// every ratio the exponential of a difference of logarithms, at most one, so that no decay, however strong, leaves
// float32's range. The first launch then leaves what the walk multiplies, g_t k_t, g_t q_t, (g_last / g_t) k_t and
// g_last, beside T and M: T and M [DC, DC], the first two [DC, DP], the third transposed [DP, DC], g_last [DP], one after
// the other, DP the state's rows filled up to 64 or 128 with zeros.
template <bool PLAIN>
__global__ __launch_bounds__(256) void k_delta_chunk_prepare(const DecayScanArgs A) {
    __shared__ float sk[DC][DMAXK + 1], sq[DC][DMAXK + 1], sL[PLAIN ? 1 : DC][DC + 1], lg[DC], sb[DC];
    const int r = blockIdx.x / A.max_chunks, chunk = blockIdx.x - r * A.max_chunks, h = blockIdx.y;
    const int tid = threadIdx.x, dim = A.dim, heads = A.heads;
    const int n_all = A.seg_len[r];
    if (chunk * DC >= n_all) return;                     // (the whole block)
    const int first = A.seg_start[r] + chunk * DC, n = min(DC, n_all - chunk * DC);
    const int qh = h / A.q_div, kh = h / A.k_div;
    for (int i = tid; i < DC * dim; i += 256) {
        const int t = i / dim, k = i - t * dim;
        const size_t row = (size_t)(first + min(t, n - 1));
        const float kv = A.k[row * A.k_ld + A.k_off + kh * dim + k], qv = A.q[row * A.q_ld + A.q_off + qh * dim + k];
        sk[t][k] = t < n ? kv : 0.f;
        sq[t][k] = t < n ? qv : 0.f;
    }
    if (tid < DC) {
        float la = 0.f, b = 0.f, dt = 1.f;
        if (tid < n) {
            const size_t row = (size_t)(first + tid);
            if (A.decay_const) {
                la = logf(fmaxf(A.decay_const[h], 1e-30f));
            } else {
                dt = ds_softplus(A.step[row * A.step_ld + A.step_off + h] + A.step_bias[h]);
                la = -A.rate[h] * dt;
            }
            if constexpr (!PLAIN) b = ds_sigmoid(A.beta[row * A.beta_ld + A.beta_off + h]);
        }
        lg[tid] = la;
        sb[tid] = b;
        // the steps, for a walk that multiplies its values by them
        A.chunk_decay[((size_t)blockIdx.x * A.heads + h) * (2 * DC) + DC + tid] = dt;
    }
    __syncthreads();
    if (tid == 0) {
        float sum = 0.f;
        for (int t = 0; t < DC; ++t) {
            sum += lg[t];
            lg[t] = sum;
        }
    }
    __syncthreads();
    const size_t at = ((size_t)blockIdx.x * heads + h);
    float* T_out = A.chunk_state + at * (2 * DC * DC);
    float* M_out = T_out + DC * DC;
    for (int i = tid; i < DC * DC; i += 256) {
        const int t = i / DC, j = i - t * DC;
        float kk = 0.f, qk = 0.f;
        if (j <= t) {
            for (int k = 0; k < dim; ++k) {
                if constexpr (!PLAIN) kk = fmaf(sk[t][k], sk[j][k], kk);
                qk = fmaf(sq[t][k], sk[j][k], qk);
            }
            const float w = expf(lg[t] - lg[j]);
            kk *= w * sb[t];
            qk *= w;
        }
        if constexpr (!PLAIN) sL[t][j] = j < t ? kk : 0.f;
        M_out[i] = qk;
    }
    if (tid < DC) A.chunk_decay[at * (2 * DC) + tid] = lg[tid];
    if constexpr (PLAIN) return;
    __syncthreads();
    if (tid < DC) {
        // column tid of (I + L)^-1 by forward substitution, then times b of that column
        float x[DC];
#pragma unroll
        for (int t = 0; t < DC; ++t) {
            float acc = t == tid ? 1.f : 0.f;
#pragma unroll
            for (int j = 0; j < t; ++j) acc = fmaf(-sL[t][j], x[j], acc);
            x[t] = acc;
        }
        const float b = sb[tid];
#pragma unroll
        for (int t = 0; t < DC; ++t) T_out[t * DC + tid] = x[t] * b;
    }
}

__host__ __device__ static inline size_t channel_chunk_floats(int dp) { return 2 * DC * DC + (3 * DC + 1) * (size_t)dp; }
__host__ __device__ static inline int channel_rows(int dim) { return dim <= 64 ? 64 : DMAXK; }

typedef float f32x4 __attribute__((ext_vector_type(4)));

// acc + x y on the matrix cores in float32: x's row lane % 16 and y's column lane % 16, inner numbers 4 i .. of group lane / 16 as
// both sides have them; the result's column is lane % 16, its rows 4 (lane / 16) + i.
__device__ __forceinline__ f32x4 dc_product(const f32x4& x, const f32x4& y, f32x4 acc) {
#pragma unroll
    for (int i = 0; i < 4; ++i) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(x[i], y[i], acc, 0, 0, 0);
    return acc;
}

// Where the entries of L that have a use, below its diagonal, lie by column: each column from the last multiple of four at or above its
// first one, so that a lane reads four tokens at once.
__host__ __device__ constexpr int channel_column(int j) {
    const int q = (j + 1) / 4;                               // the column's rows from 4 q on
    return q == 0 ? j * DC : 3 * DC + 4 * (q - 1) * DC - 8 * q * (q - 1) + (j + 1) % 4 * (DC - 4 * q);
}

// Ratios of decays are exponentials of differences of the logarithms' sums, a pair j <= t and state row at a time, and a pair's sums run over
// the state's rows in order. A thread has two neighbouring j of a t (256 such pieces below the diagonal), whose rows it reads four
// numbers at a time out of LDS; every thread asks for its column of k, q and steps at once, and sums the steps up in registers;
// a solved token of the triangle's inverse goes into all later ones side by side, and the other waves make what is left of the diagonal
// meanwhile. Bound by the pairs' exponentials and reads of LDS and by its bytes, 106 KB a chunk and head. Measured, 4 requests of 1,024
// tokens, 8 heads of 128: 44.5 us; one of 2,048 27.9. (With a pair a lane and numbers read one by one 78.5 and 44.5; ratios split at a
// token between the two, so that they become products of 16 tokens by 16 on the matrix cores, 41.5 and 27.3, and other bits.)
template <int DP>
__global__ __launch_bounds__(256, 3) void k_channel_delta_prepare(const DecayScanArgs A) {
    constexpr int LD = DP + 4, RUNS = 256 / DP, TOK = DC / RUNS;
    __shared__ __attribute__((aligned(16))) float sk[DC * LD], sq[DC * LD], lg[DC * LD], sL[channel_column(DC - 1)];
    __shared__ float sb[DC], total[DP];
    const int r = blockIdx.x / A.max_chunks, chunk = blockIdx.x - r * A.max_chunks, h = blockIdx.y;
    const int tid = threadIdx.x, dim = A.dim, heads = A.heads;
    const int n_all = A.seg_len[r];
    if (chunk * DC >= n_all) return;                     // (the whole block)
    const int first = A.seg_start[r] + chunk * DC, n = min(DC, n_all - chunk * DC);
    const int qh = h / A.q_div, kh = h / A.k_div;
    const float rate = A.rate[h] * 1.44269504088896340736f;      // logarithms to base 2
    const int col = tid % DP, run = tid / DP, t0 = run * TOK;    // this thread's state row, its tokens
    float kv[TOK], qv[TOK], la[TOK];
    {
        const int kc = min(col, dim - 1);
        const float bias = A.step_bias[h * dim + kc];
#pragma unroll
        for (int i = 0; i < TOK; ++i) {                  // (no load under a branch)
            const size_t row = (size_t)(first + min(t0 + i, n - 1));
            kv[i] = A.k[row * A.k_ld + A.k_off + kh * dim + kc];
            qv[i] = A.q[row * A.q_ld + A.q_off + qh * dim + kc];
            la[i] = A.step[row * A.step_ld + A.step_off + h * dim + kc];
        }
        if (tid < DC)
            sb[tid] = tid < n ? ds_sigmoid(A.beta[(size_t)(first + tid) * A.beta_ld + A.beta_off + h]) : 0.f;
#pragma unroll
        for (int i = 0; i < TOK; ++i) {
            const bool on = t0 + i < n && col < dim;
            kv[i] = on ? kv[i] : 0.f;
            qv[i] = on ? qv[i] : 0.f;
            sk[(t0 + i) * LD + col] = kv[i];
            sq[(t0 + i) * LD + col] = qv[i];
            la[i] = on ? -rate * ds_softplus(la[i] + bias) : 0.f;
        }
    }
    // the logarithms add up token after token, so that of two neighbours' sums the difference is one rounding away from the step
    // between them: one run's threads after the other's
    float sum = 0.f;
#pragma unroll
    for (int i = 0; i < RUNS; ++i) {
        if (run == i) {                                  // (whole waves)
            if (i > 0) sum = total[col];
#pragma unroll
            for (int j = 0; j < TOK; ++j) {
                sum += la[j];
                la[j] = sum;
                lg[(t0 + j) * LD + col] = sum;
            }
            total[col] = sum;
        }
        __syncthreads();
    }
    float* T_out = A.chunk_state + ((size_t)blockIdx.x * heads + h) * channel_chunk_floats(DP);
    float* M_out = T_out + DC * DC;
    float* kg_out = M_out + DC * DC;
    float* qg_out = kg_out + DC * DP;
    float* ke_out = qg_out + DC * DP;
    {
        const float last = lg[(DC - 1) * LD + col];
#pragma unroll
        for (int i = 0; i < TOK; ++i) {
            const float g = __builtin_amdgcn_exp2f(la[i]);
            kg_out[(t0 + i) * DP + col] = kv[i] * g;
            qg_out[(t0 + i) * DP + col] = qv[i] * g;
        }
#pragma unroll
        for (int i = 0; i < TOK; i += 4) {
            f32x4 e;
#pragma unroll
            for (int j = 0; j < 4; ++j) e[j] = kv[i + j] * __builtin_amdgcn_exp2f(last - la[i + j]);
            *reinterpret_cast<f32x4*>(&ke_out[col * DC + t0 + i]) = e;
        }
        if (run == 0) ke_out[DC * DP + col] = __builtin_amdgcn_exp2f(last);
    }
    auto four = [&](const float* rows, int t, int k) __attribute__((always_inline)) {
        return *reinterpret_cast<const f32x4*>(rows + t * LD + k);
    };
    {
        // piece tid: tokens t = 2 m - 1 and 2 m have m pieces each (31 has 16), j and j + 1 of a piece; with t odd the last one's j + 1 is t
        int m = (int)((1.0f + sqrtf(1.0f + 4.0f * (float)tid)) * 0.5f);
        if (m * (m - 1) > tid) --m;
        if (m * (m + 1) <= tid) ++m;
        const int at = tid - m * (m - 1), t = 2 * m - 1 + (at >= m ? 1 : 0), j = 2 * (at >= m ? at - m : at);
        float kk[2] = {0.f, 0.f}, qk[2] = {0.f, 0.f};
#pragma unroll 2
        for (int k = 0; k < dim; k += 4) {               // (past dim: zeros)
            const f32x4 lt = four(lg, t, k), kt = four(sk, t, k), qt = four(sq, t, k);
#pragma unroll
            for (int p = 0; p < 2; ++p) {
                const f32x4 lj = four(lg, j + p, k), kj = four(sk, j + p, k);
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const float w = kj[i] * __builtin_amdgcn_exp2f(lt[i] - lj[i]);
                    kk[p] = fmaf(kt[i], w, kk[p]);
                    qk[p] = fmaf(qt[i], w, qk[p]);
                }
            }
        }
        const float b = sb[t];
#pragma unroll
        for (int p = 0; p < 2; ++p) {
            // (column j's place is channel_column(j), rows from 4 ((j + 1) / 4) on)
            if (j + p < t) sL[channel_column(j + p) + t - ((j + p + 1) & ~3)] = kk[p] * b;
            M_out[t * DC + j + p] = qk[p];
        }
    }
    for (int i = tid; i < DC * DC; i += 256)             // above the diagonal
        if (i % DC > i / DC) M_out[i] = 0.f;
    __syncthreads();
    if (tid >= 256 - 16) {                               // the diagonal's even tokens
        const int t = 2 * (tid - (256 - 16));
        float qk = 0.f;
        for (int k = 0; k < dim; k += 4) {
            const f32x4 lt = four(lg, t, k), kt = four(sk, t, k), qt = four(sq, t, k);
#pragma unroll
            for (int i = 0; i < 4; ++i) qk = fmaf(qt[i], kt[i] * __builtin_amdgcn_exp2f(lt[i] - lt[i]), qk);
        }
        M_out[t * DC + t] = qk;
    }
    if (tid < DC) {
        // column tid of (I + L)^-1 by forward substitution, then times b of that column
        float x[DC];
#pragma unroll
        for (int t = 0; t < DC; ++t) x[t] = t == tid ? 1.f : 0.f;
#pragma unroll
        for (int j = 0; j < DC - 1; ++j) {
#pragma unroll
            for (int t = (j + 1) & ~3; t < DC; t += 4) {
                const f32x4 l = *reinterpret_cast<const f32x4*>(&sL[channel_column(j) + t - ((j + 1) & ~3)]);
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    if (t + i > j) x[t + i] = fmaf(-l[i], x[j], x[t + i]);
            }
        }
        const float b = sb[tid];
#pragma unroll
        for (int t = 0; t < DC; ++t) T_out[t * DC + tid] = x[t] * b;
    }
}

// The walk: a segment's chunks in order, a block a (segment, head, run of 16 value columns), every product on the
// matrix cores in float32 (16x16x4). The state stays in the registers of the result layout: a wave holds TPW of the
// state's tiles of 16 rows, wave w tiles w, w + 4, ... In that layout a lane of group g = lane / 16 holds rows 4 g + i
// of its column, and an inner dimension may be walked in any order: taking rows {4 g + i over the groups} as step i makes
// register i the second operand of the next product as it is, and the first operand 16 neighbouring bytes of a row of K
// (or Q, T, M). So nothing is staged and nothing moves between lanes; each wave multiplies its own rows of the state,
// the four partial sums of K S and Q S meet in LDS (two buffers in turn: one barrier a chunk), every wave makes the
// whole of U for its own update, and waves 0 and 1 finish the 16 results each. An operand of the next chunk is asked for
// right behind the last use of this chunk's, into the same registers. Bound by the chunk's chain: 60 to 68 products of 32
// cycles a wave, with the exchange in the middle. Measured, 4 requests of 1,024 tokens, 8 heads of 128, decays a channel: 88.3 us
// with a chunk's 27 requests in a row and the sums read from LDS one by one, 74.4 now (50 with neither requests nor results); one of
// 2,048 158 -> 129. With the first launch, one segment of 2,048, 16 heads: the delta rule, of 128 216 -> 205, of 64 157 -> 154, of 65 (numbers
// one by one) 300 -> 275; plain decays, of 128 157 -> 157, of 64 123 -> 117, of 65 183 -> 164; same bits. Uniform bases with 32-bit offsets in place of whole addresses: 73.9 and 128.8, not kept.
// KIND: a plain decay (U is V itself), the delta rule, the delta rule with decays a channel (whose operands the first
// launch has laid out; the others read K and Q where they lie and scale rows of the results instead). VEC: K's and
// Q's rows can be read in 16-byte pieces.
enum { WALK_DELTA = 0, WALK_PLAIN = 1, WALK_CHANNEL = 2 };

template <int KIND, int TPW>
struct ChunkIn {
    f32x4 k[2][KIND == WALK_PLAIN ? 1 : TPW], q[2][TPW];   // token 16 a + lane % 16, rows 16 T + 4 g + i of the state
    f32x4 e[2][TPW];                                       // token 16 a + 4 g + i, row 16 T + lane % 16
    f32x4 t00, t10, t11, m0, m1;                           // T's three tiles, M's for this wave's results
    f32x4 gl[KIND == WALK_CHANNEL ? TPW : 1];              // the decay over the chunk, rows 16 T + 4 g + i
    f32x4 lg[KIND == WALK_CHANNEL ? 1 : 2], dt[KIND == WALK_PLAIN ? 2 : 1], v[2];     // token 16 a + 4 g + i
    float last;
};

template <int KIND, int TPW, bool VEC>
__global__ __launch_bounds__(256) void k_chunk_walk(const DecayScanArgs A) {
    __shared__ f32x4 part[2][4][4][WAVE];                  // [buffer][wave][P of the two halves, Q of the two][lane]
    const int r = blockIdx.x, h = blockIdx.y;
    const int lane = threadIdx.x & (WAVE - 1), wave = threadIdx.x / WAVE, c = lane & 15, g = lane >> 4;
    const int heads = A.heads, dim = A.dim, vdim = A.vdim;
    const int v = blockIdx.z * 16 + c, vc = min(v, vdim - 1);
    const bool live = v < vdim;
    const int n_all = A.seg_len[r], n_chunks = (n_all + DC - 1) / DC, start = A.seg_start[r];
    const int qh = h / A.q_div, kh = h / A.k_div;
    float* S_at = A.state + (((size_t)A.slot[r] * heads + h) * dim) * vdim;
    f32x4 S[TPW];
#pragma unroll
    for (int j = 0; j < TPW; ++j)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int k = 16 * (wave + 4 * j) + 4 * g + i;
            const float x = S_at[(size_t)min(k, dim - 1) * vdim + vc];
            S[j][i] = (k < dim && live) ? x : 0.f;
        }
    // What is asked for, a piece at a time; every address is clamped and nothing is chosen here (no load may end up under a
    // branch); tokens past the end repeat the last one and meet zeros in U
    struct Place {                                         // of a chunk
        int first, n;
        const float* T;                                    // T, M, and with decays a channel the operands
        const float* decays;
    };
    constexpr int DP = TPW * 64;
    auto place = [&](int chunk) __attribute__((always_inline)) {
        chunk = min(chunk, n_chunks - 1);
        const size_t at = (size_t)(r * A.max_chunks + chunk) * heads + h;
        return Place{start + chunk * DC, min(DC, n_all - chunk * DC),
                     A.chunk_state + at * (KIND == WALK_CHANNEL ? channel_chunk_floats(DP) : (size_t)(2 * DC * DC)),
                     KIND == WALK_CHANNEL ? nullptr : A.chunk_decay + at * (2 * DC)};
    };
    ChunkIn<KIND, TPW> in;
    auto row_of = [&](const float* rows, int ld, const Place& p, int a, int j) __attribute__((always_inline)) {    // K's or Q's piece [a][j]
        const float* x = rows + (size_t)(p.first + min(16 * a + c, p.n - 1)) * ld;
        const int k0 = 16 * (wave + 4 * j) + 4 * g;        // (past dim: other numbers of the row, which meet state rows that stay zero)
        f32x4 v;
        if constexpr (VEC) {                               // rows of whole pieces
            v = *reinterpret_cast<const f32x4*>(x + min(k0, dim - 4));
        } else {
#pragma unroll
            for (int i = 0; i < 4; ++i) v[i] = x[min(k0 + i, dim - 1)];
        }
        return v;
    };
    auto load_k = [&](const Place& p, int a, int j) __attribute__((always_inline)) {
        if constexpr (KIND == WALK_CHANNEL)
            in.k[a][j] = *reinterpret_cast<const f32x4*>(p.T + 2 * DC * DC + (16 * a + c) * DP + 16 * (wave + 4 * j) + 4 * g);
        else if constexpr (KIND == WALK_DELTA)
            in.k[a][j] = row_of(A.k + A.k_off + kh * dim, A.k_ld, p, a, j);
    };
    auto load_q = [&](const Place& p, int a, int j) __attribute__((always_inline)) {
        if constexpr (KIND == WALK_CHANNEL)
            in.q[a][j] = *reinterpret_cast<const f32x4*>(p.T + 2 * DC * DC + DC * DP + (16 * a + c) * DP + 16 * (wave + 4 * j) + 4 * g);
        else
            in.q[a][j] = row_of(A.q + A.q_off + qh * dim, A.q_ld, p, a, j);
    };
    auto load_e = [&](const Place& p, int a, int j) __attribute__((always_inline)) {
        const int k = 16 * (wave + 4 * j) + c;
        if constexpr (KIND == WALK_CHANNEL) {
            in.e[a][j] = *reinterpret_cast<const f32x4*>(p.T + 2 * DC * DC + 2 * DC * DP + k * DC + 16 * a + 4 * g);
        } else {
#pragma unroll
            for (int i = 0; i < 4; ++i)
                in.e[a][j][i] = A.k[(size_t)(p.first + min(16 * a + 4 * g + i, p.n - 1)) * A.k_ld + A.k_off + kh * dim + min(k, dim - 1)];
        }
    };
    auto load_v = [&](const Place& p, int a) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < 4; ++i)
            in.v[a][i] = A.v[(size_t)(p.first + min(16 * a + 4 * g + i, p.n - 1)) * A.v_ld + A.v_off + h * vdim + vc];
    };
    auto load_t = [&](const Place& p) __attribute__((always_inline)) {
        if constexpr (KIND != WALK_PLAIN) {
            in.t00 = *reinterpret_cast<const f32x4*>(p.T + c * DC + 4 * g);
            in.t10 = *reinterpret_cast<const f32x4*>(p.T + (16 + c) * DC + 4 * g);
            in.t11 = *reinterpret_cast<const f32x4*>(p.T + (16 + c) * DC + 16 + 4 * g);
        }
    };
    auto load_m = [&](const Place& p) __attribute__((always_inline)) {
        const float* row = p.T + DC * DC + ((wave & 1) * 16 + c) * DC + 4 * g;
        in.m0 = *reinterpret_cast<const f32x4*>(row);
        in.m1 = *reinterpret_cast<const f32x4*>(row + 16);
    };
    auto load_decays = [&](const Place& p) __attribute__((always_inline)) {
        if constexpr (KIND == WALK_CHANNEL) {
#pragma unroll
            for (int j = 0; j < TPW; ++j)
                in.gl[j] = *reinterpret_cast<const f32x4*>(p.T + 2 * DC * DC + 3 * DC * DP + 16 * (wave + 4 * j) + 4 * g);
        } else {
#pragma unroll
            for (int a = 0; a < 2; ++a) {
                in.lg[a] = *reinterpret_cast<const f32x4*>(p.decays + 16 * a + 4 * g);
                if constexpr (KIND == WALK_PLAIN) in.dt[a] = *reinterpret_cast<const f32x4*>(p.decays + DC + 16 * a + 4 * g);
            }
            in.last = p.decays[DC - 1];
        }
    };
    auto held = []() __attribute__((always_inline)) { __builtin_amdgcn_sched_barrier(0); };
    const float skip = (KIND == WALK_PLAIN && A.skip) ? A.skip[h] : 0.f;
    float* out = A.out + (size_t)h * vdim + v;
    const int out_ld = heads * vdim;
    // Every piece of the next chunk is asked for right behind the last use of this chunk's, into the same registers: a chunk ahead,
    // and one request between two products, so that no wave stands in line to ask
    auto step = [&](int chunk) __attribute__((always_inline)) {
        const int first = start + chunk * DC, n = min(DC, n_all - chunk * DC), buf = chunk & 1;
        const Place next = place(chunk + 1);
        // what the state says of the chunk's keys and queries: this wave's rows of it
        f32x4 p[2], q[2];
#pragma unroll
        for (int a = 0; a < 2; ++a) p[a] = q[a] = f32x4{0.f, 0.f, 0.f, 0.f};
        if constexpr (KIND != WALK_PLAIN) {
#pragma unroll
            for (int j = 0; j < TPW; ++j)
#pragma unroll
                for (int a = 0; a < 2; ++a) {
                    p[a] = dc_product(in.k[a][j], S[j], p[a]);
                    load_k(next, a, j);
                    held();
                }
            part[buf][wave][0][lane] = p[0];
            part[buf][wave][1][lane] = p[1];
        }
#pragma unroll
        for (int j = 0; j < TPW; ++j)
#pragma unroll
            for (int a = 0; a < 2; ++a) {
                q[a] = dc_product(in.q[a][j], S[j], q[a]);
                load_q(next, a, j);
                held();
            }
        part[buf][wave][2][lane] = q[0];
        part[buf][wave][3][lane] = q[1];
        f32x4 g_of[2], u[2], vv[2];
#pragma unroll
        for (int a = 0; a < 2; ++a) {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                vv[a][i] = (16 * a + 4 * g + i < n && live) ? in.v[a][i] : 0.f;
                if constexpr (KIND != WALK_CHANNEL) g_of[a][i] = expf(in.lg[a][i]);
            }
        }
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();                      // (a bare one: the loads in flight are not waited for)
        asm volatile("" ::: "memory");
        if constexpr (KIND == WALK_PLAIN) {
#pragma unroll
            for (int a = 0; a < 2; ++a) u[a] = A.v_times_step ? vv[a] * in.dt[a] : vv[a];
        } else {
            f32x4 res[2], of[2][4];
#pragma unroll
            for (int a = 0; a < 2; ++a)
#pragma unroll
                for (int w = 0; w < 4; ++w) of[a][w] = part[buf][w][a][lane];
            held();                                        // (left alone, the compiler reads and waits one by one)
#pragma unroll
            for (int a = 0; a < 2; ++a) {
                f32x4 sum = of[a][0];
#pragma unroll
                for (int w = 1; w < 4; ++w) sum = sum + of[a][w];
                res[a] = KIND == WALK_CHANNEL ? vv[a] - sum : vv[a] - g_of[a] * sum;
            }
            const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
            u[0] = dc_product(in.t00, res[0], zero);
            load_v(next, 0);
            held();
            u[1] = dc_product(in.t10, res[0], zero);
            load_v(next, 1);
            held();
            u[1] = dc_product(in.t11, res[1], u[1]);
            load_t(next);
            held();
        }
        if constexpr (KIND == WALK_PLAIN) load_v(next, 0), load_v(next, 1);
        if (wave < 2) {                                    // (the whole wave) results of tokens 16 wave .. + 15
            f32x4 of[4];
#pragma unroll
            for (int w = 0; w < 4; ++w) of[w] = part[buf][w][2 + wave][lane];
            held();
            f32x4 o = of[0];
#pragma unroll
            for (int w = 1; w < 4; ++w) o = o + of[w];
            if constexpr (KIND != WALK_CHANNEL) o = o * (wave ? g_of[1] : g_of[0]);
            o = dc_product(in.m0, u[0], o);
            if (wave) o = dc_product(in.m1, u[1], o);
            if (KIND == WALK_PLAIN && skip != 0.f) o = o + skip * (wave ? vv[1] : vv[0]);
            const int t = 16 * wave + 4 * g;
            float* to = out + (size_t)(first + t) * out_ld;
#pragma unroll
            for (int i = 0; i < 4; ++i)
                if (t + i < n && live) to[(size_t)i * out_ld] = o[i];
        }
        load_m(next);
        held();
        // the state behind the chunk
        if constexpr (KIND != WALK_CHANNEL) {
            const float g_last = expf(in.last);
#pragma unroll
            for (int a = 0; a < 2; ++a)
#pragma unroll
                for (int i = 0; i < 4; ++i) u[a][i] *= expf(in.last - in.lg[a][i]);
#pragma unroll
            for (int j = 0; j < TPW; ++j) S[j] = S[j] * g_last;
        } else {
#pragma unroll
            for (int j = 0; j < TPW; ++j) S[j] = S[j] * in.gl[j];
        }
        load_decays(next);
#pragma unroll
        for (int j = 0; j < TPW; ++j)
#pragma unroll
            for (int a = 0; a < 2; ++a) {
                f32x4 e = in.e[a][j];
                if constexpr (KIND != WALK_CHANNEL)
#pragma unroll
                    for (int i = 0; i < 4; ++i) e[i] = 16 * (wave + 4 * j) + c < dim ? e[i] : 0.f;
                S[j] = dc_product(e, u[a], S[j]);
                load_e(next, a, j);
                held();
            }
    };
    {
        const Place p = place(0);                          // (in the order they are used, as in the loop: a wait counts what was asked for later)
#pragma unroll
        for (int j = 0; j < TPW; ++j)
#pragma unroll
            for (int a = 0; a < 2; ++a) load_k(p, a, j), held();
#pragma unroll
        for (int j = 0; j < TPW; ++j)
#pragma unroll
            for (int a = 0; a < 2; ++a) load_q(p, a, j), held();
        load_v(p, 0), held(), load_v(p, 1), held(), load_t(p), held(), load_m(p), held(), load_decays(p), held();
#pragma unroll
        for (int j = 0; j < TPW; ++j)
#pragma unroll
            for (int a = 0; a < 2; ++a) load_e(p, a, j), held();
    }
    for (int chunk = 0; chunk < n_chunks; ++chunk) step(chunk);
#pragma unroll
    for (int j = 0; j < TPW; ++j)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int k = 16 * (wave + 4 * j) + 4 * g + i;
            if (k < dim && live) S_at[(size_t)k * vdim + v] = S[j][i];
        }
}

template <int KIND, bool VEC>
static void launch_walk(const DecayScanArgs& args, int n_rows, hipStream_t s) {
    const dim3 grid(n_rows, args.heads, (args.vdim + 15) / 16);
    if (args.dim <= 64) k_chunk_walk<KIND, 1, VEC><<<grid, 256, 0, s>>>(args);
    else k_chunk_walk<KIND, 2, VEC><<<grid, 256, 0, s>>>(args);
}

extern "C" long long imparo_channel_delta_scratch(int dim) { return (long long)channel_chunk_floats(channel_rows(dim)); }

extern "C" int imparo_channel_delta_scan(const float* q, int q_ld, int q_off, int q_div, const float* k, int k_ld,
                                         int k_off, int k_div, const float* v, int v_ld, int v_off, const float* step,
                                         int step_ld, int step_off, const float* step_bias, const float* rate,
                                         const float* beta, int beta_ld, int beta_off, float* state,
                                         const int32_t* seg_start, const int32_t* seg_len, const int32_t* slot,
                                         float* out, int n_rows, int heads, int dim, int vdim, int chunk_tokens,
                                         int max_chunks, float* scratch, imparo_stream stream) {
    if (!q || !k || !v || !step || !step_bias || !rate || !beta || !state || !seg_start || !seg_len || !slot || !out)
        return IMPARO_BAD_ARGUMENT;
    if (chunk_tokens && (chunk_tokens != DC || dim > DMAXK || max_chunks < 1 || !scratch || ((uintptr_t)scratch & 15)))
        return IMPARO_BAD_ARGUMENT;
    if (n_rows < 0 || heads < 1 || dim < 1 || dim > DS_MAX_DIM || vdim < 1) return IMPARO_BAD_ARGUMENT;
    if (q_div < 1 || k_div < 1 || heads % q_div || heads % k_div) return IMPARO_BAD_ARGUMENT;
    if (q_off < 0 || k_off < 0 || v_off < 0 || q_ld < q_off + heads / q_div * dim || k_ld < k_off + heads / k_div * dim ||
        v_ld < v_off + heads * vdim || step_off < 0 || step_ld < step_off + heads * dim || beta_off < 0 ||
        beta_ld < beta_off + heads)
        return IMPARO_BAD_ARGUMENT;
    if (n_rows == 0) return IMPARO_OK;
    if ((long long)n_rows * (chunk_tokens ? max_chunks : 1) > 0x7fffffffLL) return IMPARO_BAD_ARGUMENT;
    hipStream_t s = (hipStream_t)stream;
    int ks = 1;
    while ((dim + ks - 1) / ks > DS_KPT) ks *= 2;
    const int kpt = (dim + ks - 1) / ks;
    DecayScanArgs args{};
    args.q = q, args.q_ld = q_ld, args.q_off = q_off, args.q_div = q_div;
    args.k = k, args.k_ld = k_ld, args.k_off = k_off, args.k_div = k_div;
    args.v = v, args.v_ld = v_ld, args.v_off = v_off;
    args.step = step, args.step_ld = step_ld, args.step_off = step_off, args.step_bias = step_bias, args.rate = rate;
    args.beta = beta, args.beta_ld = beta_ld, args.beta_off = beta_off;
    args.state = state, args.seg_start = seg_start, args.seg_len = seg_len, args.slot = slot, args.out = out;
    args.heads = heads, args.dim = dim, args.vdim = vdim, args.kpt = kpt;
    args.chunk_tokens = chunk_tokens, args.max_chunks = max_chunks, args.chunk_state = scratch;
    if (chunk_tokens) {
        const dim3 pgrid(n_rows * max_chunks, heads);
        if (channel_rows(dim) == 64) k_channel_delta_prepare<64><<<pgrid, 256, 0, s>>>(args);
        else k_channel_delta_prepare<DMAXK><<<pgrid, 256, 0, s>>>(args);
        launch_walk<WALK_CHANNEL, true>(args, n_rows, s);
        return launch_status();
    }
    int threads = (ks * vdim + WAVE - 1) / WAVE * WAVE;
    threads = threads > DS_MAX_THREADS ? DS_MAX_THREADS : threads;
    const int vb = threads / ks;
    const dim3 grid(n_rows, heads, (vdim + vb - 1) / vb);
#define CDS_WALK(KS)                                                                                                 \
    if (kpt % 4 == 0) k_decay_scan<KS, 0, true, true, true><<<grid, threads, 0, s>>>(args);                         \
    else k_decay_scan<KS, 0, true, false, true><<<grid, threads, 0, s>>>(args)
    switch (ks) {
        case 1: CDS_WALK(1); break;
        case 2: CDS_WALK(2); break;
        case 4: CDS_WALK(4); break;
        case 8: CDS_WALK(8); break;
        case 16: CDS_WALK(16); break;
        case 32: CDS_WALK(32); break;
        default: return IMPARO_BAD_ARGUMENT;
    }
#undef CDS_WALK
    return launch_status();
}

extern "C" int imparo_delta_chunk_tokens() { return DC; }
extern "C" int imparo_delta_chunk_max_dim() { return DMAXK; }

extern "C" int imparo_decay_scan(const float* q, int q_ld, int q_off, int q_div, const float* k, int k_ld, int k_off,
                                 int k_div, const float* v, int v_ld, int v_off, const float* decay_const,
                                 const float* step, int step_ld, int step_off, const float* step_bias,
                                 const float* rate, int v_times_step, const float* beta, int beta_ld, int beta_off,
                                 const float* skip, float* state, const int32_t* seg_start, const int32_t* seg_len,
                                 const int32_t* slot, float* out, int n_rows, int heads, int dim, int vdim,
                                 int chunk_tokens, int max_chunks, float* chunk_state, float* chunk_decay, int silu_in,
                                 imparo_stream stream) {
    if (silu_in && (chunk_tokens || beta)) return IMPARO_BAD_ARGUMENT;
    if (!q || !k || !v || !state || !seg_start || !seg_len || !slot || !out) return IMPARO_BAD_ARGUMENT;
    if (!decay_const && (!step || !step_bias || !rate)) return IMPARO_BAD_ARGUMENT;
    if (v_times_step && decay_const) return IMPARO_BAD_ARGUMENT;
    if (chunk_tokens < 0 || chunk_tokens % DS_TOKENS) return IMPARO_BAD_ARGUMENT;
    if (chunk_tokens && (max_chunks < 1 || !chunk_state || !chunk_decay)) return IMPARO_BAD_ARGUMENT;
    if (chunk_tokens && beta && (chunk_tokens != DC || dim > DMAXK || decay_const)) return IMPARO_BAD_ARGUMENT;
    if (chunk_tokens == DC && (dim > DMAXK || (((uintptr_t)chunk_state | (uintptr_t)chunk_decay) & 15))) return IMPARO_BAD_ARGUMENT;
    if (n_rows < 0 || heads < 1 || dim < 1 || dim > DS_MAX_DIM || vdim < 1) return IMPARO_BAD_ARGUMENT;
    if (q_div < 1 || k_div < 1 || heads % q_div || heads % k_div) return IMPARO_BAD_ARGUMENT;
    if (q_off < 0 || k_off < 0 || v_off < 0 || q_ld < q_off + heads / q_div * dim || k_ld < k_off + heads / k_div * dim ||
        v_ld < v_off + heads * vdim)
        return IMPARO_BAD_ARGUMENT;
    if (step && (step_off < 0 || step_ld < step_off + heads)) return IMPARO_BAD_ARGUMENT;
    if (beta && (beta_off < 0 || beta_ld < beta_off + heads)) return IMPARO_BAD_ARGUMENT;
    if (n_rows == 0) return IMPARO_OK;
    int ks = 1;
    while ((dim + ks - 1) / ks > DS_KPT) ks *= 2;
    const int kpt = (dim + ks - 1) / ks;
    hipStream_t s = (hipStream_t)stream;
    // a block is as many value columns as fill it, in whole waves
    int threads = (ks * vdim + WAVE - 1) / WAVE * WAVE;
    threads = threads > DS_MAX_THREADS ? DS_MAX_THREADS : threads;
    const int vb = threads / ks;
    const int chunks = chunk_tokens ? max_chunks : 1;
    if ((long long)n_rows * chunks > 0x7fffffffLL) return IMPARO_BAD_ARGUMENT;
    const dim3 grid(n_rows * chunks, heads, (vdim + vb - 1) / vb);
    const DecayScanArgs args{q, q_ld, q_off, q_div, k, k_ld, k_off, k_div, v, v_ld, v_off, decay_const,
                             step, step_ld, step_off, step_bias, rate, v_times_step, beta, beta_ld, beta_off, skip,
                             state, seg_start, seg_len, slot, out, heads, dim, vdim, kpt,
                             chunk_tokens, max_chunks, chunk_state, chunk_decay, silu_in};
    if (chunk_tokens == DC && dim <= DMAXK) {
        // the chunks of a segment in order, small products a chunk: chunk_state holds T and M of every chunk,
        // chunk_decay the logarithms of its decays and its steps
        if (beta && (v_times_step || skip)) return IMPARO_BAD_ARGUMENT;
        const dim3 pgrid(n_rows * max_chunks, heads);
        if (beta) k_delta_chunk_prepare<false><<<pgrid, 256, 0, s>>>(args);
        else k_delta_chunk_prepare<true><<<pgrid, 256, 0, s>>>(args);
        const bool vec = dim % 4 == 0 && q_ld % 4 == 0 && q_off % 4 == 0 && k_ld % 4 == 0 && k_off % 4 == 0 &&
                         !(((uintptr_t)q | (uintptr_t)k) & 15);
        if (beta && vec) launch_walk<WALK_DELTA, true>(args, n_rows, s);
        else if (beta) launch_walk<WALK_DELTA, false>(args, n_rows, s);
        else if (vec) launch_walk<WALK_PLAIN, true>(args, n_rows, s);
        else launch_walk<WALK_PLAIN, false>(args, n_rows, s);
        return launch_status();
    }
#define DS_PASS(KS, MODE, DELTA)                                                                                     \
    if (kpt % 4 == 0)                                                                                                \
        k_decay_scan<KS, MODE, DELTA, true><<<grid, threads, 0, s>>>(args);                                         \
    else                                                                                                             \
        k_decay_scan<KS, MODE, DELTA, false><<<grid, threads, 0, s>>>(args)
#define DS_LAUNCH(KS)                                                                                                \
    if (beta) {                                                                                                      \
        DS_PASS(KS, 0, true);                                                                                        \
    } else if (!chunk_tokens) {                                                                                      \
        DS_PASS(KS, 0, false);                                                                                       \
    } else {                                                                                                         \
        DS_PASS(KS, 1, false);                                                                                       \
        const long long entries = (long long)n_rows * heads * dim * vdim;                                            \
        k_decay_carry<<<(unsigned)((entries + 255) / 256), 256, 0, s>>>(chunk_state, chunk_decay, state, seg_len,    \
                                                                        slot, n_rows, heads, dim, vdim,              \
                                                                        chunk_tokens, max_chunks);                   \
        DS_PASS(KS, 2, false);                                                                                       \
    }
    switch (ks) {
        case 1: DS_LAUNCH(1); break;
        case 2: DS_LAUNCH(2); break;
        case 4: DS_LAUNCH(4); break;
        case 8: DS_LAUNCH(8); break;
        case 16: DS_LAUNCH(16); break;
        case 32: DS_LAUNCH(32); break;
        default: return IMPARO_BAD_ARGUMENT;
    }
#undef DS_LAUNCH
#undef DS_PASS
    return launch_status();
}

// ---------------------------------------------------------------- columns before the walk
// SiLU in place on n columns from off on of float32 rows; V neighbouring columns a thread.
template <int V>
__global__ void k_silu_columns(float* __restrict__ rows, int ld, int off, int n, long long total) {
    const int per_row = n / V;
    const long long id = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (id >= total) return;
    const long long t = id / per_row;
    float* p = rows + t * ld + off + (id - t * per_row) * V;
    if constexpr (V == 4) {
        float4 x = *reinterpret_cast<const float4*>(p);
        *reinterpret_cast<float4*>(p) = make_float4(ds_silu(x.x), ds_silu(x.y), ds_silu(x.z), ds_silu(x.w));
    } else {
        *p = ds_silu(*p);
    }
}

extern "C" int imparo_silu_columns(float* rows, int ld, int off, int n, int n_tokens, imparo_stream stream) {
    if (!rows || off < 0 || n < 1 || ld < off + n || n_tokens < 0) return IMPARO_BAD_ARGUMENT;
    if (n_tokens == 0) return IMPARO_OK;
    const bool four = n % 4 == 0 && off % 4 == 0 && ld % 4 == 0 && !((uintptr_t)rows & 15);
    const long long total = (long long)n_tokens * (four ? n / 4 : n);
    const unsigned blocks = (unsigned)((total + 255) / 256);
    if (four) k_silu_columns<4><<<blocks, 256, 0, (hipStream_t)stream>>>(rows, ld, off, n, total);
    else k_silu_columns<1><<<blocks, 256, 0, (hipStream_t)stream>>>(rows, ld, off, n, total);
    return launch_status();
}

// ---------------------------------------------------------------- a head before the walk
// One wave per (token, head) over rows [tokens, ld] float32, in place: head j is the `dim` columns from
// off + j dim. `unit`: the head is divided by sqrt(sum of its squares + unit_eps). Then the first 2 n_freq
// dimensions are rotated by position (pairs (i, i + n_freq), or neighbours (2i, 2i + 1)), then the head is
// multiplied by scale_first (heads below n_first) or scale_rest.
__global__ void k_head_prepare(float* __restrict__ rows, int ld, int off, int n_tokens, int heads, int dim, int unit,
                               float unit_eps, const float* __restrict__ inv_freq, int n_freq, int interleaved,
                               const int32_t* __restrict__ positions, int n_first, float scale_first,
                               float scale_rest) {
    const int lane = threadIdx.x & (WAVE - 1);
    const long long id = (long long)blockIdx.x * (blockDim.x / WAVE) + threadIdx.x / WAVE;
    if (id >= (long long)n_tokens * heads) return;
    const int t = (int)(id / heads), j = (int)(id - (long long)t * heads);
    float* x = rows + (size_t)t * ld + off + (size_t)j * dim;
    float f = j < n_first ? scale_first : scale_rest;
    if (unit) {
        float ss = 0.f;
        for (int i = lane; i < dim; i += WAVE) ss = fmaf(x[i], x[i], ss);
        f *= 1.0f / sqrtf(wave_sum(ss) + unit_eps);
    }
    const int pos = n_freq ? positions[t] : 0;
    for (int i = lane; i < n_freq; i += WAVE) {
        const int ia = interleaved ? 2 * i : i, ib = interleaved ? 2 * i + 1 : i + n_freq;
        float sn, cs;
        rotation_of(pos, inv_freq[i], sn, cs);
        const float a = x[ia], b = x[ib];
        x[ia] = (a * cs - b * sn) * f;
        x[ib] = (b * cs + a * sn) * f;
    }
    for (int i = 2 * n_freq + lane; i < dim; i += WAVE) x[i] *= f;
}

// The sum of squares of numbers that lie four a lane over 16 lanes, Q times (y[q][i]: number 64 q + 4 lane + i, zeros past the end), in
// the order of a wave with a value a lane: a lane's numbers, 64 apart, one after the other, then lanes 32, 16, 8, 4, 2, 1 apart. So the
// kernels in pieces and those that take any length give the same bits.
template <int Q>
__device__ __forceinline__ float squares_of_pieces(const float (&y)[Q][4]) {
    float s[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int q = 0; q < Q; ++q)
#pragma unroll
        for (int i = 0; i < 4; ++i) s[i] = fmaf(y[q][i], y[q][i], s[i]);
    // (the four sums go on in a quarter of the lanes each: seven moves between lanes and not sixteen)
    const bool b8 = threadIdx.x & 8, b4 = threadIdx.x & 4;
    const float first = (b8 ? s[2] : s[0]) + lane_xor<8>(b8 ? s[0] : s[2]);
    const float second = (b8 ? s[3] : s[1]) + lane_xor<8>(b8 ? s[1] : s[3]);
    float sum = (b4 ? second : first) + lane_xor<4>(b4 ? first : second);
    sum += lane_xor<2>(sum);
    sum += lane_xor<1>(sum);
    sum += lane_xor<8>(sum);
    sum += lane_xor<4>(sum);
    return sum;
}

// The same without a rotation, for heads of whole 16-byte pieces: 16 lanes a head, four heads a wave, which keep it in registers where
// it was read twice, a value a lane at a time. Bound by its bytes. 3,328 rows of 8 heads as unit vectors, us before and so: of 128 9.8 and
// 5.5, of 64 7.5 and 4.0, of 256 16.0 and 8.1. (In 32 lanes a head with a sum of its own order 5.6, 4.8 and, in 64, 11.5.)
template <int Q>
__global__ __launch_bounds__(256) void k_head_prepare_four(float* __restrict__ rows, int ld, int off, int n_tokens, int heads, int dim,
                                                           int unit, float unit_eps, int n_first, float scale_first, float scale_rest) {
    const int lane = threadIdx.x % 16;
    const long long all = (long long)n_tokens * heads, at = (long long)blockIdx.x * 16 + threadIdx.x / 16;
    const long long id = at < all ? at : all - 1;            // (no lane leaves before the sums)
    const int t = (int)(id / heads), j = (int)(id - (long long)t * heads);
    float* x = rows + (size_t)t * ld + off + (size_t)j * dim;
    float y[Q][4];
#pragma unroll
    for (int q = 0; q < Q; ++q) {
        const int i = 64 * q + 4 * lane;
        const float4 v = *reinterpret_cast<const float4*>(x + min(i, dim - 4));
        const bool on = i < dim;
        y[q][0] = on ? v.x : 0.f, y[q][1] = on ? v.y : 0.f, y[q][2] = on ? v.z : 0.f, y[q][3] = on ? v.w : 0.f;
    }
    float f = j < n_first ? scale_first : scale_rest;
    if (unit) f *= 1.0f / sqrtf(squares_of_pieces<Q>(y) + unit_eps);
    if (at >= all) return;
#pragma unroll
    for (int q = 0; q < Q; ++q) {
        const int i = 64 * q + 4 * lane;
        if (i < dim) *reinterpret_cast<float4*>(x + i) = make_float4(y[q][0] * f, y[q][1] * f, y[q][2] * f, y[q][3] * f);
    }
}

extern "C" int imparo_head_prepare(float* rows, int ld, int off, int n_tokens, int heads, int dim, int unit,
                                   float unit_eps, const float* inv_freq, int n_freq, int interleaved,
                                   const int32_t* positions, int n_first, float scale_first, float scale_rest,
                                   imparo_stream stream) {
    if (!rows || n_tokens < 0 || heads < 1 || dim < 1 || off < 0 || ld < off + heads * dim) return IMPARO_BAD_ARGUMENT;
    if (n_freq < 0 || 2 * n_freq > dim || (n_freq && (!inv_freq || !positions))) return IMPARO_BAD_ARGUMENT;
    if (n_tokens == 0) return IMPARO_OK;
    const long long waves = (long long)n_tokens * heads;
    if (!n_freq && dim % 4 == 0 && dim <= 256 && ld % 4 == 0 && off % 4 == 0 && !((uintptr_t)rows & 15)) {
#define HEAD_FOUR(Q)                                                                                                 \
    k_head_prepare_four<Q><<<(unsigned)((waves + 15) / 16), 256, 0, (hipStream_t)stream>>>(rows, ld, off, n_tokens, heads, dim, unit, \
                                                                                         unit_eps, n_first, scale_first, scale_rest)
        if (dim <= 64) HEAD_FOUR(1);
        else if (dim <= 128) HEAD_FOUR(2);
        else HEAD_FOUR(4);
#undef HEAD_FOUR
        return launch_status();
    }
    k_head_prepare<<<(unsigned)((waves + 3) / 4), 4 * WAVE, 0, (hipStream_t)stream>>>(
        rows, ld, off, n_tokens, heads, dim, unit, unit_eps, inv_freq, n_freq, interleaved, positions, n_first,
        scale_first, scale_rest);
    return launch_status();
}

// ---------------------------------------------------------------- the heads behind the walk
// out[t, c] for a row of `width` values in `groups` equal parts: with y = x[t, c] and g = silu(gate[t, c]) (gate_act
// 1: its sigmoid),
//   gate_first: (y g) / rms_part(y g) * w[c];   otherwise: y / rms_part(y) * w[c] * g     (w null: 1).
// A wave takes a part; for long parts a block does, with the part in registers (PER values a thread, every load
// asked for before any is used, the gate's activation taken once).
template <typename TOut>
__global__ __launch_bounds__(256) void k_gated_group_norm(const float* __restrict__ x, const float* __restrict__ gate,
                                                          int gate_ld, int gate_off, const float* __restrict__ w,
                                                          TOut* __restrict__ out, int n_tokens, int width, int groups,
                                                          float eps, int gate_first, int gate_act) {
    const int part = width / groups;
    const long long id = (long long)blockIdx.x * (blockDim.x / WAVE) + threadIdx.x / WAVE;
    const int first = threadIdx.x & (WAVE - 1);
    if (id >= (long long)n_tokens * groups) return;
    const int t = (int)(id / groups), g = (int)(id - (long long)t * groups);
    const float* xr = x + (size_t)t * width + (size_t)g * part;
    const float* gr = gate ? gate + (size_t)t * gate_ld + gate_off + (size_t)g * part : nullptr;
    float ss = 0.f;
#pragma unroll 4
    for (int i = first; i < part; i += WAVE) {
        float y = xr[i];
        if (gate_first && gr) y *= ds_gate(gr[i], gate_act);
        ss = fmaf(y, y, ss);
    }
    ss = wave_sum(ss);
    const float rs = 1.0f / sqrtf(ss / (float)part + eps);
#pragma unroll 4
    for (int i = first; i < part; i += WAVE) {
        float y = xr[i];
        const float gv = gr ? ds_gate(gr[i], gate_act) : 1.f;
        if (gate_first) y *= gv;
        y = y * rs * (w ? w[(size_t)g * part + i] : 1.f);
        if (!gate_first) y *= gv;
        store_f32<TOut>(out, (size_t)t * width + (size_t)g * part + i, y);
    }
}

// A short part of whole 16-byte pieces, Q of them a lane at most: 16 lanes a part, everything asked for at once and kept, where a wave
// asked value by value and read the part and its gate again behind the sum. Bound by its bytes. 3,328 rows of 8 parts of 64, bfloat16 out,
// 9.4 -> 6.5 us.
template <typename TOut, int Q>
__global__ __launch_bounds__(256) void k_gated_group_norm_four(const float* __restrict__ x, const float* __restrict__ gate,
                                                               int gate_ld, int gate_off, const float* __restrict__ w,
                                                               TOut* __restrict__ out, int n_tokens, int width, int groups,
                                                               float eps, int gate_first, int gate_act) {
    const int lane = threadIdx.x % 16, part = width / groups;
    const long long all = (long long)n_tokens * groups, at = (long long)blockIdx.x * 16 + threadIdx.x / 16;
    const long long id = at < all ? at : all - 1;            // (no lane leaves before the sum)
    const int t = (int)(id / groups), g = (int)(id - (long long)t * groups);
    const float* xr = x + (size_t)t * width + (size_t)g * part;
    const float* gr = gate ? gate + (size_t)t * gate_ld + gate_off + (size_t)g * part : nullptr;
    float y[Q][4], gv[Q][4], wv[Q][4];
#pragma unroll
    for (int q = 0; q < Q; ++q) {
        const int i = min(64 * q + 4 * lane, part - 4);
        const float4 a = *reinterpret_cast<const float4*>(xr + i);
        const float4 one = make_float4(1.f, 1.f, 1.f, 1.f);
        const float4 b = gr ? *reinterpret_cast<const float4*>(gr + i) : one;
        const float4 c = w ? *reinterpret_cast<const float4*>(w + (size_t)g * part + i) : one;
        y[q][0] = a.x, y[q][1] = a.y, y[q][2] = a.z, y[q][3] = a.w;
        gv[q][0] = b.x, gv[q][1] = b.y, gv[q][2] = b.z, gv[q][3] = b.w;
        wv[q][0] = c.x, wv[q][1] = c.y, wv[q][2] = c.z, wv[q][3] = c.w;
    }
#pragma unroll
    for (int q = 0; q < Q; ++q)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            gv[q][i] = gr ? ds_gate(gv[q][i], gate_act) : 1.f;
            if (gate_first) y[q][i] *= gv[q][i];
            if (64 * q + 4 * lane >= part) y[q][i] = 0.f;
        }
    const float rs = 1.0f / sqrtf(squares_of_pieces<Q>(y) / (float)part + eps);
#pragma unroll
    for (int q = 0; q < Q; ++q) {
        const int i = 64 * q + 4 * lane;
        float v[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            v[k] = y[q][k] * rs * wv[q][k];
            if (!gate_first) v[k] *= gv[q][k];
        }
        if (i >= part || at >= all) continue;
        TOut* to = out + (size_t)t * width + (size_t)g * part + i;
        if constexpr (sizeof(TOut) == 4)
            *reinterpret_cast<float4*>(to) = make_float4(v[0], v[1], v[2], v[3]);
        else
            *reinterpret_cast<uint2*>(to) = make_uint2(f32x2_to_bf16x2(v[0], v[1]), f32x2_to_bf16x2(v[2], v[3]));
    }
}

// A longer part of up to 64 PER numbers: a wave a part and a value a lane, as below, but everything asked for at once and kept, and a gate's
// activation made once. 3,328 rows of 8 parts, bfloat16 out, of 128 13.7 -> 10.1 us, of 256 19.4 -> 15.1, of 512 33.9 -> 24.6 (16 bytes a
// lane and 64 lanes a part, whose sum has to change lanes in mid-chain, 10.4, 18.3 and 33.6).
template <typename TOut, int PER>
__global__ __launch_bounds__(256) void k_gated_group_norm_kept(const float* __restrict__ x, const float* __restrict__ gate,
                                                               int gate_ld, int gate_off, const float* __restrict__ w,
                                                               TOut* __restrict__ out, int n_tokens, int width, int groups,
                                                               float eps, int gate_first, int gate_act) {
    const int lane = threadIdx.x & (WAVE - 1), part = width / groups;
    const long long id = (long long)blockIdx.x * (256 / WAVE) + threadIdx.x / WAVE;
    if (id >= (long long)n_tokens * groups) return;          // (whole waves)
    const int t = (int)(id / groups), g = (int)(id - (long long)t * groups);
    const float* xr = x + (size_t)t * width + (size_t)g * part;
    const float* gr = gate ? gate + (size_t)t * gate_ld + gate_off + (size_t)g * part : nullptr;
    float y[PER], gv[PER], wv[PER];
#pragma unroll
    for (int p = 0; p < PER; ++p) {
        const int i = min(lane + 64 * p, part - 1);
        y[p] = xr[i];
        gv[p] = gr ? gr[i] : 1.f;
        wv[p] = w ? w[(size_t)g * part + i] : 1.f;
    }
    float ss = 0.f;
#pragma unroll
    for (int p = 0; p < PER; ++p) {
        if (gr) gv[p] = ds_gate(gv[p], gate_act);
        if (gate_first) y[p] *= gv[p];
        const float mine = lane + 64 * p < part ? y[p] : 0.f;
        ss = fmaf(mine, mine, ss);
    }
    const float rs = 1.0f / sqrtf(wave_sum(ss) / (float)part + eps);
#pragma unroll
    for (int p = 0; p < PER; ++p) {
        const int i = lane + 64 * p;
        float v = y[p] * rs * wv[p];
        if (!gate_first) v *= gv[p];
        if (i < part) store_f32<TOut>(out, (size_t)t * width + (size_t)g * part + i, v);
    }
}

template <typename TOut, int PER>
__global__ __launch_bounds__(256) void k_gated_group_norm_block(const float* __restrict__ x, const float* __restrict__ gate,
                                                                int gate_ld, int gate_off, const float* __restrict__ w,
                                                                TOut* __restrict__ out, int width, int groups, float eps,
                                                                int gate_first, int gate_act) {
    __shared__ float scratch[16];
    const int part = width / groups;
    const int t = blockIdx.x / groups, g = blockIdx.x - t * groups;
    const float* xr = x + (size_t)t * width + (size_t)g * part;
    const float* gr = gate ? gate + (size_t)t * gate_ld + gate_off + (size_t)g * part : nullptr;
    float y[PER], gv[PER], wv[PER];
#pragma unroll
    for (int j = 0; j < PER; ++j) {
        const int i = min((int)threadIdx.x + j * 256, part - 1);
        y[j] = xr[i];
        gv[j] = gr ? gr[i] : 0.f;
        wv[j] = w ? w[(size_t)g * part + i] : 1.f;
    }
    float ss = 0.f;
#pragma unroll
    for (int j = 0; j < PER; ++j) {
        gv[j] = gr ? ds_gate(gv[j], gate_act) : 1.f;
        if (gate_first) y[j] *= gv[j];
        if ((int)threadIdx.x + j * 256 < part) ss = fmaf(y[j], y[j], ss);
    }
    const float rs = 1.0f / sqrtf(block_sum(ss, scratch) / (float)part + eps);
#pragma unroll
    for (int j = 0; j < PER; ++j) {
        const int i = threadIdx.x + j * 256;
        float v = y[j] * rs * wv[j];
        if (!gate_first) v *= gv[j];
        if (i < part) store_f32<TOut>(out, (size_t)t * width + (size_t)g * part + i, v);
    }
}

extern "C" int imparo_gated_group_norm(const float* x, const float* gate, int gate_ld, int gate_off, const float* w,
                                       void* out, int out_dtype, int n_tokens, int width, int groups, float eps,
                                       int gate_first, int gate_act, imparo_stream stream) {
    if (gate_act != 0 && gate_act != 1) return IMPARO_BAD_ARGUMENT;
    if (!x || !out || n_tokens < 0 || width < 1 || groups < 1 || width % groups) return IMPARO_BAD_ARGUMENT;
    if (gate && (gate_off < 0 || gate_ld < gate_off + width)) return IMPARO_BAD_ARGUMENT;
    if (out_dtype != IMPARO_F32 && out_dtype != IMPARO_BF16) return IMPARO_BAD_ARGUMENT;
    if (n_tokens == 0) return IMPARO_OK;
    hipStream_t s = (hipStream_t)stream;
    const long long parts = (long long)n_tokens * groups;
    if (parts > 0x7fffffffLL) return IMPARO_BAD_ARGUMENT;
    const int part = width / groups;
    if (part > 512 && part <= 256 * 64) {
#define GGN_BLOCK(T, PER)                                                                                            \
    k_gated_group_norm_block<T, PER><<<(unsigned)parts, 256, 0, s>>>(x, gate, gate_ld, gate_off, w, (T*)out, width, \
                                                                     groups, eps, gate_first, gate_act)
#define GGN_PER(T)                                                                                                   \
    if (part <= 256 * 4) GGN_BLOCK(T, 4);                                                                            \
    else if (part <= 256 * 8) GGN_BLOCK(T, 8);                                                                       \
    else if (part <= 256 * 16) GGN_BLOCK(T, 16);                                                                     \
    else if (part <= 256 * 32) GGN_BLOCK(T, 32);                                                                     \
    else GGN_BLOCK(T, 64)
        if (out_dtype == IMPARO_BF16) { GGN_PER(bf16_t); } else { GGN_PER(float); }
#undef GGN_PER
#undef GGN_BLOCK
        return launch_status();
    }
    if (part % 4 == 0 && part <= 512 && gate_ld % 4 == 0 && gate_off % 4 == 0 &&
        !(((uintptr_t)x | (uintptr_t)gate | (uintptr_t)w | (uintptr_t)out) & 15)) {
        // 16 lanes a part need fewer waves but go through a lane's numbers one after the other: for short parts, longer ones where there
        // are very many. us, 16 lanes | a wave a part: 512 parts of 64 3.0 | 2.4; 106,000 of 96 26.1 | 32.8, of 128 31.9 |
        // 35.3, 8,192 of 96 4.8 | 4.4, 26,624 9.5 | 10.0, of 128 11.2 | 10.3.
        const bool few = part > 32 && parts < 4096, many = parts >= (part <= 96 ? 16384 : 65536);
#define GGN_FOUR(T, Q)                                                                                               \
    k_gated_group_norm_four<T, Q><<<(unsigned)((parts + 15) / 16), 256, 0, s>>>(x, gate, gate_ld, gate_off, w, (T*)out, n_tokens, width, \
                                                                              groups, eps, gate_first, gate_act)
#define GGN_KEPT(T, PER)                                                                                             \
    k_gated_group_norm_kept<T, PER><<<(unsigned)((parts + 3) / 4), 256, 0, s>>>(x, gate, gate_ld, gate_off, w, (T*)out, n_tokens, width, \
                                                                              groups, eps, gate_first, gate_act)
#define GGN_FIT(T)                                                                                                   \
    if (part <= 64 && !few) GGN_FOUR(T, 1);                                                                          \
    else if (part <= 64) GGN_KEPT(T, 1);                                                                             \
    else if (part <= 128 && !many) GGN_KEPT(T, 2);                                                                   \
    else if (part <= 128) GGN_FOUR(T, 2);                                                                            \
    else if (part <= 256) GGN_KEPT(T, 4);                                                                            \
    else GGN_KEPT(T, 8)
        if (out_dtype == IMPARO_BF16) { GGN_FIT(bf16_t); } else { GGN_FIT(float); }
#undef GGN_FIT
#undef GGN_KEPT
#undef GGN_FOUR
        return launch_status();
    }
    const unsigned blocks = (unsigned)((parts + 3) / 4);
    if (out_dtype == IMPARO_BF16)
        k_gated_group_norm<bf16_t><<<blocks, 256, 0, s>>>(x, gate, gate_ld, gate_off, w, (bf16_t*)out, n_tokens, width,
                                                          groups, eps, gate_first, gate_act);
    else
        k_gated_group_norm<float><<<blocks, 256, 0, s>>>(x, gate, gate_ld, gate_off, w, (float*)out, n_tokens, width,
                                                         groups, eps, gate_first, gate_act);
    return launch_status();
}

// ---------------------------------------------------------------- sums of mixers and of experts
// out[t, c] (+)= sum_i f_i * rms_norm(a_i[t])[c] * w_i[c] over up to two inputs (each maybe in slices that
// are added in order first): the results of mixers that run side by side, each normed over the row.
// PER: values of the row a thread keeps in registers (256 threads x PER cover the width): every slice is read
// once, and the loads of a slice are asked for together.
template <int PER>
__global__ __launch_bounds__(256) void k_normed_sum(const float* __restrict__ a, int a_slices, const float* __restrict__ wa,
                                                    const float* __restrict__ b, int b_slices, const float* __restrict__ wb,
                                                    float* __restrict__ out, int n_tokens, int width, float eps,
                                                    float factor) {
    __shared__ float scratch[16];
    const int t = blockIdx.x;
    const size_t stride = (size_t)n_tokens * width, row = (size_t)t * width;
    float ya[PER], yb[PER];
#pragma unroll
    for (int j = 0; j < PER; ++j) ya[j] = yb[j] = 0.f;
    for (int s = 0; s < a_slices; ++s)
#pragma unroll
        for (int j = 0; j < PER; ++j) ya[j] += a[s * stride + row + min((int)threadIdx.x + j * 256, width - 1)];
    for (int s = 0; s < b_slices; ++s)
#pragma unroll
        for (int j = 0; j < PER; ++j) yb[j] += b[s * stride + row + min((int)threadIdx.x + j * 256, width - 1)];
    float ssa = 0.f, ssb = 0.f;
#pragma unroll
    for (int j = 0; j < PER; ++j)
        if ((int)threadIdx.x + j * 256 < width) {
            ssa = fmaf(ya[j], ya[j], ssa);
            ssb = fmaf(yb[j], yb[j], ssb);
        }
    const float ra = 1.0f / sqrtf(block_sum(ssa, scratch) / (float)width + eps);
    const float rb = 1.0f / sqrtf(block_sum(ssb, scratch) / (float)width + eps);
#pragma unroll
    for (int j = 0; j < PER; ++j) {
        const int i = threadIdx.x + j * 256;
        if (i < width) out[row + i] = factor * (ya[j] * ra * wa[i] + yb[j] * rb * wb[i]);
    }
}

extern "C" int imparo_normed_sum(const float* a, int a_slices, const float* wa, const float* b, int b_slices,
                                 const float* wb, float* out, int n_tokens, int width, float eps, float factor,
                                 imparo_stream stream) {
    if (!a || !b || !wa || !wb || !out || a_slices < 1 || b_slices < 1 || n_tokens < 0 || width < 1 || width > 16384)
        return IMPARO_BAD_ARGUMENT;
    if (n_tokens == 0) return IMPARO_OK;
    hipStream_t s = (hipStream_t)stream;
#define NSUM(PER) k_normed_sum<PER><<<n_tokens, 256, 0, s>>>(a, a_slices, wa, b, b_slices, wb, out, n_tokens, width, eps, factor)
    const int per = (width + 255) / 256;
    if (per <= 1) NSUM(1);
    else if (per <= 2) NSUM(2);
    else if (per <= 4) NSUM(4);
    else if (per <= 8) NSUM(8);
    else if (per <= 16) NSUM(16);
    else if (per <= 32) NSUM(32);
    else NSUM(64);
#undef NSUM
    return launch_status();
}

// out[t, c] += sigmoid(z[t, z_col]) * sum over slices of y[s, t, c]: an expert that every token uses, weighed by
// one gate a token.
__global__ void k_gated_row_add(float* __restrict__ out, const float* __restrict__ y, int y_slices,
                                const float* __restrict__ z, int z_ld, int z_col, int n_tokens, int width) {
    const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= (long long)n_tokens * width) return;
    const long long t = i / width;
    float s = 0.f;
    for (int k = 0; k < y_slices; ++k) s += y[(size_t)k * n_tokens * width + i];
    out[i] = fmaf(ds_sigmoid(z[t * z_ld + z_col]), s, out[i]);
}

extern "C" int imparo_gated_row_add(float* out, const float* y, int y_slices, const float* z, int z_ld, int z_col,
                                    int n_tokens, int width, imparo_stream stream) {
    if (!out || !y || !z || y_slices < 1 || z_col < 0 || z_ld <= z_col || n_tokens < 0 || width < 1)
        return IMPARO_BAD_ARGUMENT;
    const long long n = (long long)n_tokens * width;
    if (n == 0) return IMPARO_OK;
    k_gated_row_add<<<(unsigned)((n + 255) / 256), 256, 0, (hipStream_t)stream>>>(out, y, y_slices, z, z_ld, z_col,
                                                                                n_tokens, width);
    return launch_status();
}

// ---------------------------------------------------------------- one token of the channel delta rule, whole
// A decode step of the delta rule with a decay a channel, from the projections' rows to the rows the output projection
// reads: conv and SiLU of q, k and v with the shift of their history, unit length, the decays, the state's step, and the
// norm and gate of the heads behind it, one launch where there were four (the conv, the heads' preparation, the walk, the
// norm: 19.7 us in a step of 4 requests with 8 heads, each launch a trip through memory to the next; now 9.3). Heads of 128 by
// 128 and up to four taps. A block has one request's query/key head and the PER heads that share it, so that no other block
// reads the history it shifts; its 1,024 threads keep a piece of four rows by four columns of each head's state, asked for
// before anything else. Bound by the state's trips to memory and five meetings of the block between them.
#define CDS_DIM 128
#define CDS_MAX_TAPS 4
struct ChannelStepArgs {
    const float* rows; int ld, beta_off;         // q | k | v | .., b from beta_off on
    const float* steps; int steps_ld, gate_off;  // the decays' raw steps, the gate from gate_off on
    const float* conv_w; float* conv; int taps;  // [channels, taps], [slots, taps - 1, channels]
    const float* step_bias; const float* rate;   // [heads * dim], [heads]
    float* state;                                // [slots, heads, dim, vdim]
    const int32_t* slot;
    const float* norm;                           // [heads * vdim]
    int heads, kv_heads;
    float unit_eps, q_scale, eps;
};

__device__ __forceinline__ float cds_halves(float v) {       // the sum of the two lanes 32 apart
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

template <typename TOut, int PER>
__global__ __launch_bounds__(1024) void k_channel_delta_step(const ChannelStepArgs A, TOut* __restrict__ out) {
    constexpr int D = CDS_DIM, WAVES = 16;
    __shared__ __attribute__((aligned(16))) float sq[D], sk[D], sv[PER][D], sg[PER][D], su[PER][D];
    __shared__ __attribute__((aligned(16))) float red[PER][WAVES][D];
    __shared__ float squares[4], beta[PER], part[2 * PER];
    const int r = blockIdx.x, kh = blockIdx.y, h0 = kh * PER;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int c4 = (tid & 31) * 4, k0 = (tid >> 5) * 4;      // this thread's columns and rows of a head's state
    const int H = A.heads, Hk = A.kv_heads, channels = 2 * Hk * D + H * D;
    const size_t at = A.slot[r];
    float* S_at = A.state + (at * H + h0) * (D * D);
    float4 S[PER][4];
#pragma unroll
    for (int p = 0; p < PER; ++p)
#pragma unroll
        for (int j = 0; j < 4; ++j) S[p][j] = *reinterpret_cast<const float4*>(S_at + ((size_t)p * D + k0 + j) * D + c4);
    const float* row = A.rows + (size_t)r * A.ld;
    const float* step = A.steps + (size_t)r * A.steps_ld;
    const bool finishes = tid < PER * D;                     // one output
    const float gate = finishes ? step[A.gate_off + h0 * D + tid] : 0.f, norm = finishes ? A.norm[h0 * D + tid] : 0.f;
    if (tid < (2 + PER) * D) {                               // one channel: 128 of q, 128 of k, the heads' values
        const int ch = tid < D ? kh * D + tid : tid < 2 * D ? Hk * D + kh * D + (tid - D) : 2 * Hk * D + h0 * D + (tid - 2 * D);
        const int history = A.taps - 1;
        float* hist = A.conv + at * (size_t)history * channels + ch;
        float old[CDS_MAX_TAPS - 1], w[CDS_MAX_TAPS];
#pragma unroll
        for (int i = 0; i < CDS_MAX_TAPS - 1; ++i) old[i] = i < history ? hist[(size_t)i * channels] : 0.f;
#pragma unroll
        for (int i = 0; i < CDS_MAX_TAPS; ++i) w[i] = i < A.taps ? A.conv_w[(size_t)ch * A.taps + i] : 0.f;
        const float now = row[ch];
        float acc = 0.f, last = w[0];
#pragma unroll
        for (int i = 0; i < CDS_MAX_TAPS - 1; ++i) {         // (what lies past the history is zero)
            acc = fmaf(i < history ? w[i] : 0.f, old[i], acc);
            last = i + 1 == history ? w[i + 1] : last;
        }
        acc = fmaf(last, now, acc);
#pragma unroll
        for (int i = 0; i < CDS_MAX_TAPS - 1; ++i)
            if (i < history) hist[(size_t)i * channels] = i + 1 < history ? old[i + 1 < CDS_MAX_TAPS - 1 ? i + 1 : 0] : now;
        const float y = ds_silu(acc);
        if (tid < 2 * D) {
            (tid < D ? sq : sk)[tid & (D - 1)] = y;
            const float ss = wave_sum(y * y);                // (whole waves: a head's 128 channels are two)
            if (lane == 0) squares[wave] = ss;
        } else {
            sv[(tid - 2 * D) / D][(tid - 2 * D) & (D - 1)] = y;
        }
    } else if (tid >= 1024 - PER * D) {                      // one decay a state row (other waves than the channels')
        const int i = tid - (1024 - PER * D);
        sg[i / D][i & (D - 1)] = expf(-A.rate[h0 + i / D] * ds_softplus(step[h0 * D + i] + A.step_bias[h0 * D + i]));
        if (i < PER) beta[i] = ds_sigmoid(row[A.beta_off + h0 + i]);
    }
    __syncthreads();
    const float fq = A.q_scale * (1.0f / sqrtf(squares[0] + squares[1] + A.unit_eps));
    const float fk = 1.0f / sqrtf(squares[2] + squares[3] + A.unit_eps);
    float4 kk = *reinterpret_cast<const float4*>(&sk[k0]), qq = *reinterpret_cast<const float4*>(&sq[k0]);
    const float kj[4] = {kk.x * fk, kk.y * fk, kk.z * fk, kk.w * fk}, qj[4] = {qq.x * fq, qq.y * fq, qq.z * fq, qq.w * fq};
    // a sum over the state's rows: four a thread, two threads a wave, the waves' through LDS and in pairs (one after the other
    // they were further from 64 bits than the walk: outputs 1.63e-7, the walk 1.62e-7, so 1.54e-7)
    auto leave = [&](int p, const float (&v)[4]) __attribute__((always_inline)) {
        const float4 s = make_float4(cds_halves(v[0]), cds_halves(v[1]), cds_halves(v[2]), cds_halves(v[3]));
        if (lane < 32) *reinterpret_cast<float4*>(&red[p][wave][c4]) = s;
    };
    auto gather = [&]() __attribute__((always_inline)) {     // column tid % 128 of head tid / 128
        float v[WAVES];
#pragma unroll
        for (int w = 0; w < WAVES; ++w) v[w] = red[tid / D][w][tid & (D - 1)];
#pragma unroll
        for (int half = WAVES / 2; half > 0; half /= 2)
#pragma unroll
            for (int w = 0; w < half; ++w) v[w] += v[w + half];
        return v[0];
    };
#pragma unroll
    for (int p = 0; p < PER; ++p) {
        const float4 g4 = *reinterpret_cast<const float4*>(&sg[p][k0]);
        const float g[4] = {g4.x, g4.y, g4.z, g4.w};
        float seen[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            S[p][j] = make_float4(S[p][j].x * g[j], S[p][j].y * g[j], S[p][j].z * g[j], S[p][j].w * g[j]);
            seen[0] = fmaf(S[p][j].x, kj[j], seen[0]);
            seen[1] = fmaf(S[p][j].y, kj[j], seen[1]);
            seen[2] = fmaf(S[p][j].z, kj[j], seen[2]);
            seen[3] = fmaf(S[p][j].w, kj[j], seen[3]);
        }
        leave(p, seen);
    }
    __syncthreads();
    if (finishes) su[tid / D][tid & (D - 1)] = beta[tid / D] * (sv[tid / D][tid & (D - 1)] - gather());
    __syncthreads();
#pragma unroll
    for (int p = 0; p < PER; ++p) {
        const float4 u = *reinterpret_cast<const float4*>(&su[p][c4]);
        float o[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            S[p][j] = make_float4(fmaf(kj[j], u.x, S[p][j].x), fmaf(kj[j], u.y, S[p][j].y), fmaf(kj[j], u.z, S[p][j].z),
                                  fmaf(kj[j], u.w, S[p][j].w));
            o[0] = fmaf(S[p][j].x, qj[j], o[0]);
            o[1] = fmaf(S[p][j].y, qj[j], o[1]);
            o[2] = fmaf(S[p][j].z, qj[j], o[2]);
            o[3] = fmaf(S[p][j].w, qj[j], o[3]);
            *reinterpret_cast<float4*>(S_at + ((size_t)p * D + k0 + j) * D + c4) = S[p][j];
        }
        leave(p, o);
    }
    __syncthreads();
    float y = 0.f;
    if (finishes) {                                          // (whole waves)
        y = gather();
        const float ss = wave_sum(y * y);
        if (lane == 0) part[wave] = ss;
    }
    __syncthreads();
    if (!finishes) return;
    const int p = tid / D;
    const float rs = 1.0f / sqrtf((part[2 * p] + part[2 * p + 1]) / (float)D + A.eps);
    store_f32<TOut>(out, ((size_t)r * H + h0) * D + tid, y * rs * norm * ds_sigmoid(gate));
}

// The same a head and block, where the conv is done (it rides in the projection's launch) and the decays and the gate come
// through their bottleneck here: the head's rows of the matrix that leads back up, 64 KB of bfloat16 for a rank of 128, are
// asked for together with its state and multiplied while that is on its way, where they were a launch of their own. Nothing is
// left that two heads would share and change, so a query/key head's heads no longer share a block. Four neighbouring
// threads have a decay's or gate's sum. Measured in a graph, 4 rows of 8 heads, rank 128, width 1,024: 7.1 -> 6.0 us, and from
// the normed rows to the output projection's 17.3 us in four launches -> 10.5 in two; 1 row 16.7 -> 10.2, 16 rows 21.5 -> 13.6.
struct ChannelHeadArgs {
    const float* rows; int ld, beta_off, low_off;            // q | k | v behind conv and SiLU .., b, the bottlenecks' inner numbers
    const bf16_t* high; int high_ld, rank_a, rank_g;         // [2 * heads * 128, high_ld]: decays read columns 0 .. rank_a - 1,
                                                             // gates (from row heads * 128 on) rank_a .. rank_a + rank_g - 1
    const float* step_bias; const float* rate;               // [heads * 128], [heads]
    float* state;                                            // [slots, heads, 128, 128]
    const int32_t* slot;
    const float* norm;                                       // [heads * 128]
    int heads, kv_heads;
    float unit_eps, q_scale, eps;
};
#define CDH_RANK 128

template <typename TOut>
__global__ __launch_bounds__(1024) void k_channel_delta_head(const ChannelHeadArgs A, TOut* __restrict__ out) {
    constexpr int D = CDS_DIM, WAVES = 16;
    __shared__ __attribute__((aligned(16))) float sq[D], sk[D], sv[D], sg[D], su[D], gates[D], low[2 * CDH_RANK];
    __shared__ __attribute__((aligned(16))) float red[WAVES][D];
    __shared__ float squares[4], part[2], beta;
    const int r = blockIdx.x, h = blockIdx.y, kh = h / (A.heads / A.kv_heads);
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int c4 = (tid & 31) * 4, k0 = (tid >> 5) * 4;      // this thread's columns and rows of the state
    const float* row = A.rows + (size_t)r * A.ld;
    const int ranks = A.rank_a + A.rank_g;
    // what the block needs first, then the weights, then the state
    float mine = 0.f;
    if (tid < 3 * D) mine = row[tid < D ? kh * D + tid : tid < 2 * D ? (A.kv_heads + kh) * D + (tid - D) : (2 * A.kv_heads + h) * D + (tid - 2 * D)];
    else if (tid >= 512 && tid < 512 + ranks) mine = row[A.low_off + tid - 512];
    else if (tid == 3 * D) mine = row[A.beta_off + h];
    const int dot = tid >> 2, piece = tid & 3;               // decays 0 .. 127, then gates
    const bool gate = dot >= D;
    const int rank = gate ? A.rank_g : A.rank_a;
    const bf16_t* high = A.high + (size_t)((gate ? A.heads * D : 0) + h * D + (dot & (D - 1))) * A.high_ld + (gate ? A.rank_a : 0);
    uint4 w[CDH_RANK / 32];
#pragma unroll
    for (int j = 0; j < CDH_RANK / 32; ++j) w[j] = *reinterpret_cast<const uint4*>(high + min((j * 4 + piece) * 8, rank - 8));
    const float bias = A.step_bias[h * D + (dot & (D - 1))], rate = A.rate[h];
    const float norm = A.norm[h * D + (tid & (D - 1))];
    float* S_at = A.state + ((size_t)A.slot[r] * A.heads + h) * (D * D);
    float4 S[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) S[j] = *reinterpret_cast<const float4*>(S_at + (k0 + j) * D + c4);
    if (tid < 3 * D) {
        (tid < D ? sq : tid < 2 * D ? sk : sv)[tid & (D - 1)] = mine;
        if (tid < 2 * D) {
            const float ss = wave_sum(mine * mine);          // (whole waves: a head's 128 channels are two)
            if (lane == 0) squares[wave] = ss;
        }
    } else if (tid >= 512 && tid < 512 + ranks) {
        low[tid - 512] = bf16_to_f32(f32_to_bf16(mine));     // (what the matrix that leads back up reads is bfloat16)
    } else if (tid == 3 * D) {
        beta = ds_sigmoid(mine);
    }
    __syncthreads();
    {
        float sum = 0.f;
#pragma unroll
        for (int j = 0; j < CDH_RANK / 32; ++j) {
            const int at = (j * 4 + piece) * 8;
            if (at >= rank) continue;
            const float4 a = *reinterpret_cast<const float4*>(&low[(gate ? A.rank_a : 0) + at]);
            const float4 b = *reinterpret_cast<const float4*>(&low[(gate ? A.rank_a : 0) + at + 4]);
            const float l[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
            const unsigned u[4] = {w[j].x, w[j].y, w[j].z, w[j].w};
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                sum = fmaf(__uint_as_float(u[i] << 16), l[2 * i], sum);
                sum = fmaf(__uint_as_float(u[i] & 0xffff0000u), l[2 * i + 1], sum);
            }
        }
        sum = sum_near_first<4>(sum);
        if (piece == 0) {
            if (gate) gates[dot - D] = sum;
            else sg[dot] = expf(-rate * ds_softplus(sum + bias));
        }
    }
    __syncthreads();
    const float fq = A.q_scale * (1.0f / sqrtf(squares[0] + squares[1] + A.unit_eps));
    const float fk = 1.0f / sqrtf(squares[2] + squares[3] + A.unit_eps);
    const float4 kk = *reinterpret_cast<const float4*>(&sk[k0]), qq = *reinterpret_cast<const float4*>(&sq[k0]);
    const float4 gg = *reinterpret_cast<const float4*>(&sg[k0]);
    const float kj[4] = {kk.x * fk, kk.y * fk, kk.z * fk, kk.w * fk}, qj[4] = {qq.x * fq, qq.y * fq, qq.z * fq, qq.w * fq};
    const float g[4] = {gg.x, gg.y, gg.z, gg.w};
    // sums over the state's rows as the kernel above has them
    auto leave = [&](const float (&v)[4]) __attribute__((always_inline)) {
        const float4 s = make_float4(cds_halves(v[0]), cds_halves(v[1]), cds_halves(v[2]), cds_halves(v[3]));
        if (lane < 32) *reinterpret_cast<float4*>(&red[wave][c4]) = s;
    };
    auto gather = [&]() __attribute__((always_inline)) {
        float v[WAVES];
#pragma unroll
        for (int i = 0; i < WAVES; ++i) v[i] = red[i][tid & (D - 1)];
#pragma unroll
        for (int half = WAVES / 2; half > 0; half /= 2)
#pragma unroll
            for (int i = 0; i < half; ++i) v[i] += v[i + half];
        return v[0];
    };
    float seen[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        S[j] = make_float4(S[j].x * g[j], S[j].y * g[j], S[j].z * g[j], S[j].w * g[j]);
        seen[0] = fmaf(S[j].x, kj[j], seen[0]);
        seen[1] = fmaf(S[j].y, kj[j], seen[1]);
        seen[2] = fmaf(S[j].z, kj[j], seen[2]);
        seen[3] = fmaf(S[j].w, kj[j], seen[3]);
    }
    leave(seen);
    __syncthreads();
    if (tid < D) su[tid] = beta * (sv[tid] - gather());
    __syncthreads();
    const float4 u = *reinterpret_cast<const float4*>(&su[c4]);
    float o[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        S[j] = make_float4(fmaf(kj[j], u.x, S[j].x), fmaf(kj[j], u.y, S[j].y), fmaf(kj[j], u.z, S[j].z), fmaf(kj[j], u.w, S[j].w));
        o[0] = fmaf(S[j].x, qj[j], o[0]);
        o[1] = fmaf(S[j].y, qj[j], o[1]);
        o[2] = fmaf(S[j].z, qj[j], o[2]);
        o[3] = fmaf(S[j].w, qj[j], o[3]);
        *reinterpret_cast<float4*>(S_at + (k0 + j) * D + c4) = S[j];
    }
    leave(o);
    __syncthreads();
    float y = 0.f;
    if (tid < D) {                                           // (whole waves)
        y = gather();
        const float ss = wave_sum(y * y);
        if (lane == 0) part[wave] = ss;
    }
    __syncthreads();
    if (tid >= D) return;
    const float rs = 1.0f / sqrtf((part[0] + part[1]) / (float)D + A.eps);
    store_f32<TOut>(out, ((size_t)r * A.heads + h) * D + tid, y * rs * norm * ds_sigmoid(gates[tid]));
}

extern "C" int imparo_channel_delta_heads_takes(int heads, int kv_heads, int dim, int vdim, int taps, int rank_a, int rank_g) {
    return dim == CDS_DIM && vdim == CDS_DIM && taps >= 1 && taps <= CDS_MAX_TAPS && kv_heads > 0 && heads % kv_heads == 0 &&
           heads <= 65535 && rank_a >= 8 && rank_a <= CDH_RANK && rank_a % 8 == 0 && rank_g >= 8 && rank_g <= CDH_RANK && rank_g % 8 == 0;
}

extern "C" int imparo_channel_delta_heads(const float* rows, int ld, int beta_off, int low_off, const void* high, int high_ld,
                                          int rank_a, int rank_g, const float* step_bias, const float* rate, float* state,
                                          int n_slots, const int32_t* slot, const float* norm, void* out, int out_dtype, int n_rows,
                                          int heads, int kv_heads, float unit_eps, float q_scale, float eps, imparo_stream stream) {
    if (!rows || !high || !step_bias || !rate || !state || !slot || !norm || !out || n_rows < 0 || n_slots < 1) return IMPARO_BAD_ARGUMENT;
    if (!imparo_channel_delta_heads_takes(heads, kv_heads, CDS_DIM, CDS_DIM, 1, rank_a, rank_g)) return IMPARO_BAD_ARGUMENT;
    const int channels = (2 * kv_heads + heads) * CDS_DIM;
    if (beta_off < channels || ld < beta_off + heads || low_off < channels || ld < low_off + rank_a + rank_g ||
        high_ld < rank_a + rank_g || high_ld % 8 || ((uintptr_t)high & 15) || ((uintptr_t)state & 15))
        return IMPARO_BAD_ARGUMENT;
    if (out_dtype != IMPARO_F32 && out_dtype != IMPARO_BF16) return IMPARO_BAD_ARGUMENT;
    if (n_rows == 0) return IMPARO_OK;
    const ChannelHeadArgs a{rows, ld, beta_off, low_off, (const bf16_t*)high, high_ld, rank_a, rank_g, step_bias, rate, state, slot,
                            norm, heads, kv_heads, unit_eps, q_scale, eps};
    const dim3 grid((unsigned)n_rows, (unsigned)heads);
    hipStream_t s = (hipStream_t)stream;
    if (out_dtype == IMPARO_BF16) k_channel_delta_head<bf16_t><<<grid, 1024, 0, s>>>(a, (bf16_t*)out);
    else k_channel_delta_head<float><<<grid, 1024, 0, s>>>(a, (float*)out);
    return launch_status();
}

// Whether the launch below takes a mixer of these sizes.
extern "C" int imparo_channel_delta_step_takes(int heads, int kv_heads, int dim, int vdim, int taps) {
    return dim == CDS_DIM && vdim == CDS_DIM && taps >= 1 && taps <= CDS_MAX_TAPS && kv_heads > 0 &&
           (heads == kv_heads || heads == 2 * kv_heads);
}

extern "C" int imparo_channel_delta_step(const float* rows, int ld, int beta_off, const float* steps, int steps_ld, int gate_off,
                                         const float* conv_w, float* conv, int taps, const float* step_bias, const float* rate,
                                         float* state, int n_slots, const int32_t* slot, const float* norm, void* out,
                                         int out_dtype, int n_rows, int heads, int kv_heads, int dim, int vdim, float unit_eps,
                                         float q_scale, float eps, imparo_stream stream) {
    if (!rows || !steps || !conv_w || !step_bias || !rate || !state || !slot || !norm || !out || n_rows < 0 || n_slots < 1)
        return IMPARO_BAD_ARGUMENT;
    if (!imparo_channel_delta_step_takes(heads, kv_heads, dim, vdim, taps) || (taps > 1 && !conv)) return IMPARO_BAD_ARGUMENT;
    if (kv_heads > 65535 || beta_off < 0 || gate_off < heads * dim || ld < (2 * kv_heads + heads) * CDS_DIM ||
        ld < beta_off + heads || steps_ld < gate_off + heads * vdim || ((uintptr_t)state & 15))
        return IMPARO_BAD_ARGUMENT;
    if (out_dtype != IMPARO_F32 && out_dtype != IMPARO_BF16) return IMPARO_BAD_ARGUMENT;
    if (n_rows == 0) return IMPARO_OK;
    const ChannelStepArgs a{rows, ld, beta_off, steps, steps_ld, gate_off, conv_w, conv, taps, step_bias, rate,
                            state, slot, norm, heads, kv_heads, unit_eps, q_scale, eps};
    const dim3 grid((unsigned)n_rows, (unsigned)kv_heads);
    hipStream_t s = (hipStream_t)stream;
    if (heads == kv_heads) {
        if (out_dtype == IMPARO_BF16) k_channel_delta_step<bf16_t, 1><<<grid, 1024, 0, s>>>(a, (bf16_t*)out);
        else k_channel_delta_step<float, 1><<<grid, 1024, 0, s>>>(a, (float*)out);
    } else {
        if (out_dtype == IMPARO_BF16) k_channel_delta_step<bf16_t, 2><<<grid, 1024, 0, s>>>(a, (bf16_t*)out);
        else k_channel_delta_step<float, 2><<<grid, 1024, 0, s>>>(a, (float*)out);
    }
    return launch_status();
}

int imparo_load_code_decay_scan() {
    hipFuncAttributes attributes;
    return hipFuncGetAttributes(&attributes, reinterpret_cast<const void*>(&k_decay_carry)) == hipSuccess
               ? IMPARO_OK
               : IMPARO_LAUNCH_FAILED;
}
