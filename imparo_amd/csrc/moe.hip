// A routed feed-forward (mixture of experts) in five launches:
//   route    softmax over the router's outputs, the choice of `top` of them by score + correction,
//            the weights (the scores themselves, as they are), one wave a token;
//   plan     one block: how many (token, choice) entries each expert got, a slot for every entry
//            (the entries of one expert side by side), and the list of row tiles the products walk;
//   product  twice: a tile of one expert's slots times that expert's matrix (up with the activation
//            in its epilogue, then down), on the matrix cores in bfloat16, plain fused multiply-adds
//            in float32; the grid is sized by a bound that the host knows (no count comes back);
//   combine  a token's result: its chosen experts' rows times their weights, added in the order of
//            the choice; an expert past the last real one passes the token's input through.
// Which slot an entry gets depends on the order in which threads arrive; no result does: a row of
// a product is summed over k in one order wherever the row lies in its tile, and a token's sum
// over its experts runs in the order of its own choice.
#include "common.h"

#include <algorithm>
#include <type_traits>
#include "api.h"
#include "moe_route.h"

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

#define MOE_MAX_ROUTER 512          // router outputs (experts of both kinds)
#define MOE_MAX_EXPERTS 1024        // real experts the plan kernel keeps counters for
#define MOE_MAX_TOP 16              // experts a token chooses
#define MOE_COUNTED -1              // the rows of an empty tile that holds the number of tiles before the empty ones

extern "C" int imparo_moe_max_tiles(int n_entries, int n_experts, int tile_rows);

// ---------------------------------------------------------------- route
template <int N>
__device__ __forceinline__ void moe_better_of(float& best, int& at) {
    const float ob = lane_xor<N>(best);
    const int oa = lane_xor<N>(at);
    if (ob > best || (ob == best && oa < at)) best = ob, at = oa;
}
// the largest of the wave's, of equal ones the lowest index, in every lane
__device__ __forceinline__ void moe_best_of_wave(float& best, int& at) {
    moe_better_of<32>(best, at);
    moe_better_of<16>(best, at);
    moe_better_of<8>(best, at);
    moe_better_of<4>(best, at);
    moe_better_of<2>(best, at);
    moe_better_of<1>(best, at);
}

__device__ __forceinline__ void moe_route_token(const float* __restrict__ logits, const float* __restrict__ correction,
                                                int32_t* __restrict__ choice, float* __restrict__ weight, int t,
                                                int n_router, int top, int scoring, const MoeRouteRules rules) {
    const int lane = threadIdx.x & (WAVE - 1);
    constexpr int PER = MOE_MAX_ROUTER / WAVE;
    const int used = top + rules.always;
    choice += (size_t)t * used;
    weight += (size_t)t * used;
    if (lane < rules.always) {
        choice[top + lane] = n_router + lane;
        weight[top + lane] = 1.0f;
    }
    float z[PER], pick[PER];
    float m = -INFINITY;
#pragma unroll
    for (int j = 0; j < PER; ++j) {
        const int i = lane + j * WAVE;
        z[j] = i < n_router ? logits[(size_t)t * rules.logits_ld + i] : -INFINITY;
        m = fmaxf(m, z[j]);
    }
    if (scoring == MOE_SCORE_SIGMOID) {
        // every output scored by itself
#pragma unroll
        for (int j = 0; j < PER; ++j) z[j] = (lane + j * WAVE) < n_router ? 1.0f / (1.0f + expf(-z[j])) : 0.f;
    } else if (scoring == MOE_SCORE_SOFTMAX) {
        m = wave_max(m);
        float sum = 0.f;
#pragma unroll
        for (int j = 0; j < PER; ++j) {
            z[j] = (lane + j * WAVE) < n_router ? expf(z[j] - m) : 0.f;
            sum += z[j];
        }
        sum = wave_sum(sum);
        const float inv = 1.0f / sum;
#pragma unroll
        for (int j = 0; j < PER; ++j) z[j] *= inv;
    }
#pragma unroll
    for (int j = 0; j < PER; ++j) {
        const int i = lane + j * WAVE;
        pick[j] = i < n_router ? z[j] + (correction ? correction[i] : 0.f) : -INFINITY;
    }
    if (rules.groups > 1) {
        // lane g scores group g (at most 64 groups): the sum of its two largest choice scores, read from
        // the lanes that hold them; then `keep` rounds of a wave-wide argmax mark the groups that stay
        const int per = n_router / rules.groups;
        float gscore = -INFINITY;
        {
            float b1 = -INFINITY, b2 = -INFINITY;
            for (int e = 0; e < per; ++e) {
                // every lane reads output (lane * per + e) of its own group; lanes beyond the groups read output 0
                const int i = lane < rules.groups ? lane * per + e : 0;
                float v = -INFINITY;
#pragma unroll
                for (int j = 0; j < PER; ++j) {
                    const float got = __shfl(pick[j], i & (WAVE - 1), WAVE);
                    if (i / WAVE == j) v = got;
                }
                if (v > b1) { b2 = b1; b1 = v; } else if (v > b2) { b2 = v; }
            }
            if (lane < rules.groups) gscore = per > 1 ? b1 + b2 : b1;
        }
        unsigned long long kept = 0ull;
        for (int k = 0; k < rules.keep; ++k) {
            float best = gscore;
            int at = lane < rules.groups ? lane : 0x7fffffff;
            moe_best_of_wave(best, at);
            if (at < rules.groups) kept |= 1ull << at;
            if (lane == at) gscore = -INFINITY;
        }
#pragma unroll
        for (int j = 0; j < PER; ++j) {
            const int i = lane + j * WAVE;
            if (i < n_router && !((kept >> (i / per)) & 1ull)) pick[j] = -INFINITY;
        }
    }
    float chosen_sum = 0.f, chosen_max = -INFINITY, mine = -INFINITY;       // mine: lane k keeps the k-th choice's score
    for (int k = 0; k < top; ++k) {
        // the largest choice score that is left; of equal ones the lowest index
        float best = -INFINITY;
        int at = 0x7fffffff;
#pragma unroll
        for (int j = 0; j < PER; ++j) {
            const int i = lane + j * WAVE;
            if (pick[j] > best) { best = pick[j]; at = i; }
        }
        moe_best_of_wave(best, at);
        float s = 0.f;
#pragma unroll
        for (int j = 0; j < PER; ++j)
            if (lane + j * WAVE == at) { s = z[j]; pick[j] = -INFINITY; }
        s = wave_sum(s);           // one lane holds it
        chosen_sum += s;
        chosen_max = fmaxf(chosen_max, s);
        if (lane == k) mine = s;
        if (lane == 0) {
            choice[k] = at;
            if (scoring != MOE_SCORE_CHOSEN) weight[k] = s;
        }
    }
    if (scoring == MOE_SCORE_CHOSEN) {
        const float e = lane < top ? expf(mine - chosen_max) : 0.f;
        const float sum = wave_sum(e);
        if (lane < top) weight[lane] = e / sum * rules.scale;
        return;
    }
    if (rules.normalize || rules.scale != 1.0f) {
        const float f = (rules.normalize ? 1.0f / (chosen_sum + 1e-20f) : 1.0f) * rules.scale;
        if (lane == 0)
            for (int k = 0; k < top; ++k) weight[k] *= f;
    }
}

__global__ void k_moe_route(const float* __restrict__ logits, const float* __restrict__ correction,
                            int32_t* __restrict__ choice, float* __restrict__ weight, int n_tokens, int n_router,
                            int top, int scoring, const MoeRouteRules rules) {
    const int t = blockIdx.x * (blockDim.x / WAVE) + threadIdx.x / WAVE;
    if (t >= n_tokens) return;
    if (moe_routes_narrow(n_router, top, rules))
        moe_route_token_narrow(logits, correction, choice, weight, t, n_router, top, scoring, rules, nullptr);
    else
        moe_route_token(logits, correction, choice, weight, t, n_router, top, scoring, rules);
}

static bool moe_rules_fit(const MoeRouteRules& r, int n_router, int top) {
    if (r.logits_ld < n_router || r.groups < 1 || r.groups > WAVE || n_router % r.groups) return false;
    if (r.groups > 1 && (r.keep < 1 || r.keep > r.groups || r.keep * (n_router / r.groups) < top)) return false;
    if (r.always < 0 || top + r.always > MOE_MAX_USED) return false;
    return r.scale == r.scale;
}

extern "C" int imparo_moe_route(const float* logits, const float* correction, int32_t* choice, float* weight,
                                int n_tokens, int n_router, int top, int scoring, int logits_ld, int groups, int keep,
                                int normalize, float scale, int always, imparo_stream stream) {
    if (!logits || !choice || !weight || n_tokens < 0) return IMPARO_BAD_ARGUMENT;
    const MoeRouteRules rules{logits_ld, groups, keep, normalize, scale, always};
    if (!moe_rules_fit(rules, n_router, top)) return IMPARO_BAD_ARGUMENT;
    if (scoring < MOE_SCORE_SOFTMAX || scoring > MOE_SCORE_CHOSEN) return IMPARO_BAD_ARGUMENT;
    if (n_router < 1 || n_router > MOE_MAX_ROUTER || top < 1 || top > n_router || top > MOE_MAX_TOP)
        return IMPARO_BAD_ARGUMENT;
    if (n_tokens == 0) return IMPARO_OK;
    k_moe_route<<<(n_tokens + 3) / 4, 4 * WAVE, 0, (hipStream_t)stream>>>(logits, correction, choice, weight, n_tokens,
                                                                         n_router, top, scoring, rules);
    return launch_status();
}

// ---------------------------------------------------------------- plan
// tiles[3 i ..]: expert, first slot, rows of tile i; where the list has ended expert -1, the number of tiles that hold rows,
// MOE_COUNTED (k_moe_gemm_dma deals the tiles to the XCDs by that number).
struct MoePlanShared {
    int count[MOE_MAX_EXPERTS], first[MOE_MAX_EXPERTS], first_tile[MOE_MAX_EXPERTS + 1];
};

// From every expert's count its first slot and first tile
__device__ __forceinline__ void moe_plan_firsts(MoePlanShared& sh, int n_experts, int tile_rows) {
    int* count = sh.count;
    int* first = sh.first;
    int* first_tile = sh.first_tile;
    const int tid = threadIdx.x;
    if (n_experts <= WAVE) {
        if (tid < WAVE) {                    // a lane an expert
            const int c = tid < n_experts ? count[tid] : 0, t = (c + tile_rows - 1) / tile_rows;
            int slots = 0, n_tiles = 0, all = 0;
            for (int e = 0; e < n_experts; ++e) {
                const int ce = __builtin_amdgcn_readlane(c, e), te = __builtin_amdgcn_readlane(t, e);
                slots += e < tid ? ce : 0;
                n_tiles += e < tid ? te : 0;
                all += te;
            }
            if (tid < n_experts) {
                first[tid] = slots;
                first_tile[tid] = n_tiles;
            }
            if (tid == 0) first_tile[n_experts] = all;
        }
    } else if (tid == 0) {
        int slots = 0, n_tiles = 0;
        for (int e = 0; e < n_experts; ++e) {
            first[e] = slots;
            first_tile[e] = n_tiles;
            slots += count[e];
            n_tiles += (count[e] + tile_rows - 1) / tile_rows;
        }
        first_tile[n_experts] = n_tiles;
    }
}

__device__ __forceinline__ void moe_plan_tiles(const MoePlanShared& sh, int n_experts, int tile_rows, int32_t* __restrict__ tiles,
                                               int max_tiles) {
    const int* count = sh.count;
    const int* first = sh.first;
    const int* first_tile = sh.first_tile;
    const int tid = threadIdx.x;
    for (int e = tid; e < n_experts; e += blockDim.x) {
        const int n = count[e];
        int i = first_tile[e];
        for (int r = 0; r < n && i < max_tiles; r += tile_rows, ++i) {
            tiles[3 * i] = e;
            tiles[3 * i + 1] = first[e] + r;
            tiles[3 * i + 2] = min(tile_rows, n - r);
        }
    }
    for (int i = first_tile[n_experts] + tid; i < max_tiles; i += blockDim.x) {
        tiles[3 * i] = -1;
        tiles[3 * i + 1] = first_tile[n_experts];       // an empty tile says how many come before the first empty one,
        tiles[3 * i + 2] = MOE_COUNTED;                 // and that it says so
    }
}

__device__ __forceinline__ void moe_plan_block(MoePlanShared& sh, const int32_t* __restrict__ choice, int n_entries,
                                               int n_experts, int tile_rows, int32_t* __restrict__ slot_of_entry,
                                               int32_t* __restrict__ entry_of_slot, int32_t* __restrict__ tiles,
                                               int max_tiles) {
    int* count = sh.count;
    int* first = sh.first;
    const int tid = threadIdx.x;
    for (int e = tid; e < n_experts; e += blockDim.x) count[e] = 0;
    __syncthreads();
    for (int i = tid; i < n_entries; i += blockDim.x) {
        const int e = choice[i];
        if (e >= 0 && e < n_experts) atomicAdd(&count[e], 1);
    }
    __syncthreads();
    moe_plan_firsts(sh, n_experts, tile_rows);
    __syncthreads();
    moe_plan_tiles(sh, n_experts, tile_rows, tiles, max_tiles);
    __syncthreads();
    for (int e = tid; e < n_experts; e += blockDim.x) count[e] = 0;      // now the cursor of each expert
    __syncthreads();
    for (int i = tid; i < n_entries; i += blockDim.x) {
        const int e = choice[i];
        int slot = -1;
        if (e >= 0 && e < n_experts) {
            slot = first[e] + atomicAdd(&count[e], 1);
            entry_of_slot[slot] = i;
        }
        slot_of_entry[i] = slot;
    }
}

__global__ __launch_bounds__(1024) void k_moe_plan(const int32_t* __restrict__ choice, int n_entries, int n_experts,
                                                   int tile_rows, int32_t* __restrict__ slot_of_entry,
                                                   int32_t* __restrict__ entry_of_slot, int32_t* __restrict__ tiles,
                                                   int max_tiles) {
    __shared__ MoePlanShared sh;
    moe_plan_block(sh, choice, n_entries, n_experts, tile_rows, slot_of_entry, entry_of_slot, tiles, max_tiles);
}

// Route and plan in one launch, for the few tokens of a decode step: the block's waves route the tokens in
// turn, then the block plans what they chose.
#define MOE_ROUTE_PLAN_TOKENS 64
__global__ __launch_bounds__(1024) void k_moe_route_plan(const float* __restrict__ logits,
                                                         const float* __restrict__ correction,
                                                         int32_t* __restrict__ choice, float* __restrict__ weight,
                                                         int n_tokens, int n_router, int top, int scoring,
                                                         const MoeRouteRules rules, int n_experts, int tile_rows,
                                                         int32_t* __restrict__ slot_of_entry,
                                                         int32_t* __restrict__ entry_of_slot,
                                                         int32_t* __restrict__ tiles, int max_tiles) {
    __shared__ MoePlanShared sh;
    __shared__ int32_t chosen[MOE_ROUTE_PLAN_TOKENS * MOE_MAX_USED];       // (the plan need not wait for memory to give it back)
    const int entries = n_tokens * (top + rules.always);
    if (moe_routes_narrow(n_router, top, rules)) {
        for (int t = threadIdx.x / WAVE; t < n_tokens; t += blockDim.x / WAVE)
            moe_route_token_narrow(logits, correction, choice, weight, t, n_router, top, scoring, rules, chosen);
        __syncthreads();
        moe_plan_block(sh, chosen, entries, n_experts, tile_rows, slot_of_entry, entry_of_slot, tiles, max_tiles);
        return;
    }
    for (int t = threadIdx.x / WAVE; t < n_tokens; t += blockDim.x / WAVE)
        moe_route_token(logits, correction, choice, weight, t, n_router, top, scoring, rules);
    __threadfence_block();
    __syncthreads();
    moe_plan_block(sh, choice, entries, n_experts, tile_rows, slot_of_entry, entry_of_slot, tiles, max_tiles);
}

extern "C" int imparo_moe_route_plan_tokens() { return MOE_ROUTE_PLAN_TOKENS; }

extern "C" int imparo_moe_route_plan(const float* logits, const float* correction, int32_t* choice, float* weight,
                                     int n_tokens, int n_router, int top, int scoring, int n_experts, int tile_rows,
                                     int32_t* slot_of_entry, int32_t* entry_of_slot, int32_t* tiles, int max_tiles,
                                     int logits_ld, int groups, int keep, int normalize, float scale, int always,
                                     imparo_stream stream) {
    if (!logits || !choice || !weight || !slot_of_entry || !entry_of_slot || !tiles) return IMPARO_BAD_ARGUMENT;
    const MoeRouteRules rules{logits_ld, groups, keep, normalize, scale, always};
    if (!moe_rules_fit(rules, n_router, top)) return IMPARO_BAD_ARGUMENT;
    if (scoring < MOE_SCORE_SOFTMAX || scoring > MOE_SCORE_CHOSEN) return IMPARO_BAD_ARGUMENT;
    if (n_tokens < 0 || n_tokens > MOE_ROUTE_PLAN_TOKENS) return IMPARO_BAD_ARGUMENT;
    if (n_router < 1 || n_router > MOE_MAX_ROUTER || top < 1 || top > n_router || top > MOE_MAX_TOP)
        return IMPARO_BAD_ARGUMENT;
    if (n_experts < 0 || n_experts > MOE_MAX_EXPERTS || tile_rows < 1) return IMPARO_BAD_ARGUMENT;
    if (max_tiles < imparo_moe_max_tiles(n_tokens * (top + always), n_experts, tile_rows)) return IMPARO_SCRATCH_TOO_SMALL;
    if (n_tokens == 0) return IMPARO_OK;
    k_moe_route_plan<<<1, 1024, 0, (hipStream_t)stream>>>(logits, correction, choice, weight, n_tokens, n_router, top,
                                                          scoring, rules, n_experts, tile_rows, slot_of_entry, entry_of_slot,
                                                          tiles, max_tiles);
    return launch_status();
}

// ---------------------------------------------------------------- a prompt's router, choice and plan in two launches
// The router's product, the choice and every expert's count in one launch: a block brings 16 tokens' rows and the router's into LDS,
// all loads at once, one wave walks K in the order of the tile products (so that the logits are their bits and no near tie
// turns), then each of eight waves chooses for two tokens out of LDS and the block counts what they chose. The second launch places the
// entries: a block of 64 tokens adds up the counts of all blocks and of those before it, which is where its own entries
// start, so that no block waits for another. Bound by the trips to memory and the walk's chain of products.
// Measured, 2,048 tokens of 1,024, 4 of 8 chosen and one for all: product, choice and plan 9.3 + 3.9 + 9.8 us, now 8.9 + 4.4.
// The product as a tile of 128 rows had 16 blocks that streamed their activations alone, the plan one block for all entries.
#define MOE_ROUTER_TOKENS 16
#define MOE_ROUTER_MAX 32           // outputs, and the experts of the plan
#define MOE_ROUTER_K 1024           // of K in LDS at once
#define MOE_ROUTER_LD (MOE_ROUTER_K + 8)
#define MOE_PLACE_TOKENS 64

__global__ __launch_bounds__(512) void k_moe_router(const bf16_t* __restrict__ X, const bf16_t* __restrict__ W,
                                                    const float* __restrict__ bias, const float* __restrict__ correction,
                                                    int32_t* __restrict__ choice, float* __restrict__ weight,
                                                    int32_t* __restrict__ counts, int n_tokens, int n_router, int K, int top,
                                                    int scoring, const MoeRouteRules rules, int n_experts) {
    extern __shared__ __attribute__((aligned(16))) bf16_t rows[];        // [MOE_ROUTER_TOKENS + n_router][MOE_ROUTER_LD]: tokens, then outputs
    __shared__ float logits[MOE_ROUTER_TOKENS][MOE_ROUTER_MAX + 1];
    __shared__ int32_t chosen[MOE_ROUTER_TOKENS * MOE_MAX_USED];
    __shared__ int count[MOE_ROUTER_MAX];
    constexpr int WAVES = 8, PIECES = MOE_ROUTER_K / 8, AHEAD = 8;
    const int tid = threadIdx.x, lane = tid & (WAVE - 1), wave = __builtin_amdgcn_readfirstlane(tid / WAVE);
    const int t0 = blockIdx.x * MOE_ROUTER_TOKENS, n = min(MOE_ROUTER_TOKENS, n_tokens - t0), used = top + rules.always;
    if (tid < MOE_ROUTER_MAX) count[tid] = 0;
    union Frag {
        uint4 u;
        bf16x8 v;
    };
    f32x16 acc;
#pragma unroll
    for (int i = 0; i < 16; ++i) acc[i] = 0.f;
    for (int k0 = 0; k0 < K; k0 += MOE_ROUTER_K) {
        const int part = min(K - k0, MOE_ROUTER_K);          // (a multiple of 128)
        // a wave takes a row and half of what is here of it at a time, rows of tokens past the end the last one's
        const int piece = (wave & 1) * (PIECES / 2) + lane, all = MOE_ROUTER_TOKENS + n_router;
        const int at = k0 + min(piece * 8, part - 8);
        __syncthreads();                                     // (the part before has been read)
        for (int r0 = wave >> 1; r0 < all; r0 += 4 * AHEAD) {
            uint4 v[AHEAD];
#pragma unroll
            for (int i = 0; i < AHEAD; ++i) {
                const int r = min(r0 + 4 * i, all - 1);
                const bf16_t* row = r < MOE_ROUTER_TOKENS ? X + (size_t)(t0 + min(r, n - 1)) * K : W + (size_t)(r - MOE_ROUTER_TOKENS) * K;
                v[i] = *reinterpret_cast<const uint4*>(row + at);
            }
#pragma unroll
            for (int i = 0; i < AHEAD; ++i)
                if (r0 + 4 * i < all) *reinterpret_cast<uint4*>(&rows[(r0 + 4 * i) * MOE_ROUTER_LD + piece * 8]) = v[i];
        }
        __syncthreads();
        if (wave == 0) {
            // (rows 16 .. 31 of the product are rows 0 .. 15 again)
            const bf16_t* x = rows + (lane & 15) * MOE_ROUTER_LD + (lane >> 5) * 8;
            const bf16_t* w = rows + (MOE_ROUTER_TOKENS + min(lane & 31, n_router - 1)) * MOE_ROUTER_LD + (lane >> 5) * 8;
            Frag a[2][4], b[2][4];
            auto read = [&](int k, Frag (&fa)[4], Frag (&fb)[4]) __attribute__((always_inline)) {
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    fa[i].u = *reinterpret_cast<const uint4*>(x + k + 16 * i);
                    fb[i].u = *reinterpret_cast<const uint4*>(w + k + 16 * i);
                }
                __builtin_amdgcn_sched_barrier(0);           // (the next operands are asked for before a product waits for these)
            };
            auto multiply = [&](const Frag (&fa)[4], const Frag (&fb)[4]) __attribute__((always_inline)) {
#pragma unroll
                for (int i = 0; i < 4; ++i) acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[i].v, fb[i].v, acc, 0, 0, 0);
                __builtin_amdgcn_sched_barrier(0);
            };
            read(0, a[0], b[0]);
            for (int k = 0; k < part; k += 128) {
                read(k + 64, a[1], b[1]);
                multiply(a[0], b[0]);
                read(min(k + 128, part - 64), a[0], b[0]);
                multiply(a[1], b[1]);
            }
        }
    }
    if (wave == 0) {                                         // lane: output lane % 32 of 8 tokens
        const int o = lane & 31;
        const float bo = bias && o < n_router ? bias[o] : 0.f;
#pragma unroll
        for (int i = 0; i < 8; ++i) logits[(i >> 2) * 8 + (lane >> 5) * 4 + (i & 3)][o] = acc[i] + bo;
    }
    __syncthreads();
    for (int t = wave; t < n; t += WAVES)
        moe_route_lanes(lane < n_router ? logits[t][min(lane, MOE_ROUTER_MAX)] : -INFINITY, correction, choice + (size_t)t0 * used,
                        weight + (size_t)t0 * used, t, n_router, top, scoring, rules, chosen);
    __syncthreads();
    for (int i = tid; i < n * used; i += blockDim.x) {
        const int e = chosen[i];
        if (e >= 0 && e < n_experts) atomicAdd(&count[e], 1);
    }
    __syncthreads();
    if (tid < n_experts) counts[(size_t)blockIdx.x * n_experts + tid] = count[tid];
}

__global__ __launch_bounds__(512) void k_moe_place(const int32_t* __restrict__ choice, const int32_t* __restrict__ counts, int n_tokens,
                                                   int used, int n_experts, int tile_rows, int32_t* __restrict__ slot_of_entry,
                                                   int32_t* __restrict__ entry_of_slot, int32_t* __restrict__ tiles, int max_tiles) {
    constexpr int PER = MOE_PLACE_TOKENS / MOE_ROUTER_TOKENS;
    __shared__ MoePlanShared sh;
    __shared__ int next[MOE_ROUTER_MAX];                 // the block's next slot of an expert, from the expert's first
    const int tid = threadIdx.x, blocks = (n_tokens + MOE_ROUTER_TOKENS - 1) / MOE_ROUTER_TOKENS;
    const int first_entry = blockIdx.x * MOE_PLACE_TOKENS * used, entries = min(MOE_PLACE_TOKENS, n_tokens - (int)blockIdx.x * MOE_PLACE_TOKENS) * used;
    if (tid < MOE_ROUTER_MAX) sh.count[tid] = 0, next[tid] = 0;
    __syncthreads();
    const int stripes = blockDim.x / n_experts, e = tid % n_experts;
    if (tid < stripes * n_experts) {
        int all = 0, before = 0;
#pragma unroll 4
        for (int b = tid / n_experts; b < blocks; b += stripes) {
            const int c = counts[(size_t)b * n_experts + e];
            all += c;
            before += b < (int)blockIdx.x * PER ? c : 0;
        }
        atomicAdd(&sh.count[e], all);
        atomicAdd(&next[e], before);
    }
    __syncthreads();
    moe_plan_firsts(sh, n_experts, tile_rows);
    __syncthreads();
    if (blockIdx.x == 0) moe_plan_tiles(sh, n_experts, tile_rows, tiles, max_tiles);
    for (int i = tid; i < entries; i += blockDim.x) {
        const int mine = choice[first_entry + i];
        int slot = -1;
        if (mine >= 0 && mine < n_experts) {
            slot = sh.first[mine] + atomicAdd(&next[mine], 1);
            entry_of_slot[slot] = first_entry + i;
        }
        slot_of_entry[first_entry + i] = slot;
    }
}

// Whether the two launches take so many tokens and a router of so many outputs over rows of k: where the product alone would go to
// the tiles whose order the walk keeps (more than 128 rows, a K in 128s), and a 32 of outputs holds them.
extern "C" int imparo_moe_router_takes(int n_tokens, int n_router, int n_experts, int top, int groups, int always, int k) {
    return n_tokens > 128 && (long long)n_tokens * k < (1LL << 31) && n_router >= 1 && n_router <= MOE_ROUTER_MAX && n_experts >= 1 && n_experts <= MOE_ROUTER_MAX && top >= 1 && top <= n_router &&
           top <= MOE_MAX_TOP && always >= 0 && top + always <= MOE_MAX_USED && groups == 1 &&
           k >= 128 && k % 128 == 0;
}

// ... and where they are faster than the three. What they save is the plan by one block, 0.7 ns an entry, and a launch; what they cost is
// that each 16 tokens read the whole router and one wave walks K, in rounds of as many blocks as the CUs' LDS holds at once (three a CU
// with up to 9 outputs, two up to 21, one above). In one round K is walked as fast as the tiles walk it, in more it
// is not, and the entries have to pay for that. Measured, us three launches | two, 4 chosen: 2,048 tokens of 1,024, 8 outputs 18.9 | 11.1, 32
// outputs 20.0 | 14.5, of 8,192 46.2 | 49.0; 8,192 of 2,048, 32 outputs 44.8 | 35.9, of 4,096 52.2 | 61.9; 16,384 of 8,192, 22 outputs 102.5 | 164;
// one chosen, 16 outputs of 2,048 37.0 | 38.4; 512 tokens of 128, 32 outputs 12.1 | 12.9. Of 931 forms one is slower by more than 2 %, by 3.
extern "C" int imparo_moe_router_pays(int n_tokens, int n_router, int top, int k) {
    const bool one_round = n_tokens <= (n_router <= 9 ? 3 : n_router <= 21 ? 2 : 1) * 256 * MOE_ROUTER_TOKENS;
    if (n_router <= 9) return one_round || k <= 4096 * top;
    if (n_router <= 21) return one_round ? k <= 4096 || n_tokens <= 4096 || top >= 4 : k <= 1280 * top;
    if (!one_round) return top >= 2 && k <= 512 * top;
    if (n_tokens < 2048) return n_router <= 24 || k >= 512 || n_tokens * top >= 4096;
    return k <= 3072 || (top >= 4 && k <= 4096) || top >= 8;
}

extern "C" int imparo_moe_router_blocks(int n_tokens) { return (n_tokens + MOE_ROUTER_TOKENS - 1) / MOE_ROUTER_TOKENS; }

extern "C" int imparo_moe_router_plan(const void* x, const void* w, const float* bias, const float* correction, int32_t* choice,
                                      float* weight, int32_t* counts, int n_tokens, int n_router, int k, int top, int scoring,
                                      int normalize, float scale, int always, int n_experts, int tile_rows, int32_t* slot_of_entry,
                                      int32_t* entry_of_slot, int32_t* tiles, int max_tiles, imparo_stream stream) {
    if (!x || !w || !choice || !weight || !counts || !slot_of_entry || !entry_of_slot || !tiles || n_tokens < 0) return IMPARO_BAD_ARGUMENT;
    if (!imparo_moe_router_takes(n_tokens, n_router, n_experts, top, 1, always, k) || scale != scale || tile_rows < 1) return IMPARO_BAD_ARGUMENT;
    if (scoring < MOE_SCORE_SOFTMAX || scoring > MOE_SCORE_CHOSEN || (((uintptr_t)x | (uintptr_t)w) & 15)) return IMPARO_BAD_ARGUMENT;
    if ((long long)n_tokens * (top + always) > 0x7fffffffLL) return IMPARO_BAD_ARGUMENT;
    if (max_tiles < imparo_moe_max_tiles(n_tokens * (top + always), n_experts, tile_rows)) return IMPARO_SCRATCH_TOO_SMALL;
    const MoeRouteRules rules{n_router, 1, 1, normalize, scale, always};
    const unsigned blocks = (unsigned)imparo_moe_router_blocks(n_tokens);
    hipStream_t s = (hipStream_t)stream;
    const int lds_bytes = (MOE_ROUTER_TOKENS + n_router) * MOE_ROUTER_LD * (int)sizeof(bf16_t);
    if (hipFuncSetAttribute((const void*)k_moe_router, hipFuncAttributeMaxDynamicSharedMemorySize,
                            (MOE_ROUTER_TOKENS + MOE_ROUTER_MAX) * MOE_ROUTER_LD * (int)sizeof(bf16_t)) != hipSuccess)
        return IMPARO_LAUNCH_FAILED;
    k_moe_router<<<blocks, 512, lds_bytes, s>>>((const bf16_t*)x, (const bf16_t*)w, bias, correction, choice, weight, counts, n_tokens,
                                                n_router, k, top, scoring, rules, n_experts);
    const int status = launch_status();
    if (status != IMPARO_OK) return status;
    k_moe_place<<<(n_tokens + MOE_PLACE_TOKENS - 1) / MOE_PLACE_TOKENS, 512, 0, s>>>(choice, counts, n_tokens, top + always, n_experts,
                                                                                   tile_rows, slot_of_entry, entry_of_slot, tiles,
                                                                                   max_tiles);
    return launch_status();
}

extern "C" int imparo_moe_max_tiles(int n_entries, int n_experts, int tile_rows) {
    if (n_entries <= 0 || tile_rows <= 0) return 0;
    return (n_entries + tile_rows - 1) / tile_rows + (n_experts < n_entries ? n_experts : n_entries);
}

// Rows of a product's tile for this many entries over this many experts: the wide tile where an
// expert's share fills it, the narrow one else (many experts), tiles of 16 for the few entries of a decode step.
extern "C" int imparo_moe_tile_rows(int n_entries, int n_experts, int dtype) {
    if (dtype != IMPARO_BF16) return 64;
    if (n_entries <= 128) return 16;          // a decode step: the experts' matrices are streamed once, few rows each
    return (n_experts > 0 && n_entries / n_experts >= 96) ? 128 : 64;
}

extern "C" int imparo_moe_plan(const int32_t* choice, int n_entries, int n_experts, int tile_rows,
                               int32_t* slot_of_entry, int32_t* entry_of_slot, int32_t* tiles, int max_tiles,
                               imparo_stream stream) {
    if (!choice || !slot_of_entry || !entry_of_slot || !tiles || n_entries < 0) return IMPARO_BAD_ARGUMENT;
    if (n_experts < 0 || n_experts > MOE_MAX_EXPERTS || tile_rows < 1) return IMPARO_BAD_ARGUMENT;
    if (max_tiles < imparo_moe_max_tiles(n_entries, n_experts, tile_rows)) return IMPARO_SCRATCH_TOO_SMALL;
    if (n_entries == 0) return IMPARO_OK;
    k_moe_plan<<<1, 1024, 0, (hipStream_t)stream>>>(choice, n_entries, n_experts, tile_rows, slot_of_entry,
                                                    entry_of_slot, tiles, max_tiles);
    return launch_status();
}

// ---------------------------------------------------------------- products
#define MOE_EPI_NONE 0
#define MOE_EPI_RELU2 1        // max(z, 0)^2
#define MOE_EPI_GATED 2        // bfloat16 only: an expert's rows are 32 gate rows, the 32 up rows that belong to them, and so
                               // on; out has half as many columns: act(w g, w u) (moe_act below)

// What the gated epilogue needs beside its products: a bound for every expert (limits null: SiLU without bounds), and
// the factor w of a slot, the weight of its entry (weight null: 1).
struct MoeGate {
    const float* limits;
    float alpha;
    const float* weight;
    int n_entries;
};

// act(g, u) = silu(g) u, or with limit > 0 the gated unit with bounds g' sigmoid(alpha g') (u' + 1),
// g' = min(g, limit), u' = clamp(u, -limit, limit).
__device__ __forceinline__ float moe_act(float g, float u, float limit, float alpha) {
    if (limit > 0.f) {
        g = fminf(g, limit);
        u = fminf(fmaxf(u, -limit), limit) + 1.0f;
    } else {
        alpha = 1.0f;
    }
    return g / (1.0f + expf(-alpha * g)) * u;
}
// the same with the hardware's exp2 and reciprocal, for results that are rounded to bfloat16
__device__ __forceinline__ float moe_act_fast(float g, float u, float limit, float alpha) {
    if (limit > 0.f) {
        g = fminf(g, limit);
        u = fminf(fmaxf(u, -limit), limit) + 1.0f;
    } else {
        alpha = 1.0f;
    }
    return g * __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(-1.44269504f * alpha * g)) * u;
}
// a slot's factor; a slot that no entry has counts for nothing
__device__ __forceinline__ float moe_slot_weight(const MoeGate& gate, const int32_t* __restrict__ entry_of_slot, int slot) {
    if (!gate.weight) return 1.0f;
    const int e = entry_of_slot[slot];
    return (e >= 0 && e < gate.n_entries) ? gate.weight[e] : 0.f;
}

__device__ __forceinline__ float moe_epilogue(float v, int epi) {
    if (epi == MOE_EPI_RELU2) {
        v = fmaxf(v, 0.f);
        v *= v;
    }
    return v;
}

// What a tile's products become: a wave's WM x WN of 32 x 32 at (wave / ACROSS, wave % ACROSS) of the block's tile go
// through the epilogue to their slots' rows.
template <int WM, int WN, int ACROSS, typename TOut, bool GATED>
__device__ __forceinline__ void moe_store_tile(const f32x16 (&acc)[WM][WN], TOut* __restrict__ out,
                                               const int32_t* __restrict__ entry_of_slot, const MoeGate& gate, int expert,
                                               int row0, int rows, int n0, int N, int epi) {
    static_assert(!GATED || WN == 2, "a wave's two tiles side by side are a gate's and its up's");
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int wm = wave / ACROSS, wn = wave % ACROSS;
    // a lane holds column lane % 32 of a 32 x 32 product, rows 8 (r / 4) + 4 (lane / 32) + r % 4
    if constexpr (GATED) {
        const float limit = gate.limits ? gate.limits[expert] : 0.f;
        const int n = (n0 + wn * 64) / 2 + (lane & 31);
        if (n < N / 2)
#pragma unroll
            for (int i = 0; i < WM; ++i)
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    const int m = wm * 32 * WM + i * 32 + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3);
                    if (m >= rows) continue;
                    const float w = moe_slot_weight(gate, entry_of_slot, row0 + m);
                    store_f32<TOut>(out, (size_t)(row0 + m) * (N / 2) + n,
                                    moe_act_fast(w * acc[i][0][r], w * acc[i][WN - 1][r], limit, gate.alpha));
                }
        return;
    }
#pragma unroll
    for (int i = 0; i < WM; ++i)
#pragma unroll
        for (int j = 0; j < WN; ++j) {
            const int n = n0 + wn * 32 * WN + j * 32 + (lane & 31);
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const int m = wm * 32 * WM + i * 32 + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3);
                if (m < rows && n < N) store_f32<TOut>(out, (size_t)(row0 + m) * N + n, moe_epilogue(acc[i][j][r], epi));
            }
        }
}

// out[slot, n] = epi(sum_k a[row(slot), k] * w[expert, n, k]) for the slots of one tile. row(slot) is the
// slot itself, or with gather_div the token of the slot's entry (entry / gather_div). Four waves as 2 x 2,
// each WM x WN products of 32 x 32; K in steps of 64 through two LDS stages, the next step's loads in
// registers while this one is multiplied. K is a multiple of 8.
template <int WM, int WN, typename TOut, bool GATED = false>
__global__ __launch_bounds__(256) void k_moe_gemm_bf16(const bf16_t* __restrict__ A, int a_ld, int gather_div,
                                                       const int32_t* __restrict__ entry_of_slot,
                                                       const bf16_t* __restrict__ W, TOut* __restrict__ out,
                                                       const int32_t* __restrict__ tiles, int N, int K, int epi,
                                                       MoeGate gate = {}) {
    constexpr int TM = 64 * WM, TN = 64 * WN, LD = 72, BK = 64;
    __shared__ __attribute__((aligned(16))) bf16_t As[2][TM * LD];
    __shared__ __attribute__((aligned(16))) bf16_t Bs[2][TN * LD];
    const int expert = tiles[3 * blockIdx.x];
    if (expert < 0) return;
    const int row0 = tiles[3 * blockIdx.x + 1], rows = tiles[3 * blockIdx.x + 2];
    const int n0 = blockIdx.y * TN;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int wm = wave >> 1, wn = wave & 1;
    const bf16_t* Wb = W + (size_t)expert * N * K;
    const int kc = (tid & 7) * 8;
    const bf16_t* pa[TM / 32];
    const bf16_t* pb[TN / 32];
#pragma unroll
    for (int j = 0; j < TM / 32; ++j) {
        const int slot = row0 + min((tid >> 3) + 32 * j, rows - 1);
        const int src = gather_div ? entry_of_slot[slot] / gather_div : slot;
        pa[j] = A + (size_t)src * a_ld;
    }
#pragma unroll
    for (int j = 0; j < TN / 32; ++j) pb[j] = Wb + (size_t)min(n0 + (tid >> 3) + 32 * j, N - 1) * K;
    typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
    // two sets of registers, each holding one K-step's loads: a step's loads are asked for two steps ahead
    u32x4 ra0[TM / 32], rb0[TN / 32], ra1[TM / 32], rb1[TN / 32];
    const u32x4 zero = {0u, 0u, 0u, 0u};
    const int nk = (K + BK - 1) / BK;
    // the loads of K-step kt into registers; what lies beyond K comes as zeros (K is a multiple of 8, so a
    // piece of 8 is inside or outside as a whole) from an address inside the row; a step past the last
    // reads the last again and is never stored
#define MOE_FETCH(kt, ra, rb)                                                                                       \
    {                                                                                                               \
        const int k_ = min((kt), nk - 1) * BK + kc;                                                                 \
        const bool in_ = k_ < K;                                                                                    \
        const int kk_ = in_ ? k_ : 0;                                                                               \
        _Pragma("unroll") for (int j = 0; j < TM / 32; ++j) {                                                       \
            const u32x4 v_ = *reinterpret_cast<const u32x4*>(pa[j] + kk_);                                          \
            ra[j] = in_ ? v_ : zero;                                                                                \
        }                                                                                                           \
        _Pragma("unroll") for (int j = 0; j < TN / 32; ++j) {                                                       \
            const u32x4 v_ = *reinterpret_cast<const u32x4*>(pb[j] + kk_);                                          \
            rb[j] = in_ ? v_ : zero;                                                                                \
        }                                                                                                           \
    }
#define MOE_STASH(buf_, ra, rb)                                                                                     \
    {                                                                                                               \
        _Pragma("unroll") for (int j = 0; j < TM / 32; ++j)                                                         \
            *reinterpret_cast<u32x4*>(&As[buf_][((tid >> 3) + 32 * j) * LD + kc]) = ra[j];                          \
        _Pragma("unroll") for (int j = 0; j < TN / 32; ++j)                                                         \
            *reinterpret_cast<u32x4*>(&Bs[buf_][((tid >> 3) + 32 * j) * LD + kc]) = rb[j];                          \
    }
#define MOE_MULTIPLY(buf_)                                                                                          \
    _Pragma("unroll") for (int ks = 0; ks < BK / 16; ++ks) {                                                        \
        bf16x8 fa[WM], fb[WN];                                                                                      \
        _Pragma("unroll") for (int i = 0; i < WM; ++i)                                                              \
            fa[i] = *reinterpret_cast<const bf16x8*>(&As[buf_][a_base + i * 32 * LD + ks * 16]);                    \
        _Pragma("unroll") for (int j = 0; j < WN; ++j)                                                              \
            fb[j] = *reinterpret_cast<const bf16x8*>(&Bs[buf_][b_base + j * 32 * LD + ks * 16]);                    \
        _Pragma("unroll") for (int i = 0; i < WM; ++i)                                                              \
            _Pragma("unroll") for (int j = 0; j < WN; ++j)                                                          \
                acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[i], fb[j], acc[i][j], 0, 0, 0);              \
    }
    f32x16 acc[WM][WN];
#pragma unroll
    for (int i = 0; i < WM; ++i)
#pragma unroll
        for (int j = 0; j < WN; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;
    const int a_base = (wm * 32 * WM + (lane & 31)) * LD + (lane >> 5) * 8;
    const int b_base = (wn * 32 * WN + (lane & 31)) * LD + (lane >> 5) * 8;
    MOE_FETCH(0, ra0, rb0);
    MOE_FETCH(1, ra1, rb1);
    MOE_STASH(0, ra0, rb0);
    MOE_FETCH(2, ra0, rb0);
    __syncthreads();
    // step kt is multiplied out of stage kt % 2 while step kt + 1 goes from its registers into the other
    // stage and those registers take the loads of step kt + 3
    for (int kt = 0; kt < nk; kt += 2) {
        MOE_MULTIPLY(0);
        if (kt + 1 < nk) MOE_STASH(1, ra1, rb1);
        MOE_FETCH(kt + 3, ra1, rb1);
        __syncthreads();
        if (kt + 1 < nk) {
            MOE_MULTIPLY(1);
            if (kt + 2 < nk) MOE_STASH(0, ra0, rb0);
            MOE_FETCH(kt + 4, ra0, rb0);
            __syncthreads();
        }
    }
#undef MOE_FETCH
#undef MOE_STASH
#undef MOE_MULTIPLY
    moe_store_tile<WM, WN, 2, TOut, GATED>(acc, out, entry_of_slot, gate, expert, row0, rows, n0, N, epi);
}

// The same product for tiles of 128 rows by 256 whose K is a multiple of 64: operands go from memory straight into LDS
// (16 bytes a lane, eight rows of 128 bytes a load, the pieces of a row exchanged by its number instead of padded: no
// bank conflicts), three stages, the loads of two K-steps in flight while one is multiplied; eight waves of 64 x 64, one
// block a CU. A K-step is four sub-steps of 16; the barrier sits before the last one's products, which cover the reads
// of the next step's first sub-step. Each output is summed over k in the same order as above: the same bits. Tiles that
// share an expert's weight rows or its slots are neighbours on one XCD. Bound by the path into LDS and out of it (a
// wave's outputs read 16 KB of fragments a step). Measured, 10,240 slots of 9 experts: 1,536 by 1,024, gated, 52 us
// (the kernel above: 85); 1,024 by 768, float32 out, 34 us (53). Tiles of 128
// by 128 on two stages, two blocks a CU, were no faster.
#define MOE_DMA_BK 64
#define MOE_DMA_M 128
#define MOE_DMA_N 256
#define MOE_DMA_STAGE ((MOE_DMA_M + MOE_DMA_N) * MOE_DMA_BK)      // elements of a stage: slots' rows, then weight rows
#define MOE_DMA_LDS (3 * MOE_DMA_STAGE * (int)sizeof(bf16_t))
#define MOE_GROUP_M 8
template <typename TOut, bool GATED>
__global__ __launch_bounds__(512) void k_moe_gemm_dma(const bf16_t* __restrict__ A, int a_ld, int gather_div,
                                                      const int32_t* __restrict__ entry_of_slot,
                                                      const bf16_t* __restrict__ W, TOut* __restrict__ out,
                                                      const int32_t* __restrict__ tiles, int max_tiles, int tiles_n, int N,
                                                      int K, int epi, MoeGate gate) {
    constexpr int BK = MOE_DMA_BK, LA = MOE_DMA_M / 64, LW = MOE_DMA_N / 64;   // load instructions a wave and a step
    extern __shared__ __attribute__((aligned(1024))) bf16_t stages[];
    // the tiles that hold slots are dealt to the XCDs evenly (the grid is sized for more, and an XCD with a few blocks
    // more than its CUs take at once runs a round of its own for them)
    const int32_t* last = tiles + 3 * (max_tiles - 1);
    const int n_tiles = last[0] < 0 && last[2] == MOE_COUNTED ? min(last[1], max_tiles) : max_tiles;
    const int total = n_tiles * tiles_n;
    const int per_xcd = (total + 7) / 8;
    const int logical = (int)(blockIdx.x % 8) * per_xcd + (int)(blockIdx.x / 8);
    if ((int)(blockIdx.x / 8) >= per_xcd || logical >= total) return;
    const int per_group = MOE_GROUP_M * tiles_n;
    const int first_m = (logical / per_group) * MOE_GROUP_M;
    const int gsize = min(n_tiles - first_m, MOE_GROUP_M);
    const int tile = first_m + (logical % per_group) % gsize;
    const int n0 = (logical % per_group) / gsize * MOE_DMA_N;
    const int expert = tiles[3 * tile];
    if (expert < 0) return;
    const int row0 = tiles[3 * tile + 1], rows = tiles[3 * tile + 2];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int wm = wave >> 2, wn = wave & 3;
    // loading: instruction j of a wave fills rows 64 j + 8 wave .. + 7; lane -> row lane / 8, place lane % 8, where the
    // piece lane % 8 ^ swz(row) lies, swz(r) = (r & 7) ^ ((r >> 3) & 1)
    const int load_row = wave * 8 + (lane >> 3);
    const int load_piece = ((lane & 7) ^ (lane >> 3) ^ (wave & 1)) * 8;
    const bf16_t* from[LA + LW];
#pragma unroll
    for (int j = 0; j < LA; ++j) {
        const int slot = row0 + min(load_row + 64 * j, rows - 1);
        const int src = gather_div ? entry_of_slot[slot] / gather_div : slot;
        from[j] = A + (size_t)src * a_ld + load_piece;
    }
#pragma unroll
    for (int j = 0; j < LW; ++j) from[LA + j] = W + ((size_t)expert * N + min(n0 + load_row + 64 * j, N - 1)) * K + load_piece;
    const unsigned lds = (unsigned)(size_t)(__attribute__((address_space(3))) bf16_t*)stages;
    auto load_step = [&](int stage, int kt) __attribute__((always_inline)) {
        const unsigned to = __builtin_amdgcn_readfirstlane(lds + (stage * MOE_DMA_STAGE + wave * 8 * BK) * 2);
#pragma unroll
        for (int j = 0; j < LA + LW; ++j) load_to_lds_uncounted(from[j] + kt * BK, to + j * 64 * BK * 2);
    };
    // fragments: lane holds row lane % 32, K-half lane / 32 of a 32 x 16 piece; sub-step ks is pieces 2 ks, 2 ks + 1
    const int frag_row = lane & 31;
    const int swz = (frag_row & 7) ^ ((frag_row >> 3) & 1);
    const int a_base = (wm * 64 + frag_row) * BK + (((lane >> 5) ^ swz) << 3);
    const int b_base = (MOE_DMA_M + wn * 64 + frag_row) * BK + (((lane >> 5) ^ swz) << 3);
    f32x16 acc[2][2];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;
    auto read = [&](int stage, int ks, bf16x8 (&fa)[2], bf16x8 (&fb)[2]) __attribute__((always_inline)) {
        const bf16_t* at = stages + stage * MOE_DMA_STAGE;
#pragma unroll
        for (int i = 0; i < 2; ++i) fa[i] = *reinterpret_cast<const bf16x8*>(&at[(a_base ^ (ks << 4)) + i * 32 * BK]);
#pragma unroll
        for (int j = 0; j < 2; ++j) fb[j] = *reinterpret_cast<const bf16x8*>(&at[(b_base ^ (ks << 4)) + j * 32 * BK]);
    };
    auto multiply = [&](const bf16x8 (&fa)[2], const bf16x8 (&fb)[2]) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int j = 0; j < 2; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[i], fb[j], acc[i][j], 0, 0, 0);
    };
    const int nk = K / BK;
    bf16x8 fa0[2], fb0[2], fa1[2], fb1[2];
    load_step(0, 0);
    load_step(1, min(1, nk - 1));
    load_step(2, min(2, nk - 1));
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 * (LA + LW)) : "memory");
    __builtin_amdgcn_s_barrier();
    read(0, 0, fa0, fb0);
    int cur = 0;
    // K-step kt out of stage `cur`: on entry set 0 holds its first sub-step and the loads of steps kt + 1 and kt + 2 are
    // in flight; on exit set 0 holds the first sub-step of kt + 1 and those of kt + 2 and kt + 3 are. `after`: how many steps
    // follow, as far as it matters: the last three ask for nothing (2,048 tokens, 4 of 8 experts and a shared one, gate and up
    // over 1,024 46.2 us, the way back over 768 29.1, with the last step brought three times more 47.5 and 30.2)
    auto k_step = [&](int kt, auto after) __attribute__((always_inline)) {
        constexpr int AFTER = decltype(after)::value;
        const int next = cur == 2 ? 0 : cur + 1;
        read(cur, 1, fa1, fb1);
        multiply(fa0, fb0);
        __builtin_amdgcn_sched_barrier(0);                   // (reads and products stay where they are written)
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
        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(AFTER > 1 ? LA + LW : 0) : "memory");
        __builtin_amdgcn_s_barrier();
        read(next, 0, fa0, fb0);
        if constexpr (AFTER > 2) load_step(cur, kt + 3);
        multiply(fa1, fb1);
        __builtin_amdgcn_sched_barrier(0);
        cur = next;
    };
    int kt = 0;
    for (; kt + 3 < nk; ++kt) k_step(kt, std::integral_constant<int, 3>{});
    if (nk > 2) k_step(kt++, std::integral_constant<int, 2>{});
    if (nk > 1) k_step(kt++, std::integral_constant<int, 1>{});
    k_step(kt, std::integral_constant<int, 0>{});
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");         // (of a K of one step or two the last one came more than once)
    moe_store_tile<2, 2, 4, TOut, GATED>(acc, out, entry_of_slot, gate, expert, row0, rows, n0, N, epi);
}

// Few rows an expert (a decode step): a block takes a tile of 16 weight rows of one expert, gated a tile of gate rows and the
// up rows that belong to them, 32 rows further on, and up to 16 slots. A tile is the M side of 16x16x32 products; K is cut in
// four neighbouring parts over the block's waves, walked in runs of 64, U of them a round, and everything a round needs is
// asked for at once, from memory straight into the operand registers, as in decode_rows.hip (what bounds it is reading the
// experts' matrices and the trips to memory behind one another: the tile list, then the weights and the slots' tokens, whose
// rows come last, so nothing but products stands behind them). A lane takes 16 consecutive k of its row, so that four lanes
// read a row's 128 bytes side by side; the slots' rows are read with the same k order, which is all a dot product asks for.
// The waves' partial sums meet in LDS and are added in wave order. 4 of 8 experts and a shared one, 8 tokens: gate and up,
// 1,536 rows by 1,024 an expert, 9.4 us (12.0 with two runs a wave at a time, selects before every product and the blocks
// unevenly over the XCDs), the way back, 1,024 by 768, 6.2 (7.1); one token 6.3 and 4.6 (7.4 and 5.2). Over 3,920 forms of 4 to
// 128 experts 1.23 times as fast as that on average, 90 slower by more than 3 % and 0.1 us: gated, K of 1,024 and 2,048 over
// few rows, by 12 % at the most.
// DIRECT: no plan at all. A step of at most 16 tokens fits one tile of slots, so a block of expert `y` takes all tokens, finds
// in their choices (`tiles`: [max_tiles tokens, gather_div used]) which of them use the expert, and leaves where nobody does;
// rows of `out` (and of A, unless the tokens' own rows are read: bit 0 of `own_rows`) go by entry, token * used + place in its list
// (a token's choices differ: of two entries with the same expert the first is made). A row of the tile sums
// over k as it does in any other, so results have the bits of planned ones. Not faster by itself, and worth it for the launches that go
// with the plan (imparo_moe_direct_pays): cold weights, direct | planned us, gate and up, way back: 9 experts of 768 by 1,024, five a token, 1 token 6.8 | 5.9, 4.6 | 4.5,
// 8 tokens 8.1 | 8.3, 6.0 | 5.8; 16 of 512 by 2,048, four a token, 1 token 9.1 | 7.1, 4.5 | 4.0, 8 tokens 13.5 | 13.3, 8.1 | 7.5; 32 of
// 512 by 1,024, four a token, whose blocks mostly leave, 8 tokens 11.0 | 9.9, 6.8 | 5.9.
#define MOE_ROWS_WAVES 4
#define MOE_DIRECT_TOKENS 16
#define MOE_DIRECT_USED 8
template <typename TOut, bool GATED, int RT, int U, bool DIRECT = false>
__global__ __launch_bounds__(MOE_ROWS_WAVES * 64) void k_moe_gemm_rows16(const bf16_t* __restrict__ A, int a_ld, int gather_div,
                                                         const int32_t* __restrict__ entry_of_slot,
                                                         const bf16_t* __restrict__ W, TOut* __restrict__ out,
                                                         const int32_t* __restrict__ tiles, int max_tiles,
                                                         int N, int K, int epi, MoeGate gate, int own_rows) {
    typedef float f32x4 __attribute__((ext_vector_type(4)));
    typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
    constexpr int GROUPS = GATED ? RT / 2 : RT;          // of 16 outputs a block
    static_assert(!GATED || RT % 2 == 0, "as many gate tiles as up tiles");
    extern __shared__ float4 moe_part[];                 // [waves][RT][WAVE]
    // The tiles that hold slots come first in the grid, so that the XCDs, which take its blocks in turn, have equally many of
    // them (9 tiles of 12 by 24 blocks, tile after tile along the grid: 36 on two XCDs of 32 CUs and 24 on the others, 12.0 us
    // where this way it is 10.1).
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), waves = blockDim.x >> 6;
    const int c = lane & 15, g = lane >> 4;
    const int n0 = (int)blockIdx.x * 16 * GROUPS;
    int expert, row0 = 0, rows, entry = 0, slot;
    bool live;                                           // this lane's column of the tile is a slot of the expert's
    const bf16_t* arow;
    const int runs = (K + 63) / 64, a_wave = (runs + MOE_ROWS_WAVES - 1) / MOE_ROWS_WAVES;
    const int run_lo = wave * a_wave, run_hi = min(runs, run_lo + a_wave);
    u32x4 w[RT][U][2], x[U][2];
    // (no load under a branch: what lies past K is read again from inside the row, and its weights count as zeros)
    auto k_of = [&](int run, int h) { return min(min(run, runs - 1) * 64 + g * 16 + h * 8, K - 8); };
    auto ask_rows = [&](int first) __attribute__((always_inline)) {
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
            for (int h = 0; h < 2; ++h) x[u][h] = *reinterpret_cast<const u32x4*>(arow + k_of(first + u, h));
        __builtin_amdgcn_sched_barrier(0);
    };
    auto weight_row = [&](int t) {
        const int f = n0 + (t % GROUPS) * 16 + c;
        return W + ((size_t)expert * N + (GATED ? (f >> 5) * 64 + (f & 31) + (t / GROUPS) * 32 : min(f, N - 1))) * K;
    };
    auto ask_weights = [&](int first) __attribute__((always_inline)) {
#pragma unroll
        for (int t = 0; t < RT; ++t) {
            const bf16_t* wrow = weight_row(t);
#pragma unroll
            for (int u = 0; u < U; ++u)
#pragma unroll
                for (int h = 0; h < 2; ++h) w[t][u][h] = *reinterpret_cast<const u32x4*>(wrow + k_of(first + u, h));
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    if constexpr (DIRECT) {
        expert = blockIdx.y;
        rows = max_tiles;
        const int token = min(c, rows - 1), used = gather_div;
        // (all tokens' choices, at most 128, in two loads of the wave: who uses the expert is then two masks)
        const int entries = rows * used;
        int choice[2];
#pragma unroll
        for (int i = 0; i < 2; ++i) choice[i] = tiles[min(lane + 64 * i, entries - 1)];
        if (own_rows & 1) {                              // (the choices are on their way beside them)
            arow = A + (size_t)token * a_ld;
            ask_rows(run_lo);
        }
        // (where hardly an expert goes unchosen its rows are asked for before that is known: one trip to memory less. From four
        // entries an expert on; at two one in eight is unchosen, and its weights cost more than the trip: 16 experts of
        // 2,048 by 1,024, two a token, 16 tokens a layer 46.3 -> 40.9 us without)
        if (own_rows & 2) ask_weights(run_lo);
        const unsigned long long lo = __ballot(lane < entries && choice[0] == expert);
        const unsigned long long hi = __ballot(lane + 64 < entries && choice[1] == expert);
        const int bit = token * used;
        const unsigned long long mine = bit >= 64 ? hi >> (bit - 64) : bit ? lo >> bit | hi << (64 - bit) : lo;
        const int at = __ffsll((long long)(mine & ((1ull << used) - 1))) - 1;
        live = at >= 0 && c < rows;
        const unsigned long long who = __ballot(live);
        if (who == 0) return;
        entry = slot = token * used + max(at, 0);
        // (a column that is nobody's reads what the first one reads)
        if (!(own_rows & 1)) arow = A + (size_t)(live ? slot : __shfl(slot, __ffsll(who) - 1)) * a_ld;
    } else {
    const int32_t* last = tiles + 3 * (max_tiles - 1);
    // (what the tile holds is read beside the number of tiles, and nothing of either under a condition: one trip to memory of
    // 0.6 us, and not three)
    const unsigned tile = blockIdx.z * gridDim.y + blockIdx.y, listed = min(tile, (unsigned)max_tiles - 1);
    expert = tiles[3 * listed], row0 = tiles[3 * listed + 1], rows = tiles[3 * listed + 2];
    const int last_expert = last[0], last_rows = last[2];
    int counted = last[1];
    asm volatile("" : "+s"(counted));                    // (or it is asked for when the others have come)
    const int n_tiles = (last_expert < 0) & (last_rows == MOE_COUNTED) ? min(counted, max_tiles) : max_tiles;
    if ((int)(tile >= (unsigned)n_tiles) | (expert < 0) | (row0 < 0) | (rows < 1)) return;
    slot = row0 + min(c, rows - 1);
    live = c < rows;
    entry = entry_of_slot ? entry_of_slot[slot] : 0;
    }
    if (!DIRECT || !(own_rows & 2)) ask_weights(run_lo);
    if constexpr (!DIRECT) arow = A + (size_t)(gather_div ? entry / gather_div : slot) * a_ld;
    if (!DIRECT || !(own_rows & 1)) ask_rows(run_lo);
    const float limit = GATED && gate.limits ? gate.limits[expert] : 0.f;
    const float sw = GATED && !DIRECT ? moe_slot_weight(gate, entry_of_slot, slot) : 1.f;
    const size_t out_row = DIRECT ? entry : row0 + c;
    f32x4 acc[RT];
#pragma unroll
    for (int t = 0; t < RT; ++t) acc[t] = f32x4{0.f, 0.f, 0.f, 0.f};
    for (int first = run_lo; first < run_hi;) {
        if ((first + U) * 64 > K) {                      // (for the last runs of a K that is no multiple of 64 only)
#pragma unroll
            for (int u = 0; u < U; ++u)
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    const bool in = (first + u) * 64 + g * 16 + h * 8 < K;
                    x[u][h] = in ? x[u][h] : u32x4{0u, 0u, 0u, 0u};
#pragma unroll
                    for (int t = 0; t < RT; ++t) w[t][u][h] = in ? w[t][u][h] : u32x4{0u, 0u, 0u, 0u};
                }
        }
#pragma unroll
        for (int t = 0; t < RT; ++t)
#pragma unroll
            for (int u = 0; u < U; ++u) {
                if (first + u >= run_hi) continue;
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, w[t][u][h]),
                                                                     __builtin_bit_cast(bf16x8, x[u][h]), acc[t], 0, 0, 0);
                }
            }
        first += U;
        if (first < run_hi) {
            ask_weights(first);
            ask_rows(first);
        }
    }
#pragma unroll
    for (int t = 0; t < RT; ++t) moe_part[(wave * RT + t) * WAVE + lane] = make_float4(acc[t][0], acc[t][1], acc[t][2], acc[t][3]);
    __syncthreads();
    auto total = [&](int t, float (&v)[4]) __attribute__((always_inline)) {
        float4 p[MOE_ROWS_WAVES];
#pragma unroll
        for (int q = 0; q < MOE_ROWS_WAVES; ++q) p[q] = moe_part[(min(q, waves - 1) * RT + t) * WAVE + lane];
        v[0] = p[0].x, v[1] = p[0].y, v[2] = p[0].z, v[3] = p[0].w;
#pragma unroll
        for (int q = 1; q < MOE_ROWS_WAVES; ++q)
            if (q < waves) v[0] += p[q].x, v[1] += p[q].y, v[2] += p[q].z, v[3] += p[q].w;
    };
    // a lane holds slot c, outputs 4 g + i of a group
    for (int t = wave; t < GROUPS; t += MOE_ROWS_WAVES) {
        float v[4];
        total(t, v);
        const int n = n0 + t * 16 + 4 * g;
        if constexpr (GATED) {
            float up[4];
            total(t + GROUPS, up);
            if (!live) continue;
#pragma unroll
            for (int i = 0; i < 4; ++i) v[i] = moe_act_fast(sw * v[i], sw * up[i], limit, gate.alpha);
            TOut* dst = out + out_row * (N / 2) + n;
            if (((uintptr_t)out & 7) == 0)               // (N / 2 is a multiple of 32, and the output bfloat16)
                *reinterpret_cast<uint2*>(dst) = make_uint2(f32x2_to_bf16x2(v[0], v[1]), f32x2_to_bf16x2(v[2], v[3]));
            else
                for (int i = 0; i < 4; ++i) store_f32<TOut>(dst, i, v[i]);
        } else if (live) {
#pragma unroll
            for (int i = 0; i < 4; ++i)
                if (n + i < N) store_f32<TOut>(out, out_row * N + n + i, moe_epilogue(v[i], epi));
        }
    }
}

// One tile a block whatever the number of tiles: with four (fewer blocks that share the slots' rows) every form but short rows
// of many experts was slower, by up to 1.4 times (20 slots of 128 experts, 1,024 by 1,024: 9.5 us and 13.6). Runs at once: all
// of a wave up to three, then four where they come out even, or two where a run is a gate row's and an up row's (K of 2,048,
// gated, one slot: four 7.4 us, two 6.8).
template <typename TOut, bool GATED, bool DIRECT = false>
static void launch_rows16(const bf16_t* a, int a_ld, int gather_div, const int32_t* entry_of_slot, const bf16_t* w, TOut* out,
                          const int32_t* tiles, int max_tiles, int n, int k, int epi, const MoeGate& gate, hipStream_t s,
                          int n_experts = 0, int own_rows = 0) {
    constexpr int RT = GATED ? 2 : 1;
    const int runs = (k + 63) / 64, a_wave = (runs + MOE_ROWS_WAVES - 1) / MOE_ROWS_WAVES;
    const int waves = (runs + a_wave - 1) / a_wave;      // (all that have a run: four, or fewer with a short K)
    const int tall = DIRECT ? n_experts : std::min(max_tiles, 32768);
    const dim3 grid((unsigned)(((GATED ? n / 2 : n) + 15) / 16), (unsigned)tall, DIRECT ? 1u : (unsigned)((max_tiles + tall - 1) / tall));
    const size_t lds = (size_t)waves * RT * WAVE * sizeof(float4);
#define ROWS16_U(U)                                                                                                  \
    k_moe_gemm_rows16<TOut, GATED, RT, U, DIRECT><<<grid, waves * 64, lds, s>>>(a, a_ld, gather_div, entry_of_slot, w, out,  \
                                                                        tiles, max_tiles, n, k, epi, gate, own_rows)
    if (a_wave == 1) ROWS16_U(1);
    else if (a_wave == 3) ROWS16_U(3);
    else if (!GATED && a_wave % 4 == 0) ROWS16_U(4);
    else ROWS16_U(2);
#undef ROWS16_U
}

// The products of a step of few tokens straight from the tokens' choices (k_moe_gemm_rows16, DIRECT): without a plan. For few
// experts, as the blocks of those that nobody chose come all the same.
extern "C" int imparo_moe_direct_takes(int n_tokens, int used, int n_experts) {
    return n_tokens >= 1 && n_tokens <= MOE_DIRECT_TOKENS && used >= 1 && used <= MOE_DIRECT_USED && n_experts >= 1 && n_experts <= 24;
}
// ... and where a layer with them is the faster one, its router riding with the norm. That saves two launches, 4 to 6 us; the blocks of
// experts that nobody chose, which grow with all experts' weights, cost more than that past some size. Norm, router, choice, both products
// and the next norm in us, planned | so: 9 experts of 768 by 1,024, five a token, 1 token 25.2 | 21.3, 8 tokens 31.6 | 25.2; 16 of 2,048 by
// 1,024, four, 8 tokens 43.7 | 38.8, of 4,096 by 1,024 16 tokens 76.0 | 80.7; 8 of 1,408 by 2,048, four, 1 token 36.1 | 35.8, 16 of 1,024
// by 2,048 31.0 | 33.2. Of 864 forms with up to 16 experts none that goes this way is more than 1 % slower.
extern "C" int imparo_moe_direct_pays(int n_tokens, int used, int n_experts, int width, int hidden) {
    const long long all = (long long)n_experts * width * hidden;
    return n_tokens * used <= 2 || (width <= 1024 ? all <= 32LL << 20 : all < 24LL << 20);
}

// own_rows: row t of `a` is read for every entry of token t, else row t * used + j for its j-th; out has a row an entry.
extern "C" int imparo_moe_gemm_direct(const void* a, int a_ld, int own_rows, const int32_t* choice, int n_tokens, int used,
                                      int n_experts, const void* w, void* out, int out_dtype, int n, int k, int epilogue,
                                      const float* limits, float alpha, imparo_stream stream) {
    if (!a || !choice || !w || !out || n < 1 || k < 8 || k % 8 || a_ld < k || a_ld % 8) return IMPARO_BAD_ARGUMENT;
    if (!imparo_moe_direct_takes(n_tokens, used, n_experts) || ((uintptr_t)a | (uintptr_t)w) % 16) return IMPARO_BAD_ARGUMENT;
    if (epilogue < MOE_EPI_NONE || epilogue > MOE_EPI_GATED) return IMPARO_BAD_ARGUMENT;
    hipStream_t s = (hipStream_t)stream;
    const MoeGate gate{limits, alpha, nullptr, 0};
    const int flags = (own_rows ? 1 : 0) | (n_tokens * used >= 4 * n_experts ? 2 : 0);
    if (epilogue == MOE_EPI_GATED) {
        if (out_dtype != IMPARO_BF16 || n % 64) return IMPARO_BAD_ARGUMENT;
        launch_rows16<bf16_t, true, true>((const bf16_t*)a, a_ld, used, nullptr, (const bf16_t*)w, (bf16_t*)out, choice, n_tokens, n, k,
                                          epilogue, gate, s, n_experts, flags);
    } else if (out_dtype == IMPARO_F32) {
        launch_rows16<float, false, true>((const bf16_t*)a, a_ld, used, nullptr, (const bf16_t*)w, (float*)out, choice, n_tokens, n, k,
                                          epilogue, gate, s, n_experts, flags);
    } else {
        return IMPARO_BAD_ARGUMENT;
    }
    return launch_status();
}

// The same in float32: a tile of 64 slots by 64 outputs, K in steps of 16 through LDS, every output
// summed over k = 0, 1, 2, ... by fused multiply-adds, whatever the tile holds beside it.
__global__ __launch_bounds__(256) void k_moe_gemm_f32(const float* __restrict__ A, int a_ld, int gather_div,
                                                      const int32_t* __restrict__ entry_of_slot,
                                                      const float* __restrict__ W, float* __restrict__ out,
                                                      const int32_t* __restrict__ tiles, int N, int K, int epi) {
    constexpr int TM = 64, TN = 64, BK = 16, LD = 68;
    __shared__ float As[BK][LD], Bs[BK][LD];
    const int expert = tiles[3 * blockIdx.x];
    if (expert < 0) return;
    const int row0 = tiles[3 * blockIdx.x + 1], rows = tiles[3 * blockIdx.x + 2];
    const int n0 = blockIdx.y * TN;
    const int tid = threadIdx.x, ty = tid >> 4, tx = tid & 15;
    const float* Wb = W + (size_t)expert * N * K;
    const float* pa[4];
    const float* pb[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const int r = (tid >> 4) + 16 * j;
        const int slot = row0 + min(r, rows - 1);
        const int src = gather_div ? entry_of_slot[slot] / gather_div : slot;
        pa[j] = A + (size_t)src * a_ld;
        pb[j] = Wb + (size_t)min(n0 + r, N - 1) * K;
    }
    float acc[4][4];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] = 0.f;
    for (int k0 = 0; k0 < K; k0 += BK) {
        const int k = k0 + tx;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            As[tx][(tid >> 4) + 16 * j] = k < K ? pa[j][k] : 0.f;
            Bs[tx][(tid >> 4) + 16 * j] = k < K ? pb[j][k] : 0.f;
        }
        __syncthreads();
#pragma unroll
        for (int kk = 0; kk < BK; ++kk) {
            float a[4], b[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) a[i] = As[kk][ty * 4 + i];
#pragma unroll
            for (int j = 0; j < 4; ++j) b[j] = Bs[kk][tx * 4 + j];
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int j = 0; j < 4; ++j) acc[i][j] = fmaf(a[i], b[j], acc[i][j]);
        }
        __syncthreads();
    }
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int m = ty * 4 + i, n = n0 + tx * 4 + j;
            if (m < rows && n < N) out[(size_t)(row0 + m) * N + n] = moe_epilogue(acc[i][j], epi);
        }
}

extern "C" int imparo_moe_gemm(const void* a, int a_ld, int gather_div, const int32_t* entry_of_slot, const void* w,
                               void* out, int out_dtype, int dtype, const int32_t* tiles, int max_tiles, int tile_rows,
                               int n, int k, int epilogue, const float* limits, float alpha, const float* entry_weight,
                               int n_entries, imparo_stream stream) {
    if (!a || !w || !out || !tiles || max_tiles < 0 || n < 1 || k < 1 || a_ld < k || gather_div < 0)
        return IMPARO_BAD_ARGUMENT;
    if (gather_div && !entry_of_slot) return IMPARO_BAD_ARGUMENT;
    if (epilogue < MOE_EPI_NONE || epilogue > MOE_EPI_GATED) return IMPARO_BAD_ARGUMENT;
    if (epilogue == MOE_EPI_GATED && (dtype != IMPARO_BF16 || out_dtype != IMPARO_BF16 || n % 64 || (entry_weight && !entry_of_slot)))
        return IMPARO_BAD_ARGUMENT;
    if (max_tiles == 0) return IMPARO_OK;
    hipStream_t s = (hipStream_t)stream;
    const MoeGate gate{limits, alpha, entry_weight, n_entries};
    if (dtype == IMPARO_F32) {
        if (out_dtype != IMPARO_F32 || tile_rows != 64) return IMPARO_BAD_ARGUMENT;
        k_moe_gemm_f32<<<dim3(max_tiles, (n + 63) / 64), 256, 0, s>>>((const float*)a, a_ld, gather_div, entry_of_slot,
                                                                     (const float*)w, (float*)out, tiles, n, k, epilogue);
        return launch_status();
    }
    if (dtype != IMPARO_BF16 || k % 8 || a_ld % 8 || ((uintptr_t)a | (uintptr_t)w) % 16) return IMPARO_BAD_ARGUMENT;
#define MOE_LAUNCH(WM, WN, TO)                                                                                       \
    k_moe_gemm_bf16<WM, WN, TO><<<dim3(max_tiles, (n + 64 * WN - 1) / (64 * WN)), 256, 0, s>>>(                      \
        (const bf16_t*)a, a_ld, gather_div, entry_of_slot, (const bf16_t*)w, (TO*)out, tiles, n, k, epilogue)
#define MOE_LAUNCH_GATED(WM)                                                                                         \
    k_moe_gemm_bf16<WM, 2, bf16_t, true><<<dim3(max_tiles, (n + 127) / 128), 256, 0, s>>>(                           \
        (const bf16_t*)a, a_ld, gather_div, entry_of_slot, (const bf16_t*)w, (bf16_t*)out, tiles, n, k, epilogue, gate)
    // Tiles of 128 rows whose K comes in the steps that go straight into LDS: where 256 columns a tile leave no more than a
    // quarter of the columns empty beside tiles of 128, and cost no more rounds of the CUs (256 blocks of these at once, 512
    // of the others; a round of these is the shorter one by a quarter and more). 8,192 slots of 8 experts, 896 columns, K = 512: 2
    // rounds 25.6 us, the other kernel's one 21.6; 32,768 slots, 5 rounds 65, the others' 4 73. From K = 128 on: with 64 there
    // is nothing to keep in flight (8,192 slots, 1,024 columns 16.8 us, 16.0).
    const int tiles_n = (n + MOE_DMA_N - 1) / MOE_DMA_N, narrow_n = (n + 127) / 128;
    const long long blocks = ((long long)max_tiles * tiles_n + 7) / 8 * 8;
    const long long rounds = ((long long)max_tiles * tiles_n + 255) / 256, narrow_rounds = ((long long)max_tiles * narrow_n + 511) / 512;
    if (tile_rows == 128 && k % MOE_DMA_BK == 0 && k > MOE_DMA_BK && 4 * tiles_n * MOE_DMA_N <= 5 * narrow_n * 128 &&
        4 * rounds <= 5 * narrow_rounds && blocks < (1LL << 23)) {       // (a launch holds fewer than 2^32 threads along x)
#define MOE_LAUNCH_DMA(TO, G)                                                                                        \
    do {                                                                                                             \
        if (hipFuncSetAttribute((const void*)k_moe_gemm_dma<TO, G>, hipFuncAttributeMaxDynamicSharedMemorySize,      \
                                MOE_DMA_LDS) != hipSuccess)                                                          \
            return IMPARO_LAUNCH_FAILED;                                                                             \
        k_moe_gemm_dma<TO, G><<<(unsigned)blocks, 512, MOE_DMA_LDS, s>>>(                                            \
            (const bf16_t*)a, a_ld, gather_div, entry_of_slot, (const bf16_t*)w, (TO*)out, tiles, max_tiles, tiles_n, n, k, \
            epilogue, gate);                                                                                         \
    } while (0)
        if (epilogue == MOE_EPI_GATED) MOE_LAUNCH_DMA(bf16_t, true);
        else if (out_dtype == IMPARO_BF16) MOE_LAUNCH_DMA(bf16_t, false);
        else if (out_dtype == IMPARO_F32) MOE_LAUNCH_DMA(float, false);
        else return IMPARO_BAD_ARGUMENT;
#undef MOE_LAUNCH_DMA
        return launch_status();
    }
    if (epilogue == MOE_EPI_GATED) {
        if (tile_rows == 16)
            launch_rows16<bf16_t, true>((const bf16_t*)a, a_ld, gather_div, entry_of_slot, (const bf16_t*)w, (bf16_t*)out, tiles,
                                        max_tiles, n, k, epilogue, gate, s);
        else if (tile_rows == 64) MOE_LAUNCH_GATED(1);
        else if (tile_rows == 128) MOE_LAUNCH_GATED(2);
        else return IMPARO_BAD_ARGUMENT;
    } else if (tile_rows == 16) {
        if (out_dtype == IMPARO_BF16)
            launch_rows16<bf16_t, false>((const bf16_t*)a, a_ld, gather_div, entry_of_slot, (const bf16_t*)w, (bf16_t*)out, tiles,
                                         max_tiles, n, k, epilogue, gate, s);
        else if (out_dtype == IMPARO_F32)
            launch_rows16<float, false>((const bf16_t*)a, a_ld, gather_div, entry_of_slot, (const bf16_t*)w, (float*)out, tiles,
                                        max_tiles, n, k, epilogue, gate, s);
        else
            return IMPARO_BAD_ARGUMENT;
    } else if (tile_rows == 128) {
        if (out_dtype == IMPARO_BF16) MOE_LAUNCH(2, 2, bf16_t);
        else if (out_dtype == IMPARO_F32) MOE_LAUNCH(2, 2, float);
        else return IMPARO_BAD_ARGUMENT;
    } else if (tile_rows == 64) {
        if (n >= 128) {
            if (out_dtype == IMPARO_BF16) MOE_LAUNCH(1, 2, bf16_t);
            else if (out_dtype == IMPARO_F32) MOE_LAUNCH(1, 2, float);
            else return IMPARO_BAD_ARGUMENT;
        } else {
            if (out_dtype == IMPARO_BF16) MOE_LAUNCH(1, 1, bf16_t);
            else if (out_dtype == IMPARO_F32) MOE_LAUNCH(1, 1, float);
            else return IMPARO_BAD_ARGUMENT;
        }
    } else {
        return IMPARO_BAD_ARGUMENT;
    }
#undef MOE_LAUNCH
#undef MOE_LAUNCH_GATED
    return launch_status();
}

// ---------------------------------------------------------------- gated experts
// hidden[slot, j] = act(w g, w u) with g = gu[slot, j], u = gu[slot, half + j] (an expert's gate and up
// rows stacked in one product) and w the weight of the slot's entry (null: 1): an expert without biases that
// reads w * h has w times the products of h. Columns j >= ff (a hidden width filled up for the product
// that follows) hold zeros in gu already and give zeros. With limits the bound is that of the slot's expert, choice[entry
// of the slot].
template <typename TOut, int V>
__global__ void k_moe_gated(const float* __restrict__ gu, MoeGate gate, const int32_t* __restrict__ entry_of_slot,
                            const int32_t* __restrict__ choice, int n_experts, TOut* __restrict__ hidden, int half,
                            long long total) {
    const long long i = ((long long)blockIdx.x * blockDim.x + threadIdx.x) * V;
    if (i >= total) return;
    const long long slot = i / half;
    const int j = (int)(i - slot * half);
    const float w = moe_slot_weight(gate, entry_of_slot, (int)slot);
    const float alpha = gate.alpha;
    float limit = 0.f;
    if (gate.limits) {
        const int e = entry_of_slot[slot];          // a row behind the last slot names no entry
        limit = gate.limits[(e >= 0 && e < gate.n_entries) ? min(max(choice[e], 0), n_experts - 1) : 0];
    }
    const float* pg = gu + slot * 2 * half + j;
    if constexpr (V == 4) {
        const float4 g = *reinterpret_cast<const float4*>(pg), u = *reinterpret_cast<const float4*>(pg + half);
        const float y[4] = {moe_act(w * g.x, w * u.x, limit, alpha), moe_act(w * g.y, w * u.y, limit, alpha),
                            moe_act(w * g.z, w * u.z, limit, alpha), moe_act(w * g.w, w * u.w, limit, alpha)};
        if constexpr (sizeof(TOut) == 2)
            *reinterpret_cast<uint2*>(hidden + i) = make_uint2(f32x2_to_bf16x2(y[0], y[1]), f32x2_to_bf16x2(y[2], y[3]));
        else
            *reinterpret_cast<float4*>(hidden + i) = make_float4(y[0], y[1], y[2], y[3]);
    } else {
        store_f32<TOut>(hidden, (size_t)i, moe_act(w * pg[0], w * pg[half], limit, alpha));
    }
}

// n_slots: the entries that got a slot are the first ones of gu and hidden; where some entries have none
// (experts past the last real one) the rows behind the last slot are computed from whatever gu holds and
// never read.
extern "C" int imparo_moe_gated(const float* gu, const float* weight, const int32_t* entry_of_slot, const int32_t* choice,
                                const float* limits, int n_experts, float alpha, void* hidden, int out_dtype, int n_slots,
                                int half, imparo_stream stream) {
    if (!gu || !hidden || n_slots < 0 || half < 1 || (weight && !entry_of_slot)) return IMPARO_BAD_ARGUMENT;
    if (limits && (!entry_of_slot || !choice || n_experts < 1)) return IMPARO_BAD_ARGUMENT;
    const MoeGate gate{limits, alpha, weight, n_slots};
    if (out_dtype != IMPARO_F32 && out_dtype != IMPARO_BF16) return IMPARO_BAD_ARGUMENT;
    if (n_slots == 0) return IMPARO_OK;
    const long long total = (long long)n_slots * half;
    const bool four = half % 4 == 0 && !(((uintptr_t)gu | (uintptr_t)hidden) & 15);
    const long long n = four ? total / 4 : total;
    const int threads = n <= 16384 ? 64 : 256;                  // few values: over more CUs
    const unsigned blocks = (unsigned)((n + threads - 1) / threads);
    hipStream_t s = (hipStream_t)stream;
#define MOE_GATED(T, V)                                                                                              \
    k_moe_gated<T, V><<<blocks, threads, 0, s>>>(gu, gate, entry_of_slot, choice, n_experts, (T*)hidden, half, total)
    if (out_dtype == IMPARO_F32) {
        if (four) MOE_GATED(float, 4);
        else MOE_GATED(float, 1);
    } else {
        if (four) MOE_GATED(bf16_t, 4);
        else MOE_GATED(bf16_t, 1);
    }
#undef MOE_GATED
    return launch_status();
}

// ---------------------------------------------------------------- combine
// out[t] = sum over the token's choices, in their order, of weight * (the expert's row, or for an
// expert past the last real one the token's input).
template <typename T>
__global__ void k_moe_combine(const float* __restrict__ y, const T* __restrict__ h, const int32_t* __restrict__ choice,
                              const float* __restrict__ weight, const int32_t* __restrict__ slot_of_entry,
                              float* __restrict__ out, int width, int top, int n_experts) {
    const int t = blockIdx.x;
    __shared__ int slot[MOE_MAX_USED];
    __shared__ float w[MOE_MAX_USED];
    if (threadIdx.x < top) {
        const int e = choice[(size_t)t * top + threadIdx.x];
        slot[threadIdx.x] = e < n_experts ? slot_of_entry[(size_t)t * top + threadIdx.x] : -1;
        w[threadIdx.x] = weight ? weight[(size_t)t * top + threadIdx.x] : 1.0f;
    }
    __syncthreads();
    for (int i = threadIdx.x; i < width; i += blockDim.x) {
        float acc = 0.f;
        for (int k = 0; k < top; ++k) {
            const float v = slot[k] >= 0 ? y[(size_t)slot[k] * width + i] : load_f32<T>(h, (size_t)t * width + i);
            acc = fmaf(w[k], v, acc);
        }
        out[(size_t)t * width + i] = acc;
    }
}

extern "C" int imparo_moe_combine(const float* y, const void* h, int h_dtype, const int32_t* choice,
                                  const float* weight, const int32_t* slot_of_entry, float* out, int n_tokens,
                                  int width, int top, int n_experts, imparo_stream stream) {
    if (!y || !h || !choice || !slot_of_entry || !out || n_tokens < 0 || width < 1) return IMPARO_BAD_ARGUMENT;
    if (top < 1 || top > MOE_MAX_USED || n_experts < 0) return IMPARO_BAD_ARGUMENT;
    if (n_tokens == 0) return IMPARO_OK;
    hipStream_t s = (hipStream_t)stream;
    const int threads = width >= 1024 ? 256 : 64;
    if (h_dtype == IMPARO_F32)
        k_moe_combine<float><<<n_tokens, threads, 0, s>>>(y, (const float*)h, choice, weight, slot_of_entry, out, width,
                                                          top, n_experts);
    else if (h_dtype == IMPARO_BF16)
        k_moe_combine<bf16_t><<<n_tokens, threads, 0, s>>>(y, (const bf16_t*)h, choice, weight, slot_of_entry, out,
                                                           width, top, n_experts);
    else
        return IMPARO_BAD_ARGUMENT;
    return launch_status();
}

// ---------------------------------------------------------------- a norm on what a sublayer returns
// x[row] += d / sqrt(mean(d^2) + eps_post) * w_post, d = the sum of the delta's slices in order; then,
// with w_next, out[row] = x[row] / sqrt(mean(x[row]^2) + eps_next) * w_next. One block a row, the row in
// registers between the passes, every sum in float32 and in an order that the width alone decides. With `rows`
// only those rows are taken and the stream is left as it is (the rows whose logits are wanted).
// PER: values of the row a thread keeps in registers (the block's threads x PER cover the width); every
// load of the row (the delta's slices, the stream, both weights) is asked for before any is used.
// What a routed feed-forward leaves for this launch to combine instead of a finished delta: the experts'
// rows y [slots, width], the feed-forward's input h (for experts that pass it through), and per token its
// choice, weights and slots. delta[t] = sum_j weight[t, j] * (y[slot] or h[t]), j in the order of the choice.
struct MoeRows {
    const float* y;
    const void* h;
    const int32_t* choice;
    const float* weight;
    const int32_t* slot_of_entry;
    int h_is_bf16, top, n_experts;
};

template <typename TOut, int PER>
__global__ __launch_bounds__(256) void k_post_norm_add(float* __restrict__ x, const float* __restrict__ delta,
                                                       int n_delta, size_t delta_stride, MoeRows moe,
                                                       const int32_t* __restrict__ rows,
                                                       const float* __restrict__ w_post, float eps_post,
                                                       const float* __restrict__ w_next, float eps_next,
                                                       TOut* __restrict__ out, int width, int write_back) {
    __shared__ float scratch[16];
    const int i_out = blockIdx.x;
    const size_t src = (size_t)(rows ? rows[i_out] : i_out) * width;
    float d[PER], xv[PER], wp[PER], wn[PER];
    if (moe.y) {
        __shared__ int slot[MOE_MAX_USED];
        __shared__ float wt[MOE_MAX_USED];
        const size_t t = src / width;
        if ((int)threadIdx.x < moe.top) {
            const int e = moe.choice[t * moe.top + threadIdx.x];
            slot[threadIdx.x] = e < moe.n_experts ? moe.slot_of_entry[t * moe.top + threadIdx.x] : -1;
            wt[threadIdx.x] = moe.weight[t * moe.top + threadIdx.x];
        }
        __syncthreads();
#pragma unroll
        for (int j = 0; j < PER; ++j) d[j] = 0.f;
        for (int k = 0; k < moe.top; ++k) {
            const int sl = slot[k];
            const float w = wt[k];
#pragma unroll
            for (int j = 0; j < PER; ++j) {
                const int ii = min((int)threadIdx.x + j * 256, width - 1);
                const float v = sl >= 0 ? moe.y[(size_t)sl * width + ii]
                                        : (moe.h_is_bf16 ? load_f32<bf16_t>((const bf16_t*)moe.h, src + ii)
                                                         : load_f32<float>((const float*)moe.h, src + ii));
                d[j] = fmaf(w, v, d[j]);
            }
        }
    }
#pragma unroll
    for (int j = 0; j < PER; ++j) {
        const int i = threadIdx.x + j * 256;
        const int ii = min(i, width - 1);
        if (!moe.y) d[j] = delta[src + ii];
        xv[j] = x[src + ii];
        wp[j] = w_post[ii];
        wn[j] = w_next ? w_next[ii] : 0.f;
    }
    for (int s = 1; s < n_delta && !moe.y; ++s)
#pragma unroll
        for (int j = 0; j < PER; ++j) d[j] += delta[(size_t)s * delta_stride + src + min((int)threadIdx.x + j * 256, width - 1)];
    float ss = 0.f;
#pragma unroll
    for (int j = 0; j < PER; ++j)
        if (threadIdx.x + j * 256 < width) ss = fmaf(d[j], d[j], ss);
    const float r1 = 1.0f / sqrtf(block_sum(ss, scratch) / (float)width + eps_post);
    ss = 0.f;
#pragma unroll
    for (int j = 0; j < PER; ++j) {
        const int i = threadIdx.x + j * 256;
        xv[j] = xv[j] + d[j] * r1 * wp[j];
        if (i < width) {
            if (write_back) x[src + i] = xv[j];
            ss = fmaf(xv[j], xv[j], ss);
        }
    }
    if (!w_next) {
        // no norm follows: with an output, the new rows themselves go there in its dtype
        if (out)
#pragma unroll
            for (int j = 0; j < PER; ++j) {
                const int i = threadIdx.x + j * 256;
                if (i < width) store_f32<TOut>(out, (size_t)i_out * width + i, xv[j]);
            }
        return;
    }
    const float r2 = 1.0f / sqrtf(block_sum(ss, scratch) / (float)width + eps_next);
#pragma unroll
    for (int j = 0; j < PER; ++j) {
        const int i = threadIdx.x + j * 256;
        if (i < width) store_f32<TOut>(out, (size_t)i_out * width + i, xv[j] * r2 * wn[j]);
    }
}

static int post_norm_add_launch(float* x, const float* delta, int n_delta, MoeRows moe, int n_rows_x,
                                const int32_t* rows, const float* w_post, float eps_post, const float* w_next,
                                float eps_next, void* out, int out_dtype, int n_out, int width, imparo_stream stream) {
    if (!x || (!delta && !moe.y) || !w_post || n_delta < 1 || n_rows_x < 0 || n_out < 0 || width < 1 || width > 16384)
        return IMPARO_BAD_ARGUMENT;
    if (w_next && !out) return IMPARO_BAD_ARGUMENT;
    if (!rows && n_out != n_rows_x) return IMPARO_BAD_ARGUMENT;
    if (n_out == 0) return IMPARO_OK;
    hipStream_t s = (hipStream_t)stream;
    const size_t stride = (size_t)n_rows_x * width;
    const int write_back = rows ? 0 : 1;
    const bool to_bf16 = out && out_dtype == IMPARO_BF16;
    if (out && out_dtype != IMPARO_BF16 && out_dtype != IMPARO_F32) return IMPARO_BAD_ARGUMENT;
#define POST_NORM(PER)                                                                                              \
    if (to_bf16)                                                                                                    \
        k_post_norm_add<bf16_t, PER><<<n_out, 256, 0, s>>>(x, delta, n_delta, stride, moe, rows, w_post, eps_post,  \
                                                           w_next, eps_next, (bf16_t*)out, width, write_back);      \
    else                                                                                                            \
        k_post_norm_add<float, PER><<<n_out, 256, 0, s>>>(x, delta, n_delta, stride, moe, rows, w_post, eps_post,   \
                                                          w_next, eps_next, (float*)out, width, write_back)
    const int per = (width + 255) / 256;
    if (per <= 1) { POST_NORM(1); }
    else if (per <= 2) { POST_NORM(2); }
    else if (per <= 4) { POST_NORM(4); }
    else if (per <= 8) { POST_NORM(8); }
    else if (per <= 16) { POST_NORM(16); }
    else if (per <= 32) { POST_NORM(32); }
    else { POST_NORM(64); }
#undef POST_NORM
    return launch_status();
}

extern "C" int imparo_post_norm_add(float* x, const float* delta, int n_delta, int n_rows_x, const int32_t* rows,
                                    const float* w_post, float eps_post, const float* w_next, float eps_next,
                                    void* out, int out_dtype, int n_out, int width, imparo_stream stream) {
    return post_norm_add_launch(x, delta, n_delta, MoeRows{}, n_rows_x, rows, w_post, eps_post, w_next, eps_next, out,
                                out_dtype, n_out, width, stream);
}

// The same with the delta made in the launch from a routed feed-forward's rows (imparo_moe_combine's sum).
extern "C" int imparo_post_norm_add_moe(float* x, const float* y, const void* h, int h_dtype, const int32_t* choice,
                                        const float* weight, const int32_t* slot_of_entry, int top, int n_experts,
                                        int n_rows_x, const int32_t* rows, const float* w_post, float eps_post,
                                        const float* w_next, float eps_next, void* out, int out_dtype, int n_out,
                                        int width, imparo_stream stream) {
    if (!y || !h || !choice || !weight || !slot_of_entry || top < 1 || top > MOE_MAX_USED || n_experts < 0)
        return IMPARO_BAD_ARGUMENT;
    if (h_dtype != IMPARO_F32 && h_dtype != IMPARO_BF16) return IMPARO_BAD_ARGUMENT;
    const MoeRows moe{y, h, choice, weight, slot_of_entry, h_dtype == IMPARO_BF16, top, n_experts};
    return post_norm_add_launch(x, nullptr, 1, moe, n_rows_x, rows, w_post, eps_post, w_next, eps_next, out, out_dtype,
                                n_out, width, stream);
}

int imparo_load_code_moe() {
    hipFuncAttributes attributes;
    return hipFuncGetAttributes(&attributes, reinterpret_cast<const void*>(&k_moe_plan)) == hipSuccess ? IMPARO_OK
                                                                                                       : IMPARO_LAUNCH_FAILED;
}
