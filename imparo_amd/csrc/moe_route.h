// A token's choice among the outputs of a mixture's router, for the kernels that make it.
#pragma once
#include "common.h"

#define MOE_SCORE_SOFTMAX 0         // scores = softmax over all router outputs
#define MOE_SCORE_SIGMOID 1         // scores = sigmoid of each output
#define MOE_SCORE_CHOSEN 2          // scores = the outputs themselves; a token's weights = softmax over its chosen ones
#define MOE_MAX_USED 24             // experts a token uses: those it chooses and the ones that every token uses

// What a router may do beyond scoring and choosing. logits_ld: floats between two tokens' logits (at least
// n_router; further columns belong to someone else). groups > 1: the router outputs form that many equal
// groups of neighbours, a group's score is the sum of its two largest choice scores (score + correction), and
// only outputs of the `keep` best groups can be chosen (of equal groups the lowest). normalize: the chosen
// scores are divided by their sum + 1e-20. scale: the weights are multiplied by it at the end. always: so many
// experts, numbered behind the router's outputs, are used by every token with weight one; a token's list of experts
// has them behind its `top` chosen ones.
struct MoeRouteRules {
    int logits_ld, groups, keep, normalize;
    float scale;
    int always;
};

// A token's choice among at most 64 outputs without groups: a lane holds one output and counts the ones that come before it (larger,
// or as large with a lower index), so the k-th choice is the lane whose count is k: some five instructions an output
// instead of twelve shuffles a choice, each of which waits for LDS. Same picks, weights and order of addition. 4 of 8
// outputs: 2,048 rows 6.8 -> 3.9 us; 8 rows, with the plan made in the same launch from choices kept in LDS, 7.7 -> 4.1.
// `z`: this lane's output.
__device__ __forceinline__ void moe_route_lanes(float z, const float* __restrict__ correction, int32_t* choice,
                                                float* __restrict__ weight, int t, int n_router, int top, int scoring,
                                                const MoeRouteRules rules, int32_t* choice_too) {
    const int lane = threadIdx.x & (WAVE - 1);
    const int used = top + rules.always;
    choice += (size_t)t * used;
    weight += (size_t)t * used;
    const bool mine = lane < n_router;
    if (!mine) z = -INFINITY;
    const float shift = mine && correction ? correction[lane] : 0.f;
    if (scoring == MOE_SCORE_SIGMOID) {
        z = mine ? 1.0f / (1.0f + expf(-z)) : 0.f;
    } else if (scoring == MOE_SCORE_SOFTMAX) {
        const float m = wave_max(z);
        z = mine ? expf(z - m) : 0.f;
        z *= 1.0f / wave_sum(z);
    }
    const float pick = mine ? z + shift : -INFINITY;
    int before = 0;
    for (int i = 0; i < n_router; ++i) {
        const float other = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(pick), i));
        before += (other > pick || (other == pick && i < lane)) ? 1 : 0;
    }
    const bool valid = pick > -INFINITY;                     // (and no NaN: those are never chosen)
    float chosen_sum = 0.f, chosen_max = -INFINITY, score = -INFINITY;      // score, at: lane k keeps the k-th choice's
    int at = 0x7fffffff;
    for (int k = 0; k < top; ++k) {
        const unsigned long long who = __ballot(valid && before == k);
        const int i = who ? __ffsll((long long)who) - 1 : 0;
        const float s = who ? __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(z), i)) : 0.f;
        chosen_sum += s;
        chosen_max = fmaxf(chosen_max, s);
        if (lane == k) {
            score = s;
            at = who ? i : 0x7fffffff;
        }
    }
    float w = score;
    if (scoring == MOE_SCORE_CHOSEN) {
        const float e = lane < top ? expf(score - chosen_max) : 0.f;
        w = e / wave_sum(e) * rules.scale;
    } else if (rules.normalize || rules.scale != 1.0f) {
        w *= (rules.normalize ? 1.0f / (chosen_sum + 1e-20f) : 1.0f) * rules.scale;
    }
    if (lane < used) {
        const int e = lane < top ? at : n_router + lane - top;
        choice[lane] = e;
        weight[lane] = lane < top ? w : 1.0f;
        if (choice_too) choice_too[(size_t)t * used + lane] = e;
    }
}

__device__ __forceinline__ void moe_route_token_narrow(const float* __restrict__ logits, const float* __restrict__ correction,
                                                       int32_t* choice, float* __restrict__ weight, int t, int n_router, int top,
                                                       int scoring, const MoeRouteRules rules, int32_t* choice_too) {
    const int lane = threadIdx.x & (WAVE - 1);
    const float z = lane < n_router ? logits[(size_t)t * rules.logits_ld + lane] : -INFINITY;
    moe_route_lanes(z, correction, choice, weight, t, n_router, top, scoring, rules, choice_too);
}

// Counting costs by the output, choosing in rounds by the choice: 8,192 rows, counted | in rounds, 64 outputs: the best one 9.8 |
// 7.6 us, two 10.0 | 9.4, four 10.4 | 13.2; 32 outputs: the best one 6.7 | 7.6.
__device__ __forceinline__ bool moe_routes_narrow(int n_router, int top, const MoeRouteRules& rules) {
    return n_router <= WAVE && rules.groups == 1 && (n_router <= 32 || top >= 3);
}
