// Rules of the one-launch decode step that are plain arithmetic (host only, no HIP): when it pays, and how much memory a step reads.
#pragma once
#include <algorithm>

// Whether one launch is the faster step for `batch` >= 2 sequences of a model of width d behind `ctx` cached positions, with the
// Linear workgroups in `groups` groups: its time per layer against that of five launches, in us.
// One launch: the chain of hand-offs and, sequence by sequence, the role that is busy longest.  The Linear workgroups take 1.2
// (d = 256) to 1.85 (768) per sequence with four groups, 3.8 per 1024 of d with two, 7.2 where all of them take every stage (and then wait for the attention
// as well); the attention workgroups (two per head) next to nothing up to 256 keys, then a second range is waited for.
// Five launches: their gaps, the weights, and an attention that reads the caches at the speed of memory.
// ms per step, five launches / one: 24 x 1024, 2, 4, 6, 8 sequences, 64 cached: 0.75 / 0.34, 0.77 / 0.50, 0.78 / 0.70, 0.79 / 0.89;
// 4 at 600: 0.92 / 0.85, at 900: 0.92 / 1.00; 12 x 768, 8 at 64: 0.36 / 0.30, 4 at 600: 0.47 / 0.39, 5 at 600: 0.46 / 0.48;
// 24 x 1280, 5 at 64: 0.84 / 0.76, 4 at 900: 1.17 / 1.07; 24 x 1600, 2 at 64 .. 900: 0.92 / 0.71 .. 1.03 / 0.94, 3: 0.93 / 0.98 ..
// 1.25 / 1.30; 12 x 256, 8 at 64: 0.28 / 0.23, 3 at 900: 0.31 / 0.29, 4: 0.32 / 0.36.  Of 139 such pairs it picks the slower one, by
// more than 1 %, twice.
// The longer context only ever takes away: what does not pay up to 256 keys is within 1 % beyond, and stays per stage.
inline bool pk_pays_rule(int groups, int d, int heads, int batch, int ctx) {
    const float w = (float)d / 1024.0f, b = (float)batch, keys = (float)ctx;
    const float linear = groups >= 4 ? 0.9f + 1.27f * w : groups == 2 ? 3.8f * w : 7.2f * w;
    const float short_stages = 19.5f + 11.0f * w;
    if (7.0f + b * linear > short_stages) return false;
    if (ctx <= 256) return true;
    const float attention = (2.9f + 0.0062f * keys) * (heads <= 8 ? 0.72f : 1.0f);
    const float busy = groups >= 2 ? std::max(linear, attention) : linear + std::max(0.0f, attention - 4.7f);
    return 7.0f + b * busy <= short_stages + 3.5f + 0.002f * b * (keys - 256.0f);
}

// Bytes of weights that a token reads: int4 weights and scales of 32 each (0.625 a weight); an fp32 head 4.  The head counts as the
// type it has, whether it is in the launch or follows it.
inline double pk_token_bytes(int d, int ff, int n_layer, int vocab, bool head_int4) {
    return (((double)3 * d * d + (double)d * d + 2.0 * d * ff) * n_layer + (head_int4 ? 1.0 : 6.4) * d * vocab) * 0.625;
}

// Whether the relays touch an XCD's share of a half layer's weights one exchange before its use, so that the Linear workgroups'
// requests are served from the L2.  One sequence: where the weights do not stay in the 256 MiB Infinity Cache between steps anyway; a
// smaller model is only slowed down by it (19 x 960, 161 MB: 0.231 -> 0.237 ms per step).  Several sequences with at most two groups of
// Linear workgroups: whatever the size, ms per step without and with: 12 x 1024, 3 sequences 0.229 / 0.220; 8 x 1280, 4: 0.238 / 0.230;
// 19 x 960, 2 at 715 positions: 0.451 / 0.437; 12 x 768, 2: 0.163 / 0.163.  With four groups a workgroup has three stages' time for
// its requests: 12 x 768, 4 sequences 0.195 / 0.203.
inline bool pk_touches_ahead(double token_bytes, int batch, int groups) { return token_bytes > 200.0e6 || (batch > 1 && groups <= 2); }
