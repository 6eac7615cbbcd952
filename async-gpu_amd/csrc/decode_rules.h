// Rules of the one-launch decode step that are plain arithmetic (host only, no HIP).
#pragma once

// Bytes of weights that a token reads: int4 weights and scales of 32 each (0.625 a weight); an fp32 head 4.  The head counts as the
// type it has, whether it is in the launch or follows it.
inline double pk_token_bytes(int d, int ff, int n_layer, int vocab, bool head_int4) {
    return (((double)3 * d * d + (double)d * d + 2.0 * d * ff) * n_layer + (head_int4 ? 1.0 : 6.4) * d * vocab) * 0.625;
}
