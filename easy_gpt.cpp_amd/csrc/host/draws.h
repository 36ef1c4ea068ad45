// The uniform numbers of a batch of draws, behind a C ABI.
#pragma once
#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

// out[i]: a number in [0, 1) that is a function of (seeds[i], serials[i], counts[i]) alone, with 24 bits (exact in float32).
void egh_uniforms(int n, const uint64_t* seeds, const uint64_t* serials, const uint64_t* counts, float* out);

#ifdef __cplusplus
}
#endif
