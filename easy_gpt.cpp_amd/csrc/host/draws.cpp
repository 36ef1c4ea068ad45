#include "draws.h"

namespace {

// the finaliser of splitmix64
uint64_t mix(uint64_t z) {
    z += 0x9E3779B97F4A7C15ull;
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    return z ^ (z >> 31);
}

}  // namespace

extern "C" void egh_uniforms(int n, const uint64_t* seeds, const uint64_t* serials, const uint64_t* counts, float* out) {
    for (int i = 0; i < n; ++i)
        out[i] = static_cast<float>(mix(mix(mix(seeds[i]) ^ serials[i]) ^ counts[i]) >> 40) * (1.0f / 16777216.0f);
}
