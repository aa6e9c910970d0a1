// The numbers that a step's draws take, one per (request seed, counter): splitmix64's finaliser, 24 random bits in [0, 1),
// as sampler.py: uniform() states them.
#include <cstdint>

extern "C" void sampling_uniforms(const uint64_t* seeds, const uint64_t* counters, int n, float* out) {
  for (int i = 0; i < n; ++i) {
    uint64_t z = seeds[i] * 0x9E3779B97F4A7C15ull + (counters[i] + 1) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    z ^= z >> 31;
    out[i] = (float)(z >> 40) * 0x1p-24f;
  }
}
