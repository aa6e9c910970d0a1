// The numbers that a step's draws take, one per (request seed, counter): splitmix64's finaliser, 24 random bits in [0, 1),
// as sampler.py: uniform() states them.
//
// And the parameters of a step's rows, from the plans' own packed form (params.py: SamplingPlan.packed): lists of attributes cost
// 64 rows 10 us a step in Python, their numbers another 5, and the GPU waits for both.
#include <cstdint>

namespace {
float uniform(uint64_t seed, uint64_t counter) {
  uint64_t z = seed * 0x9E3779B97F4A7C15ull + (counter + 1) * 0xBF58476D1CE4E5B9ull;
  z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
  z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
  z ^= z >> 31;
  return (float)(z >> 40) * 0x1p-24f;
}

struct PlanRow {               // as SamplingPlan.packed writes it
  float temperature, top_p, penalty;
  int32_t top_k;
  uint64_t seed;
  int32_t greedy, penalised;
};
static_assert(sizeof(PlanRow) == 32, "a plan's bytes");
enum Found : int { kAllGreedy = 1, kPenalised = 2, kTopP = 4, kTopK = 8, kFewK = 16 };
}  // namespace

// meta [5][n]: temperature (0: greedy), top_p, uniform, penalty, top_k (int32 bits).  What the rows that draw ask for, as bits: a
// top-p cut, a top-k cut, top-k cuts of at most few_max all of them.
extern "C" int sampling_pack(const void* plans, const uint64_t* counters, int n, int few_max, float* meta) {
  const PlanRow* const rows = static_cast<const PlanRow*>(plans);
  int32_t* const top_k = reinterpret_cast<int32_t*>(meta + 4 * (long)n);
  int found = kAllGreedy | kFewK;
  for (int i = 0; i < n; ++i) {
    const PlanRow& r = rows[i];
    meta[i] = r.greedy ? 0.f : r.temperature;
    meta[n + i] = r.top_p;
    meta[3 * (long)n + i] = r.penalty;
    top_k[i] = r.top_k;
    meta[2 * (long)n + i] = uniform(r.seed, counters[i]);
    if (r.penalised) found |= kPenalised;
    if (r.greedy) continue;
    found &= ~kAllGreedy;
    if (r.top_p < 1.0f) found |= kTopP;
    if (r.top_k > 0) found |= kTopK;
    if (r.top_k <= 0 || r.top_k > few_max) found &= ~kFewK;
  }
  return found;
}
