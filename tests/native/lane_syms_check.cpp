// The tables by which a wavefront's lanes find a chain's symbol (LaneSyms of
// bigsmall_amd/csrc/refcodec_decode.hip), checked lane by lane against the plain
// decode step: the CPU runs of the kernels find symbols by another search, so
// only this and the GPU tests see these fields. For every slot exactly one lane's
// interval may hold it, and that lane's symbol, next state and need of a word must
// be the plain step's, for states at both ends of every slot's range and of its
// renormalisation bound. Prints the number of checks; exit status 0 when all hold.
#include "refcodec_decode.hip"

#include <stdio.h>

#include <random>
#include <vector>

namespace {

template <int R, bool SE>
bool check(const std::vector<uint32_t>& freq, uint64_t& checks) {
  constexpr uint32_t kLog = SE ? 12u : 10u, kTop = 32u - kLog, kM = 1u << kLog;
  std::vector<u32x2> list;
  std::vector<uint32_t> sym_of(kM), cf_of;
  uint32_t cf = 0;
  for (uint32_t f : freq) {
    for (uint32_t i = 0; i < f; ++i) sym_of[cf + i] = (uint32_t)list.size();
    u32x2 e;
    e.x = f | (cf << 16);
    e.y = 0;
    list.push_back(e);
    cf_of.push_back(cf);
    cf += f;
  }
  const uint32_t live = (uint32_t)list.size();
  std::vector<LaneSyms<R, SE>> lanes(kWave);
  for (uint32_t l = 0; l < (uint32_t)kWave; ++l) lanes[l].load((const LDS u32x2*)list.data(), live, l);
  for (uint32_t slot = 0; slot < kM; ++slot) {
    const uint32_t s = sym_of[slot], f = freq[s];
    // the slot's states that just do and just do not renormalise, and its ends
    const uint64_t edge = (((uint64_t)kL + f - 1) / f) << kLog;
    for (uint64_t base : {(uint64_t)kL, edge - kM, edge, edge + kM, ((uint64_t)1 << 32) - kM}) {
      const uint64_t xs = (base & ~(uint64_t)(kM - 1)) | slot;
      if (xs < kL || xs > 0xFFFFFFFFull) continue;
      const uint32_t x = (uint32_t)xs, h = x >> kLog;
      const uint32_t want = f * h + slot - cf_of[s];
      uint32_t hits = 0;
      for (uint32_t l = 0; l < (uint32_t)kWave; ++l) {
        const LaneSyms<R, SE>& S = lanes[l];
        const uint32_t t = (x << kTop) + S.first;
        if (t > S.last) continue;
        ++hits;
        const int r = R == 2 && t >= S.begin[R - 1] ? 1 : 0;
        const uint32_t c = (uint32_t)__mul24(S.nf[r], (int32_t)h) + (x - S.cf[r]);
        const bool need = S.bound[r] > x;
        if (l * R + r != s || c != want || need != (want < kL)) {
          fprintf(stderr, "R %d SE %d live %u slot %u x %u: lane %u symbol %u (want %u) state %u (want %u) need %d\n", R,
                  SE, live, slot, x, l, l * R + r, s, c, want, need);
          return false;
        }
      }
      if (hits != 1) {
        fprintf(stderr, "R %d SE %d live %u slot %u: %u lanes hold it\n", R, SE, live, slot, hits);
        return false;
      }
      ++checks;
    }
  }
  return true;
}

// `live` frequencies of sum m: all 1 but one, even, or random
std::vector<uint32_t> table(uint32_t live, uint32_t m, uint32_t kind, std::mt19937& rng) {
  std::vector<uint32_t> f(live, kind == 1 ? m / live : 1u);
  uint32_t rest = m;
  for (uint32_t v : f) rest -= v;
  if (kind == 2)
    for (; rest; --rest) ++f[rng() % live];
  f[rng() % live] += rest;
  return f;
}

}  // namespace

int main() {
  std::mt19937 rng(7);
  uint64_t checks = 0;
  for (uint32_t kind = 0; kind < 3; ++kind) {
    for (uint32_t live : {1u, 2u, 3u, 63u, 64u})
      if (!check<1, true>(table(live, 4096, kind, rng), checks)) return 1;
    for (uint32_t live : {1u, 2u, 64u, 65u, 127u, 128u}) {
      if (!check<2, true>(table(live, 4096, kind, rng), checks)) return 1;
      if (!check<2, false>(table(live, 1024, kind, rng), checks)) return 1;
    }
  }
  printf("checks %llu\n", (unsigned long long)checks);
  return 0;
}
