"""What tells a map of the running call from one that an earlier call left in the same memory (map_tag, map_check in
csrc/gae_norm.hip): the two functions, compiled for the host. A map's six words can be seen half old, half new, and half of a call's number
is in a word's tag, so two calls with the same half are met once in 2^32 pairs; the words that carry it fit then."""

import re
import subprocess

import pytest

from areal_amd import build

DRIVER = """
#include <cstdint>
#include <cstdio>
#define DEVI static inline
struct MapF { float a11, a12, a22, b1, b2; };
%s
struct Words { uint64_t w[6]; };
static Words of(uint64_t call, const MapF& m) {
  const float x[5] = {m.a11, m.a12, m.a22, m.b1, m.b2};
  Words r;
  for (int k = 0; k < 6; ++k)
    r.w[k] = (uint64_t)map_tag(call, k) << 32 | (k == 5 ? map_check(%s) : __builtin_bit_cast(uint32_t, x[k]));
  return r;
}
static bool fits(uint64_t call, const Words& r) {  // as gather_tile_maps
  for (int k = 0; k < 6; ++k)
    if ((uint32_t)(r.w[k] >> 32) != map_tag(call, k)) return false;
  auto f = [&](int k) { return __builtin_bit_cast(float, (uint32_t)r.w[k]); };
  const MapF m{f(0), f(1), f(2), f(3), f(4)};
  return (uint32_t)r.w[5] == map_check(%s);
}
int main() {
  uint64_t z = 88172645463325252ull;
  auto next = [&] { z ^= z << 13; z ^= z >> 7; z ^= z << 17; return z; };
  int wrong = 0, own = 0;
  for (int i = 0; i < 200000; ++i) {
    const uint64_t call = next(), other = next();
    // the same mask and discount, no values: two maps that differ in b1 alone, or in any of their numbers
    MapF now{0.5f, 0.f, 0.f, (float)(int32_t)next(), 0.f}, before = now;
    before.b1 = (float)(int32_t)next();
    if (i & 1) { before.a11 = (float)(int32_t)next(); before.a22 = (float)(int32_t)next(); }
    if (before.b1 == now.b1) continue;
    own += fits(call, of(call, now));
    for (int half = 0; half < 2; ++half) {
      const uint64_t keep = half ? 0xffffffff00000000ull : 0xffffffffull;
      const uint64_t old = (call & keep) | (other & ~keep);
      if (old == call) continue;
      for (int mask = 0; mask < 63; ++mask) {  // which words are the running call's
        Words r = of(old, before);
        const Words n = of(call, now);
        for (int k = 0; k < 6; ++k)
          if (mask >> k & 1) r.w[k] = n.w[k];
        if (!fits(call, r)) continue;
        auto same = [&] { for (int k = 0; k < 5; ++k) if ((uint32_t)r.w[k] != (uint32_t)n.w[k]) return false; return true; };
        wrong += !same();
      }
    }
  }
  printf("%%d %%d\\n", own, wrong);
}
"""


def test_a_map_of_an_earlier_call_is_told_by_more_than_half_of_its_number(tmp_path):
    try:
        compiler = build._hipcc()
    except RuntimeError:
        pytest.skip("no hipcc")
    source = (build.CSRC / "gae_norm.hip").read_text()
    functions = [re.search(rf"^DEVI uint32_t {name}\(.*?^}}", source, re.S | re.M).group(0) if name == "map_check" else
                 re.search(rf"^DEVI uint32_t {name}\(.*$", source, re.M).group(0) for name in ("map_tag", "map_check")]
    args = "call, m" if "uint64_t call, const MapF" in functions[1] else "m"
    (tmp_path / "maps.cpp").write_text(DRIVER % ("\n".join(functions), args, args))
    subprocess.run([compiler, "-x", "c++", "-std=c++17", "-O2", str(tmp_path / "maps.cpp"), "-o", str(tmp_path / "maps")], check=True)
    own, wrong = map(int, subprocess.run([tmp_path / "maps"], check=True, capture_output=True, text=True).stdout.split())
    # 25 million half-new maps of calls that share a half, each with a chance of 2^-32 left
    assert own > 199000 and wrong <= 1
