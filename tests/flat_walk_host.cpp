// gqa_flat.hpp on the CPU, a wave as an array of 64 lanes: the walks of all
// slots cover every unit once, in order, and agree with the plan; lengths that
// change between two reads leave every walk finite and every partial in the
// workspace.  Prints the number of batches checked.
#include "gqa_flat.hpp"

#include <algorithm>
#include <array>
#include <cstdio>
#include <cstdlib>
#include <random>
#include <vector>

struct HostWave {
  using Lanes = std::array<int, 64>;
  const std::vector<int>* lens;   // units of each sequence
  const std::vector<int>* later;  // ... from the `change`-th read on
  int B, slots, seq_units;
  int change;
  mutable int reads = 0;

  Lanes units(int base, Lanes& keys) const {
    const std::vector<int>& l = reads++ < change ? *lens : *later;
    Lanes u{};
    for (int i = 0; i < 64; ++i) u[i] = base + i < B ? l[base + i] : 0;
    keys = u;
    return u;
  }
  static Lanes scan(Lanes n) {
    for (int i = 1; i < 64; ++i) n[i] += n[i - 1];
    return n;
  }
  static void add(Lanes& a, const Lanes& b) {
    for (int i = 0; i < 64; ++i) a[i] += b[i];
  }
  static int read(const Lanes& v, int l) { return v[l]; }
  static int first_above(const Lanes& v, int x) {
    for (int i = 0; i < 64; ++i)
      if (v[i] > x) return i;
    return -1;
  }
  int share(int n) const { return n / slots; }
  int sequence(int n) const { return n / seq_units; }
  static int own(const Lanes& v, int lane) { return v[lane]; }
  template <typename F> void each(F f) const {
    for (int i = 0; i < 64; ++i) f(i);
  }
};

#define CHECK(c)                                                              \
  if (!(c)) {                                                                 \
    std::printf("%s: B %d slots %d change %d\n", #c, w.B, w.slots, w.change); \
    std::exit(1);                                                             \
  }

template <bool PAGED> void walk_all(const HostWave& w0, const std::vector<int>& lens, bool changing) {
  HostWave w = w0;
  std::vector<int> done(w.B, 0);
  std::vector<std::vector<int>> partials(w.B);
  for (int slot = 0; slot < w.slots; ++slot) {
    w.reads = 0;
    gqa::FlatWalk<HostWave, PAGED> walk;
    walk.start(w, slot);
    int from, cnt, pieces = 0;
    while (walk.next(w, from, cnt)) {
      CHECK(++pieces <= w.B + 1);
      CHECK(walk.b >= 0 && walk.b < w.B && from >= 0 && cnt > 0);
      if (changing) continue;
      CHECK(from == done[walk.b] && from + cnt <= lens[walk.b]);
      done[walk.b] += cnt;
      partials[walk.b].push_back(slot + walk.b);
    }
  }
  for (int b = 0; b < w.B && !changing; ++b) CHECK(done[b] == lens[b]);
  if (!PAGED) return;
  w.reads = 0;
  gqa::FlatWalk<HostWave, true>::plan(w, [&](int s, int first, int count) {
    CHECK(s >= 0 && s < w.B && count >= 0 && first >= 0 && first + count <= w.slots + w.B);
    if (changing) return;
    CHECK(count == (int)partials[s].size());
    for (int i = 0; i < count; ++i) CHECK(partials[s][i] == first + i);
  });
}

int main() {
  std::mt19937 rng(1);
  auto in = [&](int lo, int hi) { return std::uniform_int_distribution<int>(lo, hi)(rng); };
  int n = 0;
  for (int B : {1, 2, 5, 63, 64, 65, 128, 130, 200, 500})
    for (int slots : {1, 3, 32, 64, 256})
      for (int longest : {1, 3, 40}) {
        std::vector<int> lens(B), other(B), zero(B, 0);
        for (int& l : lens) l = in(0, 3) == 0 ? 0 : in(0, longest);
        for (int& l : other) l = in(0, longest);
        HostWave w{&lens, &lens, B, slots, 1, 1 << 30};
        walk_all<true>(w, lens, false);
        walk_all<true>(HostWave{&zero, &zero, B, slots, 1, 1 << 30}, zero, false);
        for (const std::vector<int>* later : {&zero, &other})
          for (int change : {0, 1, 2, 3, 5, (B + 63) / 64, (B + 63) / 64 + 1}) {
            walk_all<true>(HostWave{&lens, later, B, slots, 1, change}, lens, true);
            walk_all<true>(HostWave{later, &lens, B, slots, 1, change}, lens, true);
          }
        std::vector<int> equal(B, longest);
        walk_all<false>(HostWave{&equal, &equal, B, slots, longest, 1 << 30}, equal, false);
        ++n;
      }
  std::printf("%d batches\n", n);
}
