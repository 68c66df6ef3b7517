// The backward flush's claim of a vertex's corners (gvv_claim.hpp) under the weakest order of the
// stores: every 32-bit word of a table entry may stay from any of the corners that stored to it.  For
// random tiles of faces, the terms that arrive at each vertex are compared with the sum over its
// corners (integers, so exact).  Beside it, an entry of two words (vertex, corner), to show that the
// model tells the difference.  Host only.
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <random>
#include <vector>
#include "../gvv-differentiable-cuda-renderer_amd/csrc/gvv_claim.hpp"
using namespace gvv;

struct OneWord {
  typedef ClaimEntry Entry;
  static Entry entry(int, int c) { return claim_entry(c); }
  static int target(Entry e, const int* vid, int c) { return claim_target(e, vid, c); }
};
struct TwoWords {
  struct Entry { int v, c; };
  static Entry entry(int v, int c) { return {v, c}; }
  static int target(Entry e, const int* vid, int c) { return e.v == vid[c] ? e.c : c; }
};

template <class Claim>
static long long run(int tiles) {
  constexpr int kCap = 128, kWords = sizeof(typename Claim::Entry) / 4;
  std::mt19937 rng(3);
  long long wrong = 0;
  for (int t = 0; t < tiles; ++t) {
    const int slots = 1 + (int)(rng() % 32), corners = 3 * slots;
    const int spread = 1 << (rng() % 12);                  // few vertices .. several per entry
    std::vector<int> vid(corners);
    std::vector<long long> term(corners);
    std::map<int, long long> want, got;
    std::vector<std::vector<int>> writers(kCap);
    for (int c = 0; c < corners; ++c) {
      vid[c] = (int)(rng() % spread);
      term[c] = 1 + (int)(rng() % 1000000);
      want[vid[c]] += term[c];
      writers[vid[c] & (kCap - 1)].push_back(c);
    }
    std::vector<typename Claim::Entry> table(kCap);
    for (int h = 0; h < kCap; ++h)
      for (int w = 0; w < kWords && !writers[h].empty(); ++w) {
        const int c = writers[h][rng() % writers[h].size()];
        const typename Claim::Entry e = Claim::entry(vid[c], c);
        std::memcpy((char*)&table[h] + 4 * w, (const char*)&e + 4 * w, 4);
      }
    std::vector<int> to(corners);
    for (int c = 0; c < corners; ++c) to[c] = Claim::target(table[vid[c] & (kCap - 1)], vid.data(), c);
    for (int c = 0; c < corners; ++c) got[vid[to[c]]] += term[c];
    for (int c = 0; c < corners; ++c)
      if (to[to[c]] != to[c]) ++wrong;                     // a corner that is added to must itself be flushed
    wrong += want != got;
  }
  return wrong;
}

int main(int argc, char** argv) {
  const int tiles = argc > 1 ? atoi(argv[1]) : 20000;
  printf("one_word %lld two_words %lld entry_bytes %d\n", run<OneWord>(tiles), run<TwoWords>(tiles), (int)sizeof(ClaimEntry));
  return 0;
}
