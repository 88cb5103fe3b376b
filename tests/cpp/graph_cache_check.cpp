/* The cache of captured graphs: what is in use stays, the least recently used
 * leaves, everything is destroyed once. Graphs are numbers here. */
#include "graph_cache.hpp"

#include <cstdio>
#include <set>

int main() {
  typedef av1hip::GraphCache<int> Cache;
  const int n = (int)Cache::kMax;
  Cache c;
  std::set<int> gone;
  int twice = 0;
  auto destroy = [&](int e) { twice += !gone.insert(e).second; };
  auto check = [](bool ok, const char* what) {
    if (!ok) std::printf("%s\n", what);
    return ok ? 0 : 1;
  };
  int bad = 0;
  for (int k = 1; k <= n; ++k) c.insert((uint64_t)k, k, destroy);
  bad += check(gone.empty() && c.find(1) == 1 && c.find(77) == 77, "holds kMax graphs");
  /* 2 is now the oldest; the one replayed last is in flight while others are captured */
  for (int k = n + 1; k < 3 * n; ++k) {
    const int hot = 77;
    bad += check(c.find((uint64_t)hot) == hot, "the graph in use stays");
    c.insert((uint64_t)k, k, destroy);
    bad += check(c.size() == Cache::kMax, "kMax graphs at most");
    if (k == n + 1) bad += check(gone.count(2) && gone.size() == 1 && c.find(2) == 0, "the least recently used leaves");
  }
  bad += check(gone.count(1) && !gone.count(77), "what is not used leaves in time");
  c.clear(destroy);
  bad += check(c.size() == 0 && !twice && gone.size() == (size_t)(3 * n - 1), "each graph destroyed once");
  return bad ? 1 : 0;
}
