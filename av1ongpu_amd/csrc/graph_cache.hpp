/*
 * The captured launch sequences of a context, by the shape of the batch they
 * replay.
 */
#ifndef AV1HIP_GRAPH_CACHE_HPP
#define AV1HIP_GRAPH_CACHE_HPP

#include <stddef.h>
#include <stdint.h>

#include <algorithm>
#include <utility>
#include <vector>

namespace av1hip {

/* At most kMax graphs, the least recently used leaving first: a context has
 * at most one batch in flight when it captures another's graph, the one it
 * replayed last, so what leaves is never in use. kMax: 64 shapes in each of
 * the six size classes a key distinguishes, at 0.6 MB of device memory a graph
 * at most 0.25 GB; a capture takes 0.1 ms (320 shapes of one to ten 64x64
 * frames: 0.24 ms a batch captured, 0.15 replayed). */
template <typename Exec>
class GraphCache {
 public:
  static constexpr size_t kMax = 64 * 6;

  /* the graph of `key`, now the last used, or Exec() */
  Exec find(uint64_t key) {
    for (size_t i = v_.size(); i-- > 0;)
      if (v_[i].first == key) {
        std::rotate(v_.begin() + (ptrdiff_t)i, v_.begin() + (ptrdiff_t)i + 1, v_.end());
        return v_.back().second;
      }
    return Exec();
  }
  template <typename Destroy>
  void insert(uint64_t key, Exec exec, Destroy&& destroy) {
    if (v_.size() >= kMax) {
      destroy(v_.front().second);
      v_.erase(v_.begin());
    }
    v_.emplace_back(key, exec);
  }
  template <typename Destroy>
  void clear(Destroy&& destroy) {
    for (auto& g : v_) destroy(g.second);
    v_.clear();
  }
  size_t size() const { return v_.size(); }

 private:
  std::vector<std::pair<uint64_t, Exec>> v_; /* the least recently used first */
};

}  // namespace av1hip

#endif
