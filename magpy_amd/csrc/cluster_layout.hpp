// cluster_layout.hpp -- host rules of the cluster kernels' layout that need no
// device: which launch set the autotuner times and what it remembers.
#pragma once
#include <stddef.h>
#include <stdint.h>

#include <map>
#include <mutex>
#include <tuple>
#include <vector>

namespace mp_host {

// Layout of the interacting-cluster kernel: `block` lanes per workgroup and
// `lanes` (1 or 2) lanes per particle slot, so a workgroup holds
// block / lanes slots, which must take the largest cluster.
struct ClusterLayout {
    int block = 0, lanes = 1;
};

// The launch set with the most particles: what a run's layout is tuned on.  Its
// groups are ranges of group_begin.  (A single group can be one cluster on an empty
// card, whose blocks of 64 to 1,024 lanes differ by noise.)
inline size_t largest_set(const std::vector<std::vector<int>> &sets,
                          const std::vector<int64_t> &group_begin, int64_t *particles)
{
    size_t best = 0;
    *particles = -1;
    for (size_t i = 0; i < sets.size(); ++i) {
        int64_t n = 0;
        for (int g : sets[i]) n += group_begin[(size_t)g + 1] - group_begin[(size_t)g];
        if (n > *particles) {
            best = i;
            *particles = n;
        }
    }
    return best;
}

// What a tuned layout holds for: device, largest cluster of the run, particles of
// the timed set, precision, lanes forced by the environment (0: none).
using LayoutKey = std::tuple<int, int64_t, int64_t, int, int>;

// Tuned layouts, for the life of the process.  Threads create sessions at the same
// time (the Python binding releases the interpreter lock), so every access is locked;
// two that tune one key at once keep the later's layout.
class LayoutCache {
  public:
    bool find(const LayoutKey &key, ClusterLayout &out) const
    {
        std::lock_guard<std::mutex> lock(m);
        auto it = known.find(key);
        if (it == known.end()) return false;
        out = it->second;
        return true;
    }
    void keep(const LayoutKey &key, const ClusterLayout &l)
    {
        std::lock_guard<std::mutex> lock(m);
        known[key] = l;
    }

  private:
    mutable std::mutex m;
    std::map<LayoutKey, ClusterLayout> known;
};

}  // namespace mp_host
