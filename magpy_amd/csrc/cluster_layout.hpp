// cluster_layout.hpp -- host rules of the cluster kernels' layout that need no
// device: how clusters are packed into workgroups, which launch set the autotuner times
// and what it remembers, and how many lanes of the implicit kernel share their pair sums.
#pragma once
#include <stddef.h>
#include <stdint.h>

#include <algorithm>
#include <map>
#include <mutex>
#include <tuple>
#include <utility>
#include <vector>

namespace mp_host {

// Layout of the interacting-cluster kernel: `block` lanes per workgroup and
// `lanes` (1 or 2) lanes per particle slot, so a workgroup holds
// block / lanes slots, which must take the largest cluster.
struct ClusterLayout {
    int block = 0, lanes = 1;
};

// Cluster packing: members of a group sorted by size (largest first), each
// placed in the first block with room; a member never straddles blocks.
// Returns slot -> particle (-1 padding), and per slot the block-relative
// start lane of its member and the member size.  A member takes a multiple of
// `align` slots: those past its size are its helpers (slot_particle -1, with the
// member's start and size), so every member starts on a multiple of align.
// Blocks come out largest member first.  The dispatcher deals workgroups round
// the XCDs, their CUs and SIMDs, so those `run` apart share a SIMD; a
// workgroup's time goes with its largest member, and with up to `most_runs` runs
// every second one is reversed so that a SIMD gets a long and a short one.  More
// runs follow each other on a SIMD, where the longest first leave the shortest end.
inline void pack_clusters(const std::vector<std::pair<int64_t, int64_t>> &members, int block,
                          int align, size_t run, size_t most_runs,
                          std::vector<int64_t> &slot_particle, std::vector<int> &cbase,
                          std::vector<int> &csize)
{
    auto taken = [align](int size) { return (size + align - 1) / align * align; };
    std::vector<size_t> order(members.size());
    for (size_t i = 0; i < order.size(); ++i) order[i] = i;
    std::stable_sort(order.begin(), order.end(), [&](size_t x, size_t y) {
        return members[x].second - members[x].first > members[y].second - members[y].first;
    });
    std::vector<int> fill;                       // lanes used per block
    std::vector<std::vector<size_t>> content;    // members per block
    size_t first_open = 0;
    for (size_t oi : order) {
        const int sz = taken((int)(members[oi].second - members[oi].first));
        size_t bi = first_open;
        while (bi < fill.size() && fill[bi] + sz > block) ++bi;
        if (bi == fill.size()) {
            fill.push_back(0);
            content.emplace_back();
        }
        fill[bi] += sz;
        content[bi].push_back(oi);
        while (first_open < fill.size() && fill[first_open] == block) ++first_open;
    }
    const bool in_order = content.size() > most_runs * run;
    for (size_t b = run; !in_order && b < content.size(); b += 2 * run)
        std::reverse(content.begin() + (ptrdiff_t)b,
                     content.begin() + (ptrdiff_t)std::min(content.size(), b + run));
    const size_t nslots = fill.size() * (size_t)block;
    slot_particle.assign(nslots, -1);
    cbase.assign(nslots, 0);
    csize.assign(nslots, 0);
    for (size_t bi = 0; bi < content.size(); ++bi) {
        int lane = 0;
        for (size_t oi : content[bi]) {
            const int sz = (int)(members[oi].second - members[oi].first);
            for (int j = 0; j < taken(sz); ++j) {
                const size_t slot = bi * (size_t)block + (size_t)(lane + j);
                if (j < sz) slot_particle[slot] = members[oi].first + j;
                cbase[slot] = lane;
                csize[slot] = sz;
            }
            lane += taken(sz);
        }
    }
}

// The most runs of blocks that pack_clusters reverses (speed against blocks in order,
// means over four ensembles each of 2 to 64 and of 8 to 128 particles): the implicit
// kernel, three waves a SIMD, 1.01 to 1.06 up to three runs, 0.99 above; Heun on two
// lanes 0.99 to 1.03 in FP32 and 0.95 to 1.07 in FP64 up to five (the mean 1.01), 0.99
// above; on one lane 0.97 and 1.04 in FP32 at four, below 1 above.
inline size_t reversed_runs(bool implicit, int lanes)
{
    return implicit ? 3 : lanes == 2 ? 5 : 0;
}

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

// Lanes of the implicit cluster kernel that share their pair sums (shared_field), 2 or
// 4, for the members (particle ranges) of a launch; the results are the same.  Four
// are the faster for clusters of 9 and more, but a small member's helper lanes then
// take slots of their own.  So: two with no cluster above 8; four where all slots are
// at most a wave on every SIMD (one_wave), since the largest cluster's wave then takes
// the launch's time; else four if the slots that helpers add are a sixth of the large
// clusters' particles or fewer.  us per step with 2 / 4 lanes, 32 steps (helpers /
// large particles): 65,536 dimers 38 / 105; and one cluster of 9 with them 62 / 115;
// 6,000 of 9 and 10,000 dimers (0.37) 85 / 96; 2,000 of 64 and 20,000 dimers (0.31)
// 373 / 409, 8,000 dimers (0.13) 363 / 330; 6,000 of 16 and 3,000 dimers (0.06) 140 /
// 122.  A wave per SIMD or fewer: 64 of 32 and 512 dimers 116 / 98, one of 9 and 64
// dimers 49 / 43.
inline int field_targets(const std::vector<std::pair<int64_t, int64_t>> &members, int64_t one_wave)
{
    int64_t slots = 0, helpers = 0, large = 0;
    for (const auto &m : members) {
        const int64_t n = m.second - m.first, two = (n + 1) / 2 * 2, four = (n + 3) / 4 * 4;
        slots += four;
        if (n > 8) large += n;
        else helpers += four - two;
    }
    if (large == 0) return 2;
    return slots <= one_wave || 6 * helpers <= large ? 4 : 2;
}

}  // namespace mp_host
