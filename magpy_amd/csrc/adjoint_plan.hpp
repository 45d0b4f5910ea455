// adjoint_plan.hpp -- host rule of the adjoint maps' batches, which needs no device.
#pragma once
#include <stddef.h>
#include <stdint.h>

#include <algorithm>
#include <vector>

namespace mp_host {

// A batch of segments whose maps run in one launch: segments (the last of a block may
// hold fewer) and the most pieces that any batch of the run has.
struct MapBatch {
    int64_t segments = 1, pieces = 1;
};

// The pieces of segments [j0, j1), from the first piece of every segment
inline int64_t pieces_of(const std::vector<int32_t> &seg_first, int64_t n_pieces, int64_t j0,
                         int64_t j1)
{
    const int64_t end = j1 < (int64_t)seg_first.size() ? seg_first[(size_t)j1] : n_pieces;
    return end - seg_first[(size_t)j0];
}

// Batches of the blocks of `block` segments, split evenly: up to `lanes` lanes (a
// segment of a particle each) and 8 GiB of device memory for the segments' states and
// the pieces' maps together, seg_bytes and piece_bytes for all particles.  Dense
// samples make many pieces of a segment, so that their maps are the larger part; a
// batch of 2^18 lanes is not cut further for them, since below that the launches no
// longer fill the card, and at least one segment is one batch.
inline MapBatch map_batch(const std::vector<int32_t> &seg_first, int64_t n_pieces, int64_t block,
                          int64_t particles, int64_t lanes, int64_t seg_bytes, int64_t piece_bytes)
{
    constexpr int64_t kMemory = (int64_t)8 << 30, kLeastLanes = (int64_t)1 << 18;
    const int64_t n_seg = (int64_t)seg_first.size();
    const int64_t most = std::min({block, std::max<int64_t>(1, lanes / particles),
                                   std::max<int64_t>(1, kMemory / seg_bytes)});
    for (int64_t n = (block + most - 1) / most;; ++n) {
        MapBatch b;
        b.segments = (block + n - 1) / n;
        for (int64_t b0 = 0; b0 < n_seg; b0 += block)
            for (int64_t j0 = b0, end = std::min(n_seg, b0 + block); j0 < end; j0 += b.segments)
                b.pieces = std::max(b.pieces, pieces_of(seg_first, n_pieces, j0,
                                                        std::min(end, j0 + b.segments)));
        if (b.segments == 1 || b.segments * particles <= kLeastLanes ||
            b.segments * seg_bytes + b.pieces * piece_bytes <= kMemory)
            return b;
    }
}

}  // namespace mp_host
