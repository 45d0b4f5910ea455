// cluster_norm.h -- the squared norm over a cluster of the implicit kernel, for the
// device and, unchanged, for a host build that checks its order
// (tests/test_cluster_norm_cpu.py).
#pragma once

#if defined(__HIPCC__)
#define MP_CN __host__ __device__ inline
#else
#define MP_CN inline
#endif

namespace mp {

// The sum of the particles' squares over the slots [cb, ce) of a cluster, from the
// sums of kT = 2 or 4 neighbouring lanes, red[slot / kT]; cb is a multiple of kT.  It
// is taken over fours, (s0 + s1) + (s2 + s3) each, and eight fours as a tree, for
// either kT, since the launch's largest cluster picks kT and a member's norm, and with
// it its Newton count, must not depend on the rest of the ensemble.  kT = 4: up to 64
// sums, eight LDS reads in flight; kT = 2, clusters of up to 8: the few there are.
template <int kT>
MP_CN double cluster_square(const double *red, int cb, int ce)
{
    auto four = [&](int k) {
        if constexpr (kT == 4) return red[k / 4];
        else return k + 2 < ce ? red[k / 2] + red[k / 2 + 1] : red[k / 2];
    };
    if constexpr (kT == 2) {
        if (ce - cb <= 4) return four(cb);
        if (ce - cb <= 8) return four(cb) + four(cb + 4);
    }
    double sum = 0.0;
    for (int k = cb; k < ce; k += 32) {
        double v[8];
#if defined(__HIPCC__)
#pragma unroll
#endif
        for (int u = 0; u < 8; ++u) v[u] = four(k + 4 * u < ce ? k + 4 * u : cb);
#if defined(__HIPCC__)
#pragma unroll
#endif
        for (int u = 0; u < 8; ++u) v[u] = k + 4 * u < ce ? v[u] : 0.0;
        sum += ((v[0] + v[1]) + (v[2] + v[3])) + ((v[4] + v[5]) + (v[6] + v[7]));
    }
    return sum;
}

}  // namespace mp
