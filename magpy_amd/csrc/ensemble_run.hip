// ensemble_run.hip -- host side of the MI355X sLLG integrator and its C ABI.
//
// simulation::ensemble_run (simulation.hpp) validates the request, reduces
// every member to dimensionless units exactly as simulation::full_dynamics
// does (lib/simulation.cpp:501-583), derives the reference's sample schedule,
// uploads SoA parameter arrays, and drives the step kernels of
// sllg_kernels.hpp in blocks of steps on one HIP stream.  A session keeps that
// state resident between calls.  The extern "C" functions at the end are the
// boundary declared in include/magpy_amd.h.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <chrono>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <iterator>
#include <limits>
#include <map>
#include <memory>
#include <mutex>
#include <new>
#include <string>
#include <type_traits>
#include <vector>

#include "cluster_layout.hpp"
#include "host_util.hpp"
#include "simulation.hpp"
#include "replica_kernels.hpp"
#include "sllg_kernels.hpp"

namespace mp_host {
std::string &last_error()
{
    thread_local std::string text;
    return text;
}
}  // namespace mp_host

namespace {

using namespace mp_host;

// The applied field of lib/simulation.cpp:552-573 at reduced time t.
double applied_host(int shape, double happ, double fapp, double t)
{
    switch (shape) {
    case MP_FIELD_SINE: return happ * std::sin(2 * kPiHost * fapp * t);
    case MP_FIELD_SQUARE: return happ * ((int)(t * fapp * 2) % 2 ? -1 : 1);
    default: return happ;
    }
}

// Steps per kernel launch: long enough to amortise the launch, short enough
// to keep each launch well under a second.
int64_t steps_per_launch(int scheme, int precision)
{
    if (const char *env = std::getenv("MAGPY_AMD_STEPS_PER_LAUNCH")) {
        long long v = std::atoll(env);
        if (v > 0) return (int64_t)v;
    }
    if (scheme == MP_SCHEME_IMPLICIT_MIDPOINT) return 1 << 12;
    return precision == MP_PRECISION_FP32 ? (1 << 17) : (1 << 16);
}

// compute units of the current device
int device_cus()
{
    int dev = 0, cus = 0;
    MP_HIP(hipGetDevice(&dev));
    MP_HIP(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
    return cus;
}

template <typename T>
std::vector<T> cast_vec(const std::vector<double> &v)
{
    return std::vector<T>(v.begin(), v.end());
}

// Which Heun kernel runs n_waves integrating waves: 0 the one-wave kernel;
// FP32: 1 the two-wave kernel with the normals formed by the producing wave, 2
// the same with Box-Muller in the integrating wave; FP64: 1 (or 2) the kernel
// with three producing waves per integrating wave.  FP32: 2 while the
// integrating waves are more than one per CU and at most one per SIMD, 1 at one
// per CU or fewer, else 0 (32,768-step launches: 65,536 particles 3.63e11 /
// 3.02e11 / 2.72e11 for 2 / 1 / 0; 16,384: 0.94e11 / 1.21e11 / 0.68e11; 131,072:
// 2.99e11 / 2.82e11 / 3.66e11).  FP64: 1 up to two integrating waves per CU,
// where the producing waves have SIMDs of their own (us per step, 1 / 0, sine
// field: 1,000 particles 0.146 / 0.428, 16,384 0.157 / 0.439, 32,768 0.262 /
// 0.434, 65,536 0.493 / 0.458, 131,072 0.986 / 0.838).
// MAGPY_AMD_HEUN_TWO_WAVE=0/1/2 forces the choice.
int two_wave_mode(int n_waves, bool fp32)
{
    if (const char *env = std::getenv("MAGPY_AMD_HEUN_TWO_WAVE")) {
        const int v = std::atoi(env);
        return v <= 0 ? 0 : (v >= 2 && fp32) ? 2 : 1;
    }
    const int cus = device_cus();
    if (!fp32) return n_waves <= 2 * cus ? 1 : 0;
    if (n_waves > 4 * cus) return 0;
    return n_waves > cus ? 2 : 1;
}

// grid: blocks of kBlock lanes (n_waves = 4 grid integrating waves)
template <typename T, int kShape, bool kArray, bool kRenorm>
void launch_heun(const mp::IndepArgs<T> &a, int grid, hipStream_t s, const float *htab,
                 int two_wave)
{
    if constexpr (!kArray) {
        if (two_wave != 0) {
            // one integrating wave per workgroup (FP32: one (integrating,
            // producing) pair; two or four pairs measure the same or slower)
            const dim3 g2((unsigned)(grid * (mp::kBlock / mp::kWave))),
                b2(sizeof(T) == 4 ? 2 * mp::kWave : 4 * mp::kWave);
            if constexpr (sizeof(T) == 4) {
                auto go = [&](auto kernel) { hipLaunchKernelGGL(kernel, g2, b2, 0, s, a, htab); };
                if (htab) {
                    if (two_wave == 2)
                        go(mp::heun_indep_pc_kernel<T, mp::kConstant, true, kRenorm, true>);
                    else
                        go(mp::heun_indep_pc_kernel<T, mp::kConstant, true, kRenorm, false>);
                    return;
                }
                if (two_wave == 2) go(mp::heun_indep_pc_kernel<T, kShape, false, kRenorm, true>);
                else go(mp::heun_indep_pc_kernel<T, kShape, false, kRenorm, false>);
                return;
            }
            if constexpr (sizeof(T) == 8)
                hipLaunchKernelGGL((mp::heun_indep_pc_kernel<T, kShape, false, kRenorm, false, 3>),
                                   g2, b2, 0, s, a, htab);
            return;
        }
    }
    if constexpr (sizeof(T) == 4) {
        if (htab) {  // the table replaces per-lane field evaluation: one variant per noise kind
            hipLaunchKernelGGL((mp::heun_indep_kernel<T, mp::kConstant, kArray, true, kRenorm>),
                               dim3(grid), dim3(mp::kBlock), 0, s, a, htab);
            return;
        }
    }
    hipLaunchKernelGGL((mp::heun_indep_kernel<T, kShape, kArray, false, kRenorm>), dim3(grid),
                       dim3(mp::kBlock), 0, s, a, htab);
}

template <typename T, int kShape, bool kArray>
void launch_step(const mp::IndepArgs<T> &a, int scheme, double eps, int max_iter,
                 unsigned long long *it, unsigned long long *fl, int grid, hipStream_t s,
                 const float *htab, int two_wave)
{
    if constexpr (sizeof(T) == 8) {
        if (scheme == MP_SCHEME_IMPLICIT_MIDPOINT) {
            mp::ImplicitArgs ia{a, eps, max_iter, it, fl};
            hipLaunchKernelGGL((mp::implicit_indep_kernel<kShape, kArray>), dim3(grid),
                               dim3(mp::kBlock), 0, s, ia);
            return;
        }
    }
    if (a.renorm)
        launch_heun<T, kShape, kArray, true>(a, grid, s, htab, two_wave);
    else
        launch_heun<T, kShape, kArray, false>(a, grid, s, htab, two_wave);
}

template <typename T, bool kArray>
void launch_shape(int shape_kind, const mp::IndepArgs<T> &a, int scheme, double eps,
                  int max_iter, unsigned long long *it, unsigned long long *fl, int grid,
                  hipStream_t s, const float *htab, int tw)
{
    switch (shape_kind) {
    case mp::kSine: launch_step<T, mp::kSine, kArray>(a, scheme, eps, max_iter, it, fl, grid, s, htab, tw); break;
    case mp::kSquare: launch_step<T, mp::kSquare, kArray>(a, scheme, eps, max_iter, it, fl, grid, s, htab, tw); break;
    case mp::kConstant: launch_step<T, mp::kConstant, kArray>(a, scheme, eps, max_iter, it, fl, grid, s, htab, tw); break;
    default: launch_step<T, mp::kMixed, kArray>(a, scheme, eps, max_iter, it, fl, grid, s, htab, tw); break;
    }
}

struct Plan {
    // particles ordered by schedule group; perm[i] = original particle index
    std::vector<int64_t> perm;
    std::vector<int64_t> group_begin;        // [G+1] ranges in perm order
    std::vector<std::vector<int64_t>> sched; // per group
    std::vector<int64_t> group_steps;        // per group
    std::vector<int64_t> member_of;          // per original particle
    std::vector<int> group_of;               // per member
    std::vector<simulation::ReducedMember> red;
};

// Host copies of what the outputs need after the caller's spec is gone.
struct HostCopy {
    int64_t M = 0, P = 0, S = 0, start = 0;   // m0 is the state at step `start`
    std::vector<double> m0, ms;
    std::vector<int32_t> shape;
};

// Results of one launch set copied back to the host: states and samples go
// straight to the caller's arrays, the rest is per slot.  Sums of a sample that a
// group took at or before the run's start step are unspecified or zero.
struct GroupOut {
    std::vector<uint32_t> status;
    std::vector<double> ens;          // [S][3]        (empty when not recorded)
    int64_t newton_iters = 0, newton_fail = 0;
};

// Where the samples of a launch set go: the caller's [P][S] arrays (any may be
// null), and what a sample at or before the start step is (the start state as
// given, or unknown).
struct SampleSink {
    double *dst[3];
    const Plan &plan;
    const HostCopy &host;

    // Samples of every slot from src [S][3][n]; slot_particle[i] is the particle
    // (-1: padding).  Tiles of particles and samples keep both sides in cache.
    template <typename T>
    void take(const T *src, const std::vector<int64_t> &slot_particle) const
    {
        constexpr int64_t kTile = 16;
        const int64_t n = (int64_t)slot_particle.size(), S = host.S;
        const double nan = std::numeric_limits<double>::quiet_NaN();
        for (int64_t i0 = 0; i0 < n; i0 += kTile)
            for (int64_t s0 = 0; s0 < S; s0 += kTile)
                for (int64_t i = i0; i < std::min(n, i0 + kTile); ++i) {
                    const int64_t p = slot_particle[(size_t)i];
                    if (p < 0) continue;
                    const int64_t m = plan.member_of[(size_t)p];
                    const double ms = host.ms[(size_t)m];
                    const std::vector<int64_t> &k = plan.sched[(size_t)plan.group_of[(size_t)m]];
                    for (int64_t sa = s0; sa < std::min(S, s0 + kTile); ++sa) {
                        const int64_t at = k[(size_t)sa];
                        const T *row = at > host.start ? src + sa * 3 * n + i : nullptr;
                        for (int d = 0; d < 3; ++d) {
                            if (!dst[d]) continue;
                            const double v = row != nullptr       ? (double)row[d * n]
                                             : at == host.start ? host.m0[(size_t)p * 3 + d]
                                                                  : nan;
                            dst[d][p * S + sa] = v * ms;
                        }
                    }
                }
    }
};

struct GroupBase {
    int64_t n_done = 0, n_total = 0, launches = 0;
    virtual ~GroupBase() = default;
    virtual void enqueue(int64_t upto, hipStream_t s) = 0;
    virtual void state(double *out) = 0;               // its particles' rows of [P][3]
    virtual const std::vector<int64_t> &slots() const = 0;
    virtual const std::vector<int> &set() const = 0;   // its schedule groups
    // Device memory for one launch's records, which the sets of a run share: each
    // launch's records are taken from it before the next launch of any set
    virtual size_t record_bytes() const { return 0; }
    virtual void use_records(void *) {}
    virtual GroupOut collect(hipStream_t s, double *state_out, const SampleSink *samples) = 0;
};

// The applied field of a schedule group: whether all of its particles see the
// same one (shape, reduced amplitude, cycles per step), and which.
struct GroupField {
    bool uniform = true;
    int shape = 0;
    double amp = 0.0, fdt = 0.0;
};

GroupField group_field(const simulation::EnsembleSpec &sp, const Plan &plan, int gi)
{
    GroupField f;
    bool first = true;
    for (int64_t i = plan.group_begin[(size_t)gi]; i < plan.group_begin[(size_t)gi + 1]; ++i) {
        const int64_t m = plan.member_of[(size_t)plan.perm[(size_t)i]];
        const simulation::ReducedMember &r = plan.red[(size_t)m];
        const GroupField x{true, sp.field_shape[m], r.happ, r.fapp * r.dt};
        if (first) f = x;
        else if (x.shape != f.shape || x.amp != f.amp || x.fdt != f.fdt) f.uniform = false;
        first = false;
    }
    return f;
}

// The sample steps a launch set records and, with several groups in it, which
// record each group's samples are.
std::vector<int64_t> union_schedule(const Plan &plan, const std::vector<int> &set, int64_t start,
                                    std::vector<std::vector<int32_t>> &pick)
{
    pick.clear();
    if (set.size() == 1) return plan.sched[(size_t)set[0]];
    std::vector<int64_t> u;
    for (int gi : set)
        for (int64_t k : plan.sched[(size_t)gi])
            if (k > start) u.push_back(k);
    std::sort(u.begin(), u.end());
    u.erase(std::unique(u.begin(), u.end()), u.end());
    for (int gi : set) {
        std::vector<int32_t> row;
        for (int64_t k : plan.sched[(size_t)gi])
            row.push_back(k > start ? (int32_t)(std::lower_bound(u.begin(), u.end(), k) - u.begin())
                                    : -1);
        pick.push_back(std::move(row));
    }
    return u;
}

// Which schedule groups share a launch.  An ensemble whose members differ in
// anisotropy or damping has a reduced step per member, and where sample times
// fall on step boundaries the rounding of each decides its sample steps, so it
// can have a schedule group per member: one launch of one particle after the
// other (300 members, 2,000 FP64 steps: 178 ms).  A launch set records the union
// of its groups' sample steps, which differ by a step here and there, and each
// member's samples (and each group's sums) are picked from it after each launch, so
// that a run keeps its samples as it would with a launch per group, and the records
// of one set beside them.  Sets hold groups of equal step count whose
// kernels run the same code for them: FP64 and the implicit scheme, whose lanes
// all evaluate their own field; FP32 constant fields; and FP32 groups of
// independent particles that read their field from a table, as many rows of it.
// Not in a set: schedules too unlike (records beyond three times the samples),
// more than 1 GiB of records (the set is cut there), FP32 groups with per-lane
// fields, and runs in caller-bounded memory.
std::vector<std::vector<int>> launch_sets(const simulation::EnsembleSpec &sp, const Plan &plan,
                                          bool clusters, bool bounded_memory)
{
    const int G = (int)plan.sched.size();
    std::vector<std::vector<int>> sets;
    const bool fp32 = sp.precision == MP_PRECISION_FP32 && sp.scheme == MP_SCHEME_HEUN;
    std::map<std::pair<int, int64_t>, std::vector<int>> alike;   // (kind, steps) -> groups
    for (int g = 0; g < G; ++g) {
        int kind = 0;
        if (fp32) {
            const GroupField f = group_field(sp, plan, g);
            kind = !f.uniform ? -1 : f.shape == MP_FIELD_CONSTANT ? 1 : clusters ? -1 : 2;
            if (sp.noise == MP_NOISE_ARRAY) kind = kind == 2 ? -1 : kind;
        }
        if (bounded_memory || G == 1) kind = -1;
        if (kind < 0) sets.push_back({g});
        else alike[{kind, plan.group_steps[(size_t)g]}].push_back(g);
    }
    const int64_t table_lanes = 4 * (int64_t)device_cus() * mp::kWave;  // two_wave_mode's bound
    for (auto &[key, gs] : alike) {
        const int64_t S = sp.max_samples, most = 3 * S + 8;
        std::vector<int> cur;
        std::vector<int64_t> steps;      // the records of cur
        int64_t lanes = 0;
        for (int g : gs) {
            const int64_t len = plan.group_begin[(size_t)g + 1] - plan.group_begin[(size_t)g];
            std::vector<int64_t> u;
            std::set_union(steps.begin(), steps.end(), plan.sched[(size_t)g].begin(),
                           plan.sched[(size_t)g].end(), std::back_inserter(u));
            u.erase(std::unique(u.begin(), u.end()), u.end());
            const bool fits = (int64_t)u.size() <= most &&
                              (int64_t)u.size() * 3 * (lanes + len) * (fp32 ? 4 : 8) <= (1ll << 30) &&
                              (key.first != 2 || lanes + len <= table_lanes);
            if (!cur.empty() && !fits) {
                sets.push_back(std::move(cur));
                cur.clear();
                u = plan.sched[(size_t)g];
                lanes = 0;
            }
            cur.push_back(g);
            steps = std::move(u);
            lanes += len;
        }
        if (!cur.empty()) sets.push_back(std::move(cur));
    }
    std::sort(sets.begin(), sets.end());
    return sets;
}

template <typename T>
struct GroupRun : GroupBase {
    // n: slots of the arrays, of which a cluster's workgroups have n_slots (implicit
    // clusters: also helpers and padding, with no place in the arrays)
    int n = 0, n_slots = 0, grid = 0, block = mp::kBlock, n_waves = 0, scheme = 0, shape_kind = -1;
    int max_iter = 1000;
    double eps = 1e-9;
    bool array_noise = false, want_traj = false, want_ens = false, cluster = false;
    bool interactions = true;  // clusters: dipolar sums (the implicit scheme may run without)
    int two_wave = 0;          // Heun kernel: 0 one wave, 1/2 two waves (two_wave_mode)
    int lanes = 1;             // lanes per cluster slot (1 or 2)
    int targets = 1;           // implicit clusters: lanes that share their pair sums
    // The schedule groups of this launch set.  With several, the kernels record
    // the union of their sample steps (S of them, S_out samples per group) and
    // pick[g][s] is the record of group g's sample s (-1: at or before the start).
    // take_records keeps of them what the run asked for: the samples, in d_samples
    // as a single group's, and a sum per sample and group, in d_partial.
    std::vector<int> groups;
    int64_t S = 0, S_out = 0, s_next = 0, spl = 1;
    std::vector<int64_t> sched, slot_particle;
    std::vector<int> slot_group;              // index into groups (-1: padding)
    std::vector<std::vector<int32_t>> pick;
    DevBuf<T> d_ex, d_ey, d_ez, d_k, d_al, d_dt, d_sig, d_sr, d_happ, d_m, d_samples;   // d_m: x, y, z, each n
    DevBuf<T> d_px, d_py, d_pz, d_w;
    DevBuf<double> d_fred, d_fdt, d_dtd, d_msw, d_noise, d_partial;   // d_partial: then the sums
    DevBuf<int> d_shape, d_cbase, d_csize, d_row, d_cell;
    DevBuf<uint32_t> d_key0, d_key1, d_pid, d_status;
    DevBuf<int64_t> d_sched;
    DevBuf<unsigned long long> d_newton;      // per slot: iterations, then failures
    DevBuf<float> d_htab;      // applied field of one launch (FP32 Heun), a row per field
    bool uniform_field = false;
    DevBuf<int> d_field_shape;                // per row of d_htab
    DevBuf<double> d_field_amp, d_field_fdt;
    int64_t tab_stride = 0;
    DevBuf<int64_t> d_toff;                   // per slot: start of its row (several rows)
    DevBuf<int32_t> d_pick, d_slot_group;
    DevBuf<int32_t> d_group_slots, d_group_first;   // the slots of each group
    T *records = nullptr;      // at the end of d_samples, or the run's (use_records)
    size_t n_samples = 0;      // values of d_samples that are samples
    mp::IndepArgs<T> a{};

    // cluster_block == 0: one slot per particle of the group (independent
    // particles); otherwise members packed into blocks of cluster_block lanes,
    // cluster_lanes (1 or 2) lanes per slot.  sole_set: no other set shares its records.
    GroupRun(const simulation::EnsembleSpec &sp, const Plan &plan, const std::vector<int> &set,
             bool traj, bool ens, int cluster_block, int cluster_lanes = 1, bool sole_set = false)
        : groups(set)
    {
        const int64_t P = sp.member_offsets[sp.n_members];
        n_total = plan.group_steps[(size_t)set[0]];
        scheme = sp.scheme;
        eps = sp.implicit_tol;
        max_iter = sp.implicit_max_iter > 0 ? sp.implicit_max_iter : 1000;
        array_noise = sp.noise == MP_NOISE_ARRAY;
        interactions = sp.interactions != 0;
        want_traj = traj;
        want_ens = ens;
        spl = steps_per_launch(sp.scheme, sp.precision);
        n_done = std::min(sp.start_step, n_total);
        S_out = (int64_t)plan.sched[(size_t)set[0]].size();
        sched = union_schedule(plan, set, n_done, pick);
        S = (int64_t)sched.size();
        cluster = cluster_block > 0;
        std::vector<int> cbase, csize;
        if (cluster) {
            std::vector<std::pair<int64_t, int64_t>> members;  // particle ranges
            for (int gi : set)
                for (int64_t i = plan.group_begin[(size_t)gi];
                     i < plan.group_begin[(size_t)gi + 1];) {
                    const int64_t m = plan.member_of[(size_t)plan.perm[(size_t)i]];
                    const int64_t len = sp.member_offsets[m + 1] - sp.member_offsets[m];
                    members.emplace_back(sp.member_offsets[m], sp.member_offsets[m] + len);
                    i += len;
                }
            block = cluster_block;
            lanes = cluster_lanes;
            // workgroups that fill every SIMD once
            const size_t run =
                (size_t)std::max(1, 4 * device_cus() / ((block + mp::kWave - 1) / mp::kWave));
            const bool implicit = scheme == MP_SCHEME_IMPLICIT_MIDPOINT;
            if (implicit) targets = field_targets(members, 4 * (int64_t)device_cus() * mp::kWave);
            pack_clusters(members, block / lanes, targets, run, reversed_runs(implicit, lanes),
                          slot_particle, cbase, csize);
            n_slots = (int)slot_particle.size();
            if (implicit) {
                // arrays hold the particles alone; 8 bytes a slot find them
                std::vector<int> row((size_t)n_slots, 0), cell((size_t)n_slots, 0);
                std::vector<int64_t> particles;
                for (int i = 0; i < n_slots; ++i) {
                    cell[(size_t)i] = cbase[(size_t)i] | csize[(size_t)i] << 16;
                    if (slot_particle[(size_t)i] >= 0) {
                        row[(size_t)i] = (int)particles.size();
                        particles.push_back(slot_particle[(size_t)i]);
                    } else if (csize[(size_t)i] > 0) {   // a helper reads its neighbour's row
                        row[(size_t)i] = (int)particles.size() - 1;
                    }
                }
                slot_particle = std::move(particles);
                d_row.upload(row);
                d_cell.upload(cell);
            }
        } else {
            for (int gi : set)
                slot_particle.insert(slot_particle.end(),
                                     plan.perm.begin() + plan.group_begin[(size_t)gi],
                                     plan.perm.begin() + plan.group_begin[(size_t)gi + 1]);
        }
        n = (int)slot_particle.size();
        slot_group.assign((size_t)n, -1);
        for (int i = 0; i < n; ++i) {
            if (slot_particle[(size_t)i] < 0) continue;
            const int g = plan.group_of[(size_t)plan.member_of[(size_t)slot_particle[(size_t)i]]];
            slot_group[(size_t)i] = (int)(std::lower_bound(set.begin(), set.end(), g) - set.begin());
        }

        std::vector<double> ex(n, 0.0), ey(n, 0.0), ez(n, 1.0), k(n, 0.0), al(n, 0.0), dt(n, 0.0),
            sig(n, 0.0), sr(n, 0.0), happ(n, 0.0), fred(n, 0.0), fdt(n, 0.0), msw(n, 0.0),
            m_now(3 * (size_t)n, 0.0), px(n, 0.0), py(n, 0.0), pz(n, 0.0), w(n, 0.0);
        std::vector<int> shape(n, MP_FIELD_CONSTANT);
        std::vector<uint32_t> key0(n, 0), key1(n, 0), pid(n, 0);
        bool first = true;
        std::fill(m_now.begin() + 2 * (ptrdiff_t)n, m_now.end(), 1.0);
        for (int i = 0; i < n; ++i) {
            const int64_t p = slot_particle[(size_t)i];
            if (p < 0) continue;
            const int64_t m = plan.member_of[(size_t)p];
            const simulation::ReducedMember &r = plan.red[(size_t)m];
            const int64_t lp = p - sp.member_offsets[m];
            ex[i] = sp.anisotropy_axis[3 * p];
            ey[i] = sp.anisotropy_axis[3 * p + 1];
            ez[i] = sp.anisotropy_axis[3 * p + 2];
            const double *m0 = sp.start_state ? sp.start_state : sp.magnetisation_direction;
            for (int d = 0; d < 3; ++d) m_now[(size_t)d * n + i] = m0[3 * p + d];
            k[i] = r.k_red[(size_t)lp];
            al[i] = sp.damping[m];
            dt[i] = r.dt;
            sr[i] = r.sr[(size_t)lp];
            sig[i] = r.sr[(size_t)lp] * std::sqrt(r.dt);
            happ[i] = r.happ;
            fred[i] = r.fapp;
            fdt[i] = r.fapp * r.dt;
            shape[i] = sp.field_shape[m];
            msw[i] = sp.magnetisation[m];
            key0[i] = (uint32_t)(uint64_t)sp.seed[m];
            key1[i] = (uint32_t)((uint64_t)sp.seed[m] >> 32);
            pid[i] = (uint32_t)lp;
            if (cluster) {
                // lib/simulation.cpp:577-583 and lib/field.cpp:212-215
                const double vroot = std::pow(r.average_volume, 1. / 3);
                px[i] = sp.location[3 * p] / vroot;
                py[i] = sp.location[3 * p + 1] / vroot;
                pz[i] = sp.location[3 * p + 2] / vroot;
                const double pre = kMU0 * sp.magnetisation[m] * sp.magnetisation[m] / 8.0 /
                                   kPiHost / r.average_anisotropy;
                w[i] = pre * r.v_red[(size_t)lp];
            }
            if (first) {
                shape_kind = shape[i];
                first = false;
            } else if (shape_kind != shape[i]) {
                shape_kind = (int)mp::kMixed;
            }
        }
        // the applied field from a table, where every particle of a schedule group
        // sees the same one (a constant needs none: its table is its amplitude)
        uniform_field = sizeof(T) == 4 && scheme == MP_SCHEME_HEUN && !first;
        for (int gi : set) uniform_field = uniform_field && group_field(sp, plan, gi).uniform;
        if (set.size() > 1 && shape_kind == (int)mp::kConstant) uniform_field = false;
        if (uniform_field) {
            // groups of four aligned below n0, one entry past the last step, and
            // the next group's prefetch: 4 * groups + 5 <= spl + 12
            // several: 64 MB of rows, or rows of 4,096 steps where those are more (16 KB a
            // group; a launch per group had rows of 512 KB)
            if (set.size() > 1)
                spl = std::min(spl, std::max((int64_t)4096, ((int64_t)1 << 24) / (int64_t)set.size()));
            tab_stride = spl + 16;
            std::vector<int> row_shape;
            std::vector<double> row_amp, row_fdt;
            for (int gi : set) {
                const GroupField f = group_field(sp, plan, gi);
                row_shape.push_back(f.shape);
                row_amp.push_back(f.amp);
                row_fdt.push_back(f.fdt);
            }
            d_field_shape.upload(row_shape);
            d_field_amp.upload(row_amp);
            d_field_fdt.upload(row_fdt);
            d_htab.alloc((size_t)tab_stride * set.size());
            if (set.size() > 1) {
                std::vector<int64_t> toff((size_t)n, 0);
                for (int i = 0; i < n; ++i) toff[(size_t)i] = tab_stride * slot_group[(size_t)i];
                d_toff.upload(toff);
            }
        }
        d_ex.upload(cast_vec<T>(ex));
        d_ey.upload(cast_vec<T>(ey));
        d_ez.upload(cast_vec<T>(ez));
        d_k.upload(cast_vec<T>(k));
        d_al.upload(cast_vec<T>(al));
        d_dt.upload(cast_vec<T>(dt));
        const bool implicit = scheme == MP_SCHEME_IMPLICIT_MIDPOINT;
        if (!implicit) d_sig.upload(cast_vec<T>(sig));
        d_sr.upload(cast_vec<T>(sr));
        d_happ.upload(cast_vec<T>(happ));
        d_m.upload(cast_vec<T>(m_now));
        d_fred.upload(fred);
        if (!implicit) d_fdt.upload(fdt);
        d_dtd.upload(dt);
        d_msw.upload(msw);
        d_shape.upload(shape);
        d_key0.upload(key0);
        d_key1.upload(key1);
        d_pid.upload(pid);
        d_status.upload(std::vector<uint32_t>((size_t)n, 0));
        d_sched.upload(sched);
        if (implicit)
            d_newton.upload(std::vector<unsigned long long>(2 * (size_t)n, 0));
        if (cluster) {
            d_px.upload(cast_vec<T>(px));
            d_py.upload(cast_vec<T>(py));
            d_pz.upload(cast_vec<T>(pz));
            d_w.upload(cast_vec<T>(w));
            if (!implicit) {
                d_cbase.upload(cbase);
                d_csize.upload(csize);
            }
        }
        // cluster slots come in whole blocks of block / lanes
        grid = cluster ? n_slots / (block / lanes) : (n + block - 1) / block;
        n_waves = (grid * block) / mp::kWave;
        const bool several = set.size() > 1;
        two_wave = !cluster && !array_noise && scheme == MP_SCHEME_HEUN
                       ? two_wave_mode(n_waves, sizeof(T) == 4)
                       : 0;
        // the one-wave kernel reads one table row
        if (several && uniform_field) two_wave = std::max(two_wave, 1);
        if (want_traj) n_samples = (size_t)S_out * 3 * (size_t)n;
        const size_t own_records = sole_set ? record_bytes() / sizeof(T) : 0;
        if (n_samples + own_records) d_samples.alloc(n_samples + own_records);
        if (own_records) records = d_samples.p + n_samples;
        if (want_ens) {
            // each recorded sample writes all of its (component, wave) slots;
            // slots of samples taken at step 0 are replaced on the host.  Several
            // schedules: a slot per group
            d_partial.alloc((size_t)S_out * 3 * ((several ? set.size() : (size_t)n_waves) + 1));
            if (several) {
                std::vector<int32_t> first(set.size() + 1, 0), slots;
                for (int g : slot_group)
                    if (g >= 0) ++first[(size_t)g + 1];
                for (size_t g = 0; g < set.size(); ++g) first[g + 1] += first[g];
                slots.resize((size_t)first.back());
                std::vector<int32_t> at(first.begin(), first.end() - 1);
                for (int i = 0; i < n; ++i)
                    if (slot_group[(size_t)i] >= 0)
                        slots[(size_t)at[(size_t)slot_group[(size_t)i]]++] = i;
                d_group_first.upload(first);
                d_group_slots.upload(slots);
            }
        }
        if (several && (want_traj || want_ens)) {
            std::vector<int32_t> flat;
            for (const auto &row : pick) flat.insert(flat.end(), row.begin(), row.end());
            d_pick.upload(flat);
            d_slot_group.upload(std::vector<int32_t>(slot_group.begin(), slot_group.end()));
        }
        if (array_noise) {
            std::vector<double> nz((size_t)n_total * (size_t)n * 3, 0.0);
            for (int64_t st = 0; st < n_total; ++st)
                for (int i = 0; i < n; ++i) {
                    const int64_t p = slot_particle[(size_t)i];
                    if (p < 0) continue;
                    for (int d = 0; d < 3; ++d)
                        nz[((size_t)st * n + i) * 3 + d] = sp.noise_array[((size_t)st * P + p) * 3 + d];
                }
            d_noise.upload(nz);
        }
        a.n = n;
        a.n_waves = n_waves;
        a.ex = d_ex.p; a.ey = d_ey.p; a.ez = d_ez.p;
        a.k = d_k.p; a.alpha = d_al.p; a.dt = d_dt.p; a.sig = d_sig.p; a.sr = d_sr.p;
        a.happ = d_happ.p; a.fred = d_fred.p; a.fdt = d_fdt.p; a.dtd = d_dtd.p;
        a.shape = d_shape.p;
        a.key0 = d_key0.p; a.key1 = d_key1.p; a.pid = d_pid.p;
        a.msw = d_msw.p;
        a.mx = d_m.p; a.my = d_m.p + n; a.mz = d_m.p + 2 * (size_t)n;
        a.status = d_status.p;
        a.sched = d_sched.p;
        a.S = S;
        a.samples = several ? records : d_samples.p;
        a.ens_partial = several ? nullptr : d_partial.p;
        a.tag = sp.noise_tag;
        a.renorm = sp.renorm ? 1 : 0;
        a.noise = array_noise ? d_noise.p : nullptr;
        a.toff = d_toff.p;
    }

    const std::vector<int64_t> &slots() const override { return slot_particle; }
    const std::vector<int> &set() const override { return groups; }

    size_t record_bytes() const override
    {
        const bool shared = groups.size() > 1 && (want_traj || want_ens) && records == nullptr;
        return shared ? (size_t)S * 3 * (size_t)n * sizeof(T) : 0;
    }
    void use_records(void *p) override
    {
        if (record_bytes() == 0) return;
        records = static_cast<T *>(p);
        a.samples = records;
    }
    // the sums [S_out][3] of the set, behind its partial sums
    double *ens_sums() const { return d_partial.p + (d_partial.n - (size_t)S_out * 3); }

    // The samples and sums of the records that a launch of the steps up to n1 wrote:
    // those from s_next on.  A group takes a sample at one step, so that its sum has
    // all its terms here and does not depend on how a run is cut into launches.
    void take_records(int64_t n1, hipStream_t s)
    {
        const int32_t first = (int32_t)s_next,
                      end = (int32_t)(std::upper_bound(sched.begin() + s_next, sched.end(), n1) -
                                      sched.begin());
        if (first == end) return;
        int64_t lo = S_out, hi = 0;   // the samples that any group has there
        for (const auto &row : pick) {
            lo = std::min<int64_t>(lo, std::lower_bound(row.begin(), row.end(), first) - row.begin());
            hi = std::max<int64_t>(hi, std::lower_bound(row.begin(), row.end(), end) - row.begin());
        }
        if (lo >= hi) return;
        const int64_t G = (int64_t)groups.size(), most = 16 * (int64_t)device_cus();
        auto blocks = [&](bool wanted, int64_t threads) {
            return wanted ? (int)std::min((threads + mp::kBlock - 1) / mp::kBlock, most) : 0;
        };
        const mp::RecordArgs<T> r{records, d_pick.p, n, S_out, lo, hi, first, end};
        int team = 1;   // lanes per sum: the slots of a group on average, to a wave
        while (team < mp::kWave && team * G < (int64_t)d_group_slots.n) team *= 2;
        const mp::GroupSums q{d_group_slots.p, d_group_first.p, (int)G, team, d_msw.p, d_partial.p};
        const int sample_blocks = blocks(want_traj, (hi - lo) * n);
        const int sum_blocks = blocks(want_ens, (hi - lo) * G * team);
        hipLaunchKernelGGL(mp::take_records_kernel<T>, dim3((unsigned)(sample_blocks + sum_blocks)),
                           dim3(mp::kBlock), 0, s, r, d_slot_group.p, d_samples.p, sample_blocks, q);
        MP_HIP(hipGetLastError());
    }

    unsigned long long *newton_iters() const { return d_newton.p; }
    unsigned long long *newton_fails() const { return d_newton.p ? d_newton.p + n : nullptr; }

    void launch_cluster(hipStream_t s, const float *htab)
    {
        if constexpr (sizeof(T) == 8) {
            if (scheme == MP_SCHEME_IMPLICIT_MIDPOINT) {
                if (array_noise) launch_implicit_cluster<true>(s);
                else launch_implicit_cluster<false>(s);
                return;
            }
        }
        if (array_noise) launch_cluster_lanes<1, true>(s, htab);  // one lane per slot
        else if (lanes == 2) launch_cluster_lanes<2, false>(s, htab);
        else launch_cluster_lanes<1, false>(s, htab);
    }

    // Partners whose geometry the two-lane kernel caches per lane (in workgroups of
    // at most 256 lanes): 16 in FP32 and 8 in FP64, or 0 with
    // MAGPY_AMD_CLUSTER_CACHE=0.  Results do not depend on it.
    int cluster_cache() const
    {
        if (lanes != 2 || block > 256 || array_noise) return 0;
        if (const char *env = std::getenv("MAGPY_AMD_CLUSTER_CACHE"))
            if (std::atoi(env) == 0) return 0;
        return sizeof(T) == 4 ? 16 : 8;
    }

    template <bool kArray>
    void launch_implicit_cluster(hipStream_t s)
    {
        mp::ImplicitClusterArgs ia{
            mp::ClusterArgs<double>{a, d_px.p, d_py.p, d_pz.p, d_w.p, nullptr, nullptr}, d_row.p,
            d_cell.p, eps, max_iter, newton_iters(), newton_fails(), interactions ? 1 : 0};
        // a source per slot, a sum per `targets` slots, a flag per slot
        const size_t shmem = (size_t)block * (sizeof(mp::Source) + sizeof(int)) +
                             (size_t)(block / targets) * sizeof(double);
        auto go = [&](auto kernel) {
            hipLaunchKernelGGL(kernel, dim3(grid), dim3(block), shmem, s, ia);
        };
        auto shaped = [&](auto one_wave, auto kt) {
            constexpr bool W = decltype(one_wave)::value;
            constexpr int KT = decltype(kt)::value;
            switch (shape_kind) {
            case mp::kSine: go(mp::implicit_cluster_kernel<mp::kSine, kArray, W, KT>); break;
            case mp::kSquare: go(mp::implicit_cluster_kernel<mp::kSquare, kArray, W, KT>); break;
            case mp::kConstant: go(mp::implicit_cluster_kernel<mp::kConstant, kArray, W, KT>); break;
            default: go(mp::implicit_cluster_kernel<mp::kMixed, kArray, W, KT>); break;
            }
        };
        using Two = std::integral_constant<int, 2>;
        using Four = std::integral_constant<int, 4>;
        if (block == mp::kWave) {
            if (targets == 2) shaped(std::true_type{}, Two{});
            else shaped(std::true_type{}, Four{});
        } else {
            if (targets == 2) shaped(std::false_type{}, Two{});
            else shaped(std::false_type{}, Four{});
        }
    }

    template <int L, bool kArray>
    void launch_cluster_lanes(hipStream_t s, const float *htab)
    {
        if constexpr (L == 2 && !kArray && sizeof(T) == 8) {
            if (cluster_cache() != 0) {
                launch_cluster_variant<L, kArray, 8, 0>(s, htab);
                return;
            }
        }
        if constexpr (L == 2 && !kArray && sizeof(T) == 4) {
            if (cluster_cache() != 0) {
                if (cluster_lds_cache()) launch_cluster_variant<L, kArray, 16, 16>(s, htab);
                else launch_cluster_variant<L, kArray, 16, 0>(s, htab);
                return;
            }
        }
        launch_cluster_variant<L, kArray, 0, 0>(s, htab);
    }

    // the 16 partners after the register-cached ones keep their weights in
    // LDS (MAGPY_AMD_CLUSTER_LDS_CACHE=0: recomputed, the same bits)
    static bool cluster_lds_cache()
    {
        const char *env = std::getenv("MAGPY_AMD_CLUSTER_LDS_CACHE");
        return !(env != nullptr && std::atoi(env) == 0);
    }

    template <int L, bool kArray, int KC, int KL>
    void launch_cluster_variant(hipStream_t s, const float *htab)
    {
        mp::ClusterArgs<T> ca{a, d_px.p, d_py.p, d_pz.p, d_w.p, d_cbase.p, d_csize.p};
        const size_t shmem = 3 * (size_t)(block / L) * sizeof(mp::Vec4<T>) +
                             (size_t)KL * (size_t)block * sizeof(float2);
        auto go = [&](auto kernel) {
            hipLaunchKernelGGL(kernel, dim3(grid), dim3(block), shmem, s, ca, htab);
        };
        const bool rn = a.renorm != 0;
        if (htab) {
            if (rn) go(mp::heun_cluster_kernel<T, mp::kConstant, true, true, L, kArray, KC, KL>);
            else go(mp::heun_cluster_kernel<T, mp::kConstant, true, false, L, kArray, KC, KL>);
            return;
        }
        switch (shape_kind) {
        case mp::kSine:
            if (rn) go(mp::heun_cluster_kernel<T, mp::kSine, false, true, L, kArray, KC, KL>);
            else go(mp::heun_cluster_kernel<T, mp::kSine, false, false, L, kArray, KC, KL>);
            break;
        case mp::kSquare:
            if (rn) go(mp::heun_cluster_kernel<T, mp::kSquare, false, true, L, kArray, KC, KL>);
            else go(mp::heun_cluster_kernel<T, mp::kSquare, false, false, L, kArray, KC, KL>);
            break;
        case mp::kConstant:
            if (rn) go(mp::heun_cluster_kernel<T, mp::kConstant, false, true, L, kArray, KC, KL>);
            else go(mp::heun_cluster_kernel<T, mp::kConstant, false, false, L, kArray, KC, KL>);
            break;
        default:
            if (rn) go(mp::heun_cluster_kernel<T, mp::kMixed, false, true, L, kArray, KC, KL>);
            else go(mp::heun_cluster_kernel<T, mp::kMixed, false, false, L, kArray, KC, KL>);
            break;
        }
    }

    void enqueue(int64_t upto, hipStream_t s) override
    {
        upto = std::min(upto, n_total);
        while (n_done < upto) {
            const int64_t n1 = std::min(upto, n_done + spl);
            while (s_next < S && sched[(size_t)s_next] < n_done + 1) ++s_next;
            a.n0 = n_done;
            a.n1 = n1;
            a.s_next = s_next;
            const float *htab = nullptr;
            if (uniform_field) {
                const int64_t g0 = n_done >> 2, g1 = (n1 + 3) >> 2;
                const int64_t count = 4 * (g1 - g0) + 5;
                require(count <= tab_stride, "field table too small");
                const int64_t per_row = (count + 255) / 256;
                hipLaunchKernelGGL(mp::field_table_kernel,
                                   dim3((unsigned)(per_row * (int64_t)groups.size())), dim3(256), 0,
                                   s, d_field_shape.p, d_field_amp.p, d_field_fdt.p, 4 * g0, count,
                                   (int)per_row, tab_stride, d_htab.p);
                MP_HIP(hipGetLastError());
                htab = d_htab.p;
            }
            if (cluster)
                launch_cluster(s, htab);
            else if (array_noise)
                launch_shape<T, true>(shape_kind, a, scheme, eps, max_iter, newton_iters(), newton_fails(), grid, s,
                                      htab, false);
            else
                launch_shape<T, false>(shape_kind, a, scheme, eps, max_iter, newton_iters(), newton_fails(), grid, s,
                                       htab, two_wave);
            MP_HIP(hipGetLastError());
            if (records != nullptr) take_records(n1, s);
            ++launches;
            n_done = n1;
        }
    }

    void state(double *out) override
    {
        std::unique_ptr<T[]> h(new T[3 * (size_t)n]);
        MP_HIP(hipMemcpy(h.get(), d_m.p, 3 * (size_t)n * sizeof(T), hipMemcpyDeviceToHost));
        for (int i = 0; i < n; ++i) {
            const int64_t p = slot_particle[(size_t)i];
            if (p < 0) continue;
            for (int d = 0; d < 3; ++d) out[3 * p + d] = (double)h[(size_t)d * n + i];
        }
    }

    GroupOut collect(hipStream_t s, double *state_out, const SampleSink *sink) override
    {
        GroupOut o;
        if (want_ens) {
            auto go = [&](auto kernel, int parts) {
                hipLaunchKernelGGL(kernel, dim3((unsigned)(S_out * 3)), dim3(mp::kBlock), 0, s,
                                   d_partial.p, parts, S_out * 3, ens_sums(), d_pick.p);
                MP_HIP(hipGetLastError());
            };
            if (groups.size() > 1) go(mp::ens_reduce_kernel<true>, (int)groups.size());
            else go(mp::ens_reduce_kernel<false>, n_waves);
        }
        MP_HIP(hipStreamSynchronize(s));
        if (state_out) state(state_out);
        o.status.resize((size_t)n);
        MP_HIP(hipMemcpy(o.status.data(), d_status.p, n * sizeof(uint32_t), hipMemcpyDeviceToHost));
        if (d_newton.p) {
            std::vector<unsigned long long> c(2 * (size_t)n);
            MP_HIP(hipMemcpy(c.data(), d_newton.p, c.size() * sizeof(unsigned long long),
                             hipMemcpyDeviceToHost));
            for (int i = 0; i < n; ++i) {
                o.newton_iters += (int64_t)c[(size_t)i];
                o.newton_fail += (int64_t)c[(size_t)(n + i)];
            }
        }
        if (sink != nullptr && want_traj) {
            std::unique_ptr<T[]> h(new T[n_samples]);
            if (n_samples)
                MP_HIP(hipMemcpy(h.get(), d_samples.p, n_samples * sizeof(T),
                                 hipMemcpyDeviceToHost));
            sink->take(h.get(), slot_particle);
        }
        if (want_ens) {
            o.ens.resize((size_t)S_out * 3);
            MP_HIP(hipMemcpy(o.ens.data(), ens_sums(), o.ens.size() * sizeof(double),
                             hipMemcpyDeviceToHost));
        }
        return o;
    }
};

// ------------------------------------------------------------------ replicas
int pad_to(int64_t x, int64_t q) { return (int)((x + q - 1) / q * q); }

// Dipole tensor of one cluster in reduced units (lib/field.cpp:187-225,
// lib/simulation.cpp:577-583): D[(i,a)][(j,b)] = w_j r^-3 (3 u_a u_b - d_ab),
// w_j = mu0 Ms^2 / (8 pi K_avg) v_j / V_avg, rows and columns in the
// replica_col order, leading dimension ld, zero padded.
void dipole_tensor(const simulation::ReducedMember &r, const double *loc, double ms, size_t n,
                   int ld, std::vector<double> &D)
{
    const double vroot = std::pow(r.average_volume, 1. / 3);
    const double pre = kMU0 * ms * ms / 8.0 / kPiHost / r.average_anisotropy;
    D.assign((size_t)ld * ld, 0.0);
    for (size_t i = 0; i < n; ++i)
        for (size_t j = 0; j < n; ++j) {
            if (i == j) continue;
            double d[3], rr = 0.0;
            for (int a = 0; a < 3; ++a) {
                d[a] = (loc[3 * j + a] - loc[3 * i + a]) / vroot;
                rr += d[a] * d[a];
            }
            rr = std::sqrt(rr);
            const double c = pre * r.v_red[j] / (rr * rr * rr);
            for (int a = 0; a < 3; ++a)
                for (int b = 0; b < 3; ++b)
                    D[(size_t)mp::replica_col((int)i, a) * ld + mp::replica_col((int)j, b)] =
                        c * (3 * (d[a] / rr) * (d[b] / rr) - (a == b ? 1.0 : 0.0));
        }
}

// The tensor as the product's fragments (replica_fragment): BF16 hi and lo, or FP32.
std::vector<float> tensor_fragments(const std::vector<double> &D, int ld, int mode)
{
    std::vector<float> out((size_t)ld * ld);
    for (int pb = 0; pb < ld / 96; ++pb)
        for (int ks = 0; ks < ld / 16; ++ks)
            for (int u = 0; u < 3; ++u) {
                char *const part[2] = {
                    reinterpret_cast<char *>(out.data() + 4 * mp::replica_fragment(ld, pb, ks, u, 0)),
                    reinterpret_cast<char *>(out.data() + 4 * mp::replica_fragment(ld, pb, ks, u, 1))};
                for (int l = 0; l < mp::kWave; ++l)
                    for (int j = 0; j < 8; ++j) {
                        const int row = 96 * pb + 32 * u + (l & 31);
                        const float x = (float)D[(size_t)row * ld + mp::replica_k(ks, l, j)];
                        if (mode == MP_DIPOLAR_GEMM_F32) {
                            std::memcpy(part[j >> 2] + 16 * l + 4 * (j & 3), &x, sizeof(x));
                        } else {
                            const __bf16 hi = (__bf16)x, lo = (__bf16)(x - (float)hi);
                            std::memcpy(part[0] + 16 * l + 2 * j, &hi, sizeof(hi));
                            std::memcpy(part[1] + 16 * l + 2 * j, &lo, sizeof(lo));
                        }
                    }
            }
    return out;
}

// Replica layout sizes: particles padded to a multiple of kParticlePad
// (ld = 3 Np), replicas to a multiple of the rows of a block.
int replica_ld(int64_t n) { return 3 * pad_to(n, mp::kParticlePad); }
int replica_rows(int64_t reps) { return pad_to(reps, mp::kReplicaPad); }

// Which panels the blocks that one XCD runs share: 1 (default) the row
// panels of the state, so each XCD reads an eighth of it and all of the
// tensor (100 MB of L2 fills per 4096 x 1536 product instead of 209 MB);
// 0 (MAGPY_AMD_REPLICA_PANELS=cols) the column panels of the tensor.
int replica_row_panels()
{
    static const int v = [] {
        const char *e = std::getenv("MAGPY_AMD_REPLICA_PANELS");
        return e != nullptr && std::string(e) == "cols" ? 0 : 1;
    }();
    return v;
}

// The product runs the Heun stages in its epilogue unless
// MAGPY_AMD_REPLICA_FUSED=0 when the run is created (then it writes the
// field and separate stage kernels follow; the two give the same bits).
bool replica_fused()
{
    const char *e = std::getenv("MAGPY_AMD_REPLICA_FUSED");
    return !(e != nullptr && std::string(e) == "0");
}

// One product with the epilogue `epi` (replica_product_kernel).  Blocks of four wave
// pairs of 64 replicas share most, but a CU takes one: below a block per CU, blocks
// of one pair; and where pairs of 32 replicas still fit the card at once (two waves
// per SIMD), those, whose sums take half as long.  The sums are the same in all.
// 512 steps, ms (start: blocks of 8 waves whatever the size, particles padded to 128)
// with blocks of four pairs, pairs of 64 and pairs of 32 replicas:
//   1,000 x 64   24.0   14.5  9.8  6.4      4,096 x 256  51.7  31.7  28.8  25.7
//   64 x 400     58.7   42.1  22.3  13.9    2,048 x 512  74.4  51.6  45.0  43.0
//   1,024 x 256  37.1   28.1  16.7  10.3    3,900 x 450  86.0    -   68.5  94.7
//   4,096 x 512  92.4  70.9  75.5  -  (with the state's copy: 70.7 -> 63.8 us a product)
void launch_product(int mode, int epi, const float *state, const float *tensor,
                    const mp::ReplicaArgs &a, int rows, int cus, int64_t step, float hstage,
                    int64_t s_first, int n_rec, hipStream_t s)
{
    require(rows % mp::kReplicaPad == 0 && a.ld % (3 * mp::kParticlePad) == 0,
            "replica product: rows or ld do not fit the tiles");
    auto go = [&](auto kernel, auto w, auto t) {
        constexpr int W = decltype(w)::value, KT = decltype(t)::value;
        const int nrb = rows / (32 * KT * W), ncb = a.ld / (96 * W);
        hipLaunchKernelGGL(kernel, dim3((unsigned)(nrb * ncb)), dim3(128 * W * W), 0, s, state,
                           reinterpret_cast<const mp::f32x4 *>(tensor), a, step, hstage, s_first,
                           n_rec, nrb, ncb, replica_row_panels());
    };
    using One = std::integral_constant<int, 1>;
    using Two = std::integral_constant<int, 2>;
    auto with_epilogue = [&](auto m, auto w, auto t) {
        constexpr int M = decltype(m)::value, W = decltype(w)::value, KT = decltype(t)::value;
        if (epi == 0) go(mp::replica_product_kernel<M, 0, W, KT>, w, t);
        else if (epi == 1) go(mp::replica_product_kernel<M, 1, W, KT>, w, t);
        else go(mp::replica_product_kernel<M, 2, W, KT>, w, t);
    };
    const int64_t pairs = (int64_t)(rows / 64) * (a.ld / 96);
    auto with_mode = [&](auto m) {
        if (pairs >= 4 * (int64_t)cus) with_epilogue(m, Two{}, Two{});
        else if (pairs > 2 * (int64_t)cus) with_epilogue(m, One{}, Two{});
        else with_epilogue(m, One{}, One{});
    };
    if (mode == MP_DIPOLAR_GEMM_F32) with_mode(std::integral_constant<int, mp::kReplicaF32>{});
    else with_mode(std::integral_constant<int, mp::kReplicaBf16x3>{});
    MP_HIP(hipGetLastError());
}

// All members are one cluster replicated: two products per Heun step, with the
// stages in their epilogues or in kernels of their own.
struct ReplicaRun : GroupBase {
    int n = 0, reps = 0, ld = 0, rows = 0, mode = MP_DIPOLAR_GEMM_BF16X3, n_waves = 0, cus = 0;
    bool fused = false;
    int shape = MP_FIELD_CONSTANT;
    double happ = 0.0, fapp = 0.0, dt = 0.0;
    bool want_traj = false, want_ens = false;
    int64_t S = 0, s_next = 0;
    std::vector<int64_t> sched, slot_particle;
    DevBuf<float> d_m, d_mt, d_h, d_nz, d_kex, d_key, d_kez, d_edx, d_edy, d_edz, d_sig,
        d_tensor, d_samples;
    DevBuf<uint32_t> d_key0, d_key1, d_status;
    DevBuf<double> d_msw, d_partial, d_ens;
    DevBuf<int64_t> d_sched;
    mp::ReplicaArgs a{};

    ReplicaRun(const simulation::EnsembleSpec &sp, const Plan &plan, bool traj, bool ens, int m)
    {
        mode = m;
        cus = device_cus();
        fused = replica_fused();
        reps = (int)sp.n_members;
        n = (int)(sp.member_offsets[1] - sp.member_offsets[0]);
        ld = replica_ld(n);
        rows = replica_rows(reps);
        sched = plan.sched[0];
        S = (int64_t)sched.size();
        n_total = plan.group_steps[0];
        want_traj = traj;
        want_ens = ens;
        const simulation::ReducedMember &r = plan.red[0];
        shape = sp.field_shape[0];
        happ = r.happ;
        fapp = r.fapp;
        dt = r.dt;
        slot_particle.resize((size_t)reps * n);
        for (int rr = 0; rr < reps; ++rr)
            for (int p = 0; p < n; ++p)
                slot_particle[(size_t)rr * n + p] = sp.member_offsets[rr] + p;
        // per-particle parameters (identical across replicas)
        std::vector<double> kex(n), key(n), kez(n), edx(n), edy(n), edz(n), sig(n);
        for (int p = 0; p < n; ++p) {
            const double *e = sp.anisotropy_axis + 3 * p;
            kex[p] = r.k_red[p] * e[0];
            key[p] = r.k_red[p] * e[1];
            kez[p] = r.k_red[p] * e[2];
            edx[p] = e[0] * r.dt;
            edy[p] = e[1] * r.dt;
            edz[p] = e[2] * r.dt;
            sig[p] = r.sr[p] * std::sqrt(r.dt);
        }
        d_kex.upload(cast_vec<float>(kex));
        d_key.upload(cast_vec<float>(key));
        d_kez.upload(cast_vec<float>(kez));
        d_edx.upload(cast_vec<float>(edx));
        d_edy.upload(cast_vec<float>(edy));
        d_edz.upload(cast_vec<float>(edz));
        d_sig.upload(cast_vec<float>(sig));
        std::vector<uint32_t> k0(reps), k1(reps);
        std::vector<double> msw(reps);
        for (int rr = 0; rr < reps; ++rr) {
            k0[rr] = (uint32_t)(uint64_t)sp.seed[rr];
            k1[rr] = (uint32_t)((uint64_t)sp.seed[rr] >> 32);
            msw[rr] = sp.magnetisation[rr];
        }
        d_key0.upload(k0);
        d_key1.upload(k1);
        d_msw.upload(msw);
        // dipole tensor and its split
        std::vector<double> D;
        dipole_tensor(r, sp.location, sp.magnetisation[0], (size_t)n, ld, D);
        d_tensor.upload(tensor_fragments(D, ld, mode));
        // state, zero padded
        std::vector<float> m0((size_t)rows * ld, 0.f);
        const double *src = sp.start_state ? sp.start_state : sp.magnetisation_direction;
        for (int rr = 0; rr < reps; ++rr)
            for (int p = 0; p < n; ++p)
                for (int c = 0; c < 3; ++c)
                    m0[mp::replica_at(ld, rr, mp::replica_col(p, c))] =
                        (float)src[3 * (sp.member_offsets[rr] + p) + c];
        n_done = std::min(sp.start_step, n_total);
        d_m.upload(m0);
        d_mt.upload(std::vector<float>(m0.size(), 0.f));
        // the fused product keeps the field on chip and passes the step's
        // increments from stage 1 to stage 2; the separate stages pass the field
        if (fused) d_nz.upload(std::vector<float>(m0.size(), 0.f));
        else d_h.upload(std::vector<float>(m0.size(), 0.f));
        d_status.upload(std::vector<uint32_t>((size_t)reps * n, 0));
        d_sched.upload(sched);
        const int threads = reps * n;
        // ensemble partials: one per 32 replicas x 32 particles of the product, or per
        // wave of the stage kernels
        n_waves = (rows / 32) * (ld / 96) * (fused ? 1 : 16);
        if (want_traj) d_samples.alloc((size_t)S * 3 * (size_t)threads);
        if (want_ens) {
            d_partial.alloc((size_t)S * 3 * (size_t)n_waves);
            d_ens.alloc((size_t)S * 3);
        }
        a.n = n;
        a.reps = reps;
        a.ld = ld;
        a.n_waves = n_waves;
        a.kex = d_kex.p; a.key = d_key.p; a.kez = d_kez.p;
        a.edx = d_edx.p; a.edy = d_edy.p; a.edz = d_edz.p;
        a.sig = d_sig.p;
        a.dt = (float)r.dt;
        a.alpha = (float)sp.damping[0];
        a.key0 = d_key0.p; a.key1 = d_key1.p;
        a.msw = d_msw.p;
        a.tag = sp.noise_tag;
        a.renorm = sp.renorm ? 1 : 0;
        a.m = d_m.p; a.mt = d_mt.p; a.h = d_h.p; a.nz = d_nz.p;
        a.status = d_status.p;
        a.sched = d_sched.p;
        a.S = S;
        a.samples = want_traj ? d_samples.p : nullptr;
        a.ens_partial = want_ens ? d_partial.p : nullptr;
    }

    const std::vector<int64_t> &slots() const override { return slot_particle; }
    const std::vector<int> &set() const override
    {
        static const std::vector<int> only{0};
        return only;
    }

    void enqueue(int64_t upto, hipStream_t s) override
    {
        upto = std::min(upto, n_total);
        const dim3 grid((unsigned)((rows / 32) * (ld / 96) * 4));   // stage kernels
        while (n_done < upto) {
            const int64_t st = n_done;
            const double t1 = (double)(st + 1) * dt;
            const float h1 = (float)applied_host(shape, happ, fapp, t1);
            const float h2 = (float)applied_host(shape, happ, fapp, t1 + dt);
            while (s_next < S && sched[(size_t)s_next] < st + 1) ++s_next;
            int n_rec = 0;
            while (s_next + n_rec < S && sched[(size_t)(s_next + n_rec)] == st + 1) ++n_rec;
            if (fused) {
                launch_product(mode, 1, d_m.p, d_tensor.p, a, rows, cus, st, h1, 0, 0, s);
                launch_product(mode, 2, d_mt.p, d_tensor.p, a, rows, cus, st, h2, s_next, n_rec, s);
            } else {
                launch_product(mode, 0, d_m.p, d_tensor.p, a, rows, cus, st, 0.f, 0, 0, s);
                hipLaunchKernelGGL(mp::replica_stage1_kernel, grid, dim3(256), 0, s, a, st, h1);
                launch_product(mode, 0, d_mt.p, d_tensor.p, a, rows, cus, st, 0.f, 0, 0, s);
                hipLaunchKernelGGL(mp::replica_stage2_kernel, grid, dim3(256), 0, s, a, st, h2,
                                   s_next, n_rec);
            }
            MP_HIP(hipGetLastError());
            ++launches;
            n_done = st + 1;
        }
    }

    // The device packs the live columns to [reps n][3] in a buffer that is free
    // between steps (the increments, or the field); the host widens them piece by
    // piece.  4,096 x 512: 22 -> 6 ms against the padded rows repacked on the host.
    void state(double *out) override
    {
        const int64_t total = 3 * (int64_t)reps * n, piece = (int64_t)1 << 20;
        float *packed = fused ? d_nz.p : d_h.p;
        hipLaunchKernelGGL(mp::replica_pack_kernel, dim3((unsigned)((reps * n + 255) / 256)),
                           dim3(256), 0, nullptr, a, packed);
        MP_HIP(hipGetLastError());
        std::unique_ptr<float[]> h(new float[(size_t)std::min(total, piece)]);
        for (int64_t o = 0; o < total; o += piece) {
            const int64_t len = std::min(piece, total - o);
            MP_HIP(hipMemcpy(h.get(), packed + o, (size_t)len * sizeof(float),
                             hipMemcpyDeviceToHost));
            for (int64_t i = 0; i < len; ++i) out[o + i] = (double)h[(size_t)i];
        }
    }

    GroupOut collect(hipStream_t s, double *state_out, const SampleSink *sink) override
    {
        GroupOut o;
        if (want_ens) {
            hipLaunchKernelGGL(mp::ens_reduce_kernel<false>, dim3((unsigned)(S * 3)), dim3(mp::kBlock), 0,
                               s, d_partial.p, n_waves, S * 3, d_ens.p, nullptr);
            MP_HIP(hipGetLastError());
        }
        MP_HIP(hipStreamSynchronize(s));
        if (state_out) state(state_out);
        o.status.resize((size_t)reps * n);
        MP_HIP(hipMemcpy(o.status.data(), d_status.p, o.status.size() * sizeof(uint32_t),
                         hipMemcpyDeviceToHost));
        if (sink != nullptr && want_traj) {
            std::unique_ptr<float[]> h(new float[d_samples.n]);
            if (d_samples.n)
                MP_HIP(hipMemcpy(h.get(), d_samples.p, d_samples.n * sizeof(float),
                                 hipMemcpyDeviceToHost));
            sink->take(h.get(), slot_particle);
        }
        if (want_ens) {
            o.ens.resize((size_t)S * 3);
            MP_HIP(hipMemcpy(o.ens.data(), d_ens.p, o.ens.size() * sizeof(double),
                             hipMemcpyDeviceToHost));
        }
        return o;
    }
};

// Every member is the same cluster: only seeds and initial states differ.
bool shared_geometry(const simulation::EnsembleSpec &sp)
{
    const int64_t n = sp.member_offsets[1] - sp.member_offsets[0];
    for (int64_t m = 1; m < sp.n_members; ++m) {
        const int64_t b = sp.member_offsets[m];
        if (sp.member_offsets[m + 1] - b != n) return false;
        if (sp.magnetisation[m] != sp.magnetisation[0] || sp.damping[m] != sp.damping[0] ||
            sp.temperature[m] != sp.temperature[0] || sp.field_shape[m] != sp.field_shape[0] ||
            sp.field_amplitude[m] != sp.field_amplitude[0] ||
            sp.field_frequency[m] != sp.field_frequency[0])
            return false;
        for (int64_t p = 0; p < n; ++p) {
            if (sp.radius[b + p] != sp.radius[p] || sp.anisotropy[b + p] != sp.anisotropy[p])
                return false;
            for (int c = 0; c < 3; ++c)
                if (sp.location[3 * (b + p) + c] != sp.location[3 * p + c] ||
                    sp.anisotropy_axis[3 * (b + p) + c] != sp.anisotropy_axis[3 * p + c])
                    return false;
        }
    }
    return true;
}

}  // namespace

struct mp_session {
    Plan plan;
    HostCopy host;
    std::vector<std::unique_ptr<GroupBase>> groups;
    DevBuf<char> records;   // shared by the launch sets of several schedules
    StreamGuard sg;
    // own_stream false: launches go to the null stream and nothing is created
    explicit mp_session(bool own_stream = true) : sg(own_stream) {}
    bool want_traj = false, want_ens = false;
    int device = 0;
    int cluster_block = 0;
    int cluster_lanes = 0;
    int dipolar = 0;
    double kernel_ms = 0.0;
};

namespace simulation {

ReducedMember reduce_member(const double *radius, const double *anisotropy, size_t n,
                            double magnetisation, double damping, double temperature,
                            double time_step, double end_time, double field_amplitude,
                            double field_frequency)
{
#pragma clang fp contract(off)
    ReducedMember r;
    std::vector<double> volume(n);
    for (size_t p = 0; p < n; ++p)
        volume[p] = 4.0 / 3.0 * kPiHost * radius[p] * radius[p] * radius[p];
    double vsum = 0.0;
    for (size_t p = 0; p < n; ++p) vsum += volume[p];
    r.average_volume = vsum / (double)n;
    double ksum = 0.0;
    for (size_t p = 0; p < n; ++p) ksum += anisotropy[p];
    r.average_anisotropy = ksum / (double)n;
    r.v_red.resize(n);
    r.k_red.resize(n);
    r.sr.resize(n);
    for (size_t p = 0; p < n; ++p) {
        r.v_red[p] = volume[p] / r.average_volume;
        r.k_red[p] = anisotropy[p] / r.average_anisotropy;
        r.sr[p] = std::sqrt(damping * kKB * temperature / (r.average_anisotropy * volume[p]) /
                            (1 + damping * damping));
    }
    r.anisotropy_field = 2 * r.average_anisotropy / kMU0 / magnetisation;
    r.time_factor = kGYROMAG * kMU0 * r.anisotropy_field / (1 + damping * damping);
    r.dt = time_step * r.time_factor;
    r.end_time = end_time * r.time_factor;
    r.happ = field_amplitude / r.anisotropy_field;
    r.fapp = field_frequency / r.time_factor;
    return r;
}

int64_t sample_schedule(double dt, double end_time, int64_t max_samples, std::vector<int64_t> &k)
{
    // The reference's loop (lib/simulation.cpp:342-406) steps while
    // t = step*dt <= s*Ts and records the state one step before it stopped;
    // here the first such step is found by search instead of by stepping.
    k.assign((size_t)max_samples, 0);
    if (max_samples <= 1) return 0;
    const double ts = end_time / (double)(max_samples - 1);
    int64_t step = 0;
    double t = 0.0;
    for (int64_t s = 1; s < max_samples; ++s) {
        const double x = (double)s * ts;
        if (t <= x) {
            double guess = std::floor(x / dt);
            int64_t j = guess > 9.0e18 ? INT64_MAX / 2 : (int64_t)guess;
            if (j < step + 1) j = step + 1;
            while ((double)j * dt <= x) ++j;
            while (j - 1 > step && (double)(j - 1) * dt > x) --j;
            step = j;
            t = (double)step * dt;
        }
        k[(size_t)s] = step - 1;
    }
    return step;
}

void validate(const EnsembleSpec &sp)
{
    require(sp.n_members >= 1, "n_members must be >= 1");
    require(sp.member_offsets != nullptr, "member_offsets is required");
    require(sp.member_offsets[0] == 0, "member_offsets[0] must be 0");
    for (int64_t m = 0; m < sp.n_members; ++m)
        require(sp.member_offsets[m + 1] > sp.member_offsets[m],
                "every member needs at least one particle");
    const int64_t P = sp.member_offsets[sp.n_members];
    require(P <= (int64_t)INT32_MAX, "too many particles for one call");
    require(sp.radius && sp.anisotropy && sp.anisotropy_axis && sp.magnetisation_direction &&
                sp.location,
            "particle arrays are required");
    require(sp.magnetisation && sp.damping && sp.temperature && sp.field_shape &&
                sp.field_amplitude && sp.field_frequency && sp.seed,
            "member arrays are required");
    require(sp.max_samples >= 1,
            "max_samples must be >= 1 (-1 never terminates in the reference loop)");
    require(sp.time_step > 0 && std::isfinite(sp.time_step), "time_step must be > 0");
    require(sp.end_time >= 0 && std::isfinite(sp.end_time), "end_time must be >= 0");
    require(sp.scheme == MP_SCHEME_HEUN || sp.scheme == MP_SCHEME_IMPLICIT_MIDPOINT,
            "unknown scheme");
    require(sp.precision == MP_PRECISION_FP32 || sp.precision == MP_PRECISION_FP64,
            "unknown precision");
    require(sp.noise == MP_NOISE_PHILOX || sp.noise == MP_NOISE_ARRAY, "unknown noise source");
    require(sp.dipolar >= MP_DIPOLAR_AUTO && sp.dipolar <= MP_DIPOLAR_GEMM_F32,
            "unknown dipolar mode");
    require(sp.start_step >= 0, "start_step must be >= 0");
    require(sp.noise != MP_NOISE_ARRAY || sp.noise_array != nullptr,
            "noise_array is required for MP_NOISE_ARRAY");
    for (int64_t m = 0; m < sp.n_members; ++m) {
        const int fs = sp.field_shape[m];
        require(fs == MP_FIELD_SINE || fs == MP_FIELD_SQUARE || fs == MP_FIELD_CONSTANT,
                "Must specify valid field::options enum");
        require(sp.magnetisation[m] > 0 && sp.damping[m] >= 0 && sp.temperature[m] >= 0,
                "magnetisation must be > 0, damping and temperature >= 0");
    }
}

}  // namespace simulation

namespace {

// The smallest power-of-two block of at least one wave whose slots hold the
// largest cluster (0: none up to max_block lanes).
int cluster_min_block(int64_t nmax, int lanes, int max_block = 1024)
{
    for (int b = mp::kWave; b <= max_block; b *= 2)
        if (b / lanes >= nmax) return b;
    return 0;
}

// What the cluster kernels of a run allow: the implicit midpoint kernel and
// caller-given noise run one lane per slot; the implicit kernel's workgroups
// hold at most kImplicitClusterBlock lanes (FP64 Newton state per lane).
struct ClusterLimits {
    bool one_lane = false;
    int max_block = 1024;
};

ClusterLimits cluster_limits(const simulation::EnsembleSpec &sp)
{
    ClusterLimits c;
    c.one_lane = sp.scheme == MP_SCHEME_IMPLICIT_MIDPOINT || sp.noise == MP_NOISE_ARRAY;
    if (sp.scheme == MP_SCHEME_IMPLICIT_MIDPOINT) c.max_block = mp::kImplicitClusterBlock;
    return c;
}

// Two lanes per particle pay while one lane per particle would leave fewer
// than this many waves per CU: the pair sums of a slot run in half the time
// and the extra waves hide the LDS latency of the pair loop.
constexpr int kSplitBelowWavesPerCU = 16;

// Lanes per slot forced by MAGPY_AMD_CLUSTER_LANES (1 or 2), else 0.
int env_cluster_lanes()
{
    const char *env = std::getenv("MAGPY_AMD_CLUSTER_LANES");
    if (env == nullptr) return 0;
    return std::atoi(env) == 2 ? 2 : 1;
}

// Untimed choice of the layout: MAGPY_AMD_CLUSTER_LANES and
// MAGPY_AMD_CLUSTER_BLOCK (lanes per workgroup) when set and valid, else two
// lanes per slot for ensembles of few waves, and the smallest block.
ClusterLayout cluster_layout(int64_t nmax, int64_t particles, ClusterLimits lim = {})
{
    ClusterLayout l;
    if (lim.one_lane) {
        l.lanes = 1;
    } else if (const int forced = env_cluster_lanes()) {
        l.lanes = forced;
    } else {
        const int cus = device_cus();
        l.lanes = particles < (int64_t)kSplitBelowWavesPerCU * mp::kWave * cus ? 2 : 1;
    }
    if (cluster_min_block(nmax, l.lanes, lim.max_block) == 0) l.lanes = 1;
    if (const char *env = std::getenv("MAGPY_AMD_CLUSTER_BLOCK")) {
        const int v = std::atoi(env);
        if (v / l.lanes >= nmax && v % mp::kWave == 0 && v <= lim.max_block) {
            l.block = v;
            return l;
        }
    }
    l.block = cluster_min_block(nmax, l.lanes, lim.max_block);
    return l;
}

// Autotuner of the cluster layout: for runs long enough to repay it, time a
// few trial steps of the launch set with the most particles with every candidate (one and
// two lanes per slot, unless MAGPY_AMD_CLUSTER_LANES fixes it, each with the
// power-of-two blocks from the smallest that holds the largest cluster up to
// 1024 lanes) on throw-away copies of the state, and keep the fastest.
// Results are cached (LayoutKey) for the life of the process.  Trials run
// from the run's own first step (a resumed run starts at start_step), and a
// run too short to time them keeps the untimed layout, uncached.
ClusterLayout autotune_cluster_layout(const simulation::EnsembleSpec &sp, const Plan &plan,
                                      const std::vector<int> &set, int64_t set_particles,
                                      int64_t nmax, hipStream_t s)
{
    static LayoutCache cache;
    const int forced = env_cluster_lanes();
    const LayoutKey key{sp.device, nmax, set_particles, (int)sp.precision, forced};
    ClusterLayout best;
    if (cache.find(key, best)) return best;
    const int64_t trial_steps = 64;
    const int64_t steps = plan.group_steps[(size_t)set[0]], first = std::min(sp.start_step, steps);
    if (steps - first < 4 + trial_steps) return cluster_layout(nmax, (int64_t)plan.perm.size());
    hipEvent_t e0, e1;
    MP_HIP(hipEventCreate(&e0));
    MP_HIP(hipEventCreate(&e1));
    float best_ms = 0.f;
    for (int lanes = 1; lanes <= 2; ++lanes) {
        if (forced != 0 && lanes != forced) continue;
        const int b0 = cluster_min_block(nmax, lanes);
        for (int b = b0; b != 0 && b <= 1024; b *= 2) {
            std::unique_ptr<GroupBase> g;
            if (sp.precision == MP_PRECISION_FP32)
                g.reset(new GroupRun<float>(sp, plan, set, false, false, b, lanes));
            else
                g.reset(new GroupRun<double>(sp, plan, set, false, false, b, lanes));
            g->enqueue(g->n_done + 4, s);  // warm the code object
            MP_HIP(hipEventRecord(e0, s));
            g->enqueue(g->n_done + trial_steps, s);
            MP_HIP(hipEventRecord(e1, s));
            MP_HIP(hipStreamSynchronize(s));
            float ms = 0.f;
            MP_HIP(hipEventElapsedTime(&ms, e0, e1));
            if (best.block == 0 || ms < best_ms) {
                best.block = b;
                best.lanes = lanes;
                best_ms = ms;
            }
        }
    }
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    cache.keep(key, best);
    return best;
}

// With an arena open on this thread (the no-allocation entry point), every
// device buffer of the session comes from it, launches go to the null
// stream, no stream or event is created and the layout is not autotuned.
mp_session *session_create(const simulation::EnsembleSpec &sp, bool traj, bool ens)
{
    const bool in_arena = current_arena() != nullptr;
    simulation::validate(sp);
    int ndev = 0;
    if (hipGetDeviceCount(&ndev) != hipSuccess || ndev == 0)
        throw simulation::Error(MP_ERR_NODEV, "no HIP device visible");
    require(sp.device >= 0 && sp.device < ndev, "device ordinal out of range");
    MP_HIP(hipSetDevice(sp.device));

    std::unique_ptr<mp_session> ss(new mp_session(!in_arena));
    ss->device = sp.device;
    ss->want_traj = traj;
    ss->want_ens = ens;
    Plan &plan = ss->plan;
    const int64_t P = sp.member_offsets[sp.n_members];
    HostCopy &h = ss->host;
    h.M = sp.n_members;
    h.P = P;
    h.S = sp.max_samples;
    const double *m_start = sp.start_state ? sp.start_state : sp.magnetisation_direction;
    h.m0.assign(m_start, m_start + 3 * P);
    h.start = sp.start_step;
    h.ms.assign(sp.magnetisation, sp.magnetisation + sp.n_members);
    h.shape.assign(sp.field_shape, sp.field_shape + sp.n_members);

    // reduce every member, schedule per member, group members by schedule.
    // Every kernel reads its lane's reduced time step, so members whose
    // integer schedules (sample steps and step count) are equal share one
    // launch even when their reduced steps differ (other damping or
    // anisotropy).  FP32 Heun keeps one group per reduced step: there a
    // group whose lanes all see one applied field reads it from a shared
    // table, whose bits differ from the per-lane evaluation, and a member's
    // result must not depend on the rest of the ensemble.
    const bool merge_by_schedule =
        !(sp.precision == MP_PRECISION_FP32 && sp.scheme == MP_SCHEME_HEUN);
    plan.red.reserve((size_t)sp.n_members);
    plan.member_of.resize((size_t)P);
    std::map<std::pair<double, double>, int> step_key;        // (dt, end) -> schedule
    std::vector<std::vector<int64_t>> scheds;                 // schedule + step count
    std::map<std::vector<int64_t>, int> sched_to_group;
    std::vector<int> &member_group = plan.group_of;
    std::vector<int> group_sched;
    member_group.resize((size_t)sp.n_members);
    for (int64_t m = 0; m < sp.n_members; ++m) {
        const int64_t b = sp.member_offsets[m], e = sp.member_offsets[m + 1];
        plan.red.push_back(simulation::reduce_member(
            sp.radius + b, sp.anisotropy + b, (size_t)(e - b), sp.magnetisation[m], sp.damping[m],
            sp.temperature[m], sp.time_step, sp.end_time, sp.field_amplitude[m],
            sp.field_frequency[m]));
        for (int64_t p = b; p < e; ++p) plan.member_of[(size_t)p] = m;
        const auto key = std::make_pair(plan.red.back().dt, plan.red.back().end_time);
        auto it = step_key.find(key);
        if (it == step_key.end()) {
            std::vector<int64_t> k;
            const int64_t steps =
                simulation::sample_schedule(key.first, key.second, sp.max_samples, k);
            k.push_back(steps);
            it = step_key.emplace(key, (int)scheds.size()).first;
            scheds.push_back(std::move(k));
        }
        const int si = it->second;
        int g = -1;
        if (merge_by_schedule) {
            auto jt = sched_to_group.find(scheds[(size_t)si]);
            if (jt == sched_to_group.end())
                jt = sched_to_group.emplace(scheds[(size_t)si], (int)group_sched.size()).first;
            g = jt->second;
        } else {
            g = si;   // groups are the distinct (dt, end) pairs in order
        }
        if (g == (int)group_sched.size()) group_sched.push_back(si);
        member_group[(size_t)m] = g;
    }
    const int G = (int)group_sched.size();
    plan.group_begin.assign((size_t)G + 1, 0);
    std::vector<std::vector<int64_t>> group_members((size_t)G);
    for (int64_t m = 0; m < sp.n_members; ++m)
        group_members[(size_t)member_group[(size_t)m]].push_back(m);
    for (int g = 0; g < G; ++g) {
        for (int64_t m : group_members[(size_t)g])
            for (int64_t p = sp.member_offsets[m]; p < sp.member_offsets[m + 1]; ++p)
                plan.perm.push_back(p);
        plan.group_begin[(size_t)g + 1] = (int64_t)plan.perm.size();
        std::vector<int64_t> k = scheds[(size_t)group_sched[(size_t)g]];
        const int64_t steps = k.back();
        k.pop_back();
        plan.sched.push_back(std::move(k));
        plan.group_steps.push_back(steps);
    }
    if (sp.noise == MP_NOISE_ARRAY)
        for (int g = 0; g < G; ++g)
            require(plan.group_steps[(size_t)g] <= sp.noise_steps,
                    "Exceeded allocated random number array size (noise_steps < steps)");
    // interacting clusters: one block holds whole clusters, so the block must
    // be at least the largest cluster.  The implicit scheme couples a
    // cluster's particles through its Newton norms even without interactions
    // (one 3N system per cluster, lib/integrators.cpp:576-651), so it takes
    // the cluster path for any member of several particles.
    ClusterLayout layout;
    int64_t nmax = 1;
    if (sp.interactions || sp.scheme == MP_SCHEME_IMPLICIT_MIDPOINT) {
        for (int64_t m = 0; m < sp.n_members; ++m)
            nmax = std::max(nmax, sp.member_offsets[m + 1] - sp.member_offsets[m]);
        if (nmax > 1) {
            const ClusterLimits lim = cluster_limits(sp);
            layout = cluster_layout(nmax, (int64_t)plan.perm.size(), lim);
            if (layout.block == 0)
                throw simulation::Error(
                    MP_ERR_UNSUPPORTED,
                    sp.scheme == MP_SCHEME_IMPLICIT_MIDPOINT
                        ? "the implicit midpoint scheme supports clusters of at most " +
                              std::to_string(lim.max_block) + " particles"
                        : std::string("clusters of more than 1024 particles are not supported"));
        }
    }
    int cluster_block = layout.block;
    // replicas of one cluster: the dipolar field as one product per stage
    int gemm = 0;
    if (cluster_block != 0 && G == 1 && sp.scheme == MP_SCHEME_HEUN &&
        sp.noise == MP_NOISE_PHILOX && sp.precision == MP_PRECISION_FP32 &&
        sp.dipolar != MP_DIPOLAR_PAIRS && shared_geometry(sp)) {
        const int64_t n = sp.member_offsets[1] - sp.member_offsets[0];
        if (sp.dipolar == MP_DIPOLAR_GEMM_BF16X3 || sp.dipolar == MP_DIPOLAR_GEMM_F32)
            gemm = sp.dipolar;
        else if (sp.n_members >= 64 && n >= 32)
            gemm = MP_DIPOLAR_GEMM_BF16X3;
    }
    if (gemm != 0) {
        ss->cluster_block = 0;
        ss->dipolar = gemm;
        UploadScope uploads;
        ss->groups.emplace_back(new ReplicaRun(sp, plan, traj, ens, gemm));
        uploads.flush();
        return ss.release();
    }
    if (sp.dipolar == MP_DIPOLAR_GEMM_BF16X3 || sp.dipolar == MP_DIPOLAR_GEMM_F32)
        throw simulation::Error(MP_ERR_UNSUPPORTED,
                                "the dipolar product needs an FP32 Heun ensemble of replicas of "
                                "one cluster with the Philox stream");
    const std::vector<std::vector<int>> sets = launch_sets(sp, plan, cluster_block != 0, in_arena);
    // pair sums: pick the block size by timing the candidates on long runs
    if (cluster_block != 0 && std::getenv("MAGPY_AMD_CLUSTER_BLOCK") == nullptr &&
        sp.noise == MP_NOISE_PHILOX && sp.scheme == MP_SCHEME_HEUN && !in_arena) {
        int64_t particles = 0;
        const std::vector<int> &timed = sets[largest_set(sets, plan.group_begin, &particles)];
        if (plan.group_steps[(size_t)timed[0]] >= 20000)
            layout = autotune_cluster_layout(sp, plan, timed, particles, nmax, ss->sg.s);
    }
    cluster_block = layout.block;
    ss->dipolar = cluster_block && sp.interactions ? MP_DIPOLAR_PAIRS : 0;
    ss->cluster_block = cluster_block;
    ss->cluster_lanes = cluster_block ? layout.lanes : 0;
    UploadScope uploads;
    for (const std::vector<int> &set : sets) {
        if (sp.precision == MP_PRECISION_FP32 && sp.scheme == MP_SCHEME_HEUN)
            ss->groups.emplace_back(
                new GroupRun<float>(sp, plan, set, traj, ens, cluster_block, layout.lanes,
                                    sets.size() == 1));
        else
            ss->groups.emplace_back(
                new GroupRun<double>(sp, plan, set, traj, ens, cluster_block, layout.lanes,
                                     sets.size() == 1));
    }
    uploads.flush();
    size_t record_bytes = 0;
    for (auto &g : ss->groups) record_bytes = std::max(record_bytes, g->record_bytes());
    ss->records.alloc(record_bytes);
    for (auto &g : ss->groups) g->use_records(ss->records.p);
    return ss.release();
}

void session_advance(mp_session *ss, int64_t n)
{
    MP_HIP(hipSetDevice(ss->device));
    if (ss->sg.e0 == nullptr) {
        // no events of its own: the host's clock around the synchronised block
        const auto t0 = std::chrono::steady_clock::now();
        for (auto &g : ss->groups) g->enqueue(g->n_done + n, ss->sg.s);
        MP_HIP(hipStreamSynchronize(ss->sg.s));
        ss->kernel_ms +=
            std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - t0)
                .count();
        return;
    }
    MP_HIP(hipEventRecord(ss->sg.e0, ss->sg.s));
    for (auto &g : ss->groups) g->enqueue(g->n_done + n, ss->sg.s);
    MP_HIP(hipEventRecord(ss->sg.e1, ss->sg.s));
    MP_HIP(hipStreamSynchronize(ss->sg.s));
    float ms = 0.f;
    MP_HIP(hipEventElapsedTime(&ms, ss->sg.e0, ss->sg.e1));
    ss->kernel_ms += ms;
}

void session_finish(mp_session *ss, mp_ensemble_out &out)
{
    int64_t remaining = 0;
    for (auto &g : ss->groups) remaining = std::max(remaining, g->n_total - g->n_done);
    if (remaining > 0) session_advance(ss, remaining);
    MP_HIP(hipSetDevice(ss->device));
    const HostCopy &h = ss->host;
    const Plan &plan = ss->plan;
    const int64_t S = h.S;
    const bool want_traj = ss->want_traj && (out.mx || out.my || out.mz);
    const SampleSink sink{{out.mx, out.my, out.mz}, plan, h};
    std::vector<double> ens;
    if (out.ens_m && ss->want_ens) ens.assign((size_t)S * 3, 0.0);
    int64_t newton_iters = 0, newton_fail = 0;
    for (auto &run : ss->groups) {
        const GroupOut o = run->collect(ss->sg.s, out.final_state, want_traj ? &sink : nullptr);
        const std::vector<int64_t> &slots = run->slots();
        if (out.status)
            for (size_t i = 0; i < slots.size(); ++i)
                if (slots[i] >= 0) out.status[slots[i]] = o.status[i];
        newton_iters += o.newton_iters;
        newton_fail += o.newton_fail;
        // samples recorded at the start step are the start state exactly as
        // given; samples before a resumed run's start step are not known
        const double nan = std::numeric_limits<double>::quiet_NaN();
        if (!ens.empty())
            for (int64_t s = 0; s < S; ++s) {
                // what the set's groups recorded of sample s, and the start states
                // of those that took it at the start step
                bool known = true, all = true;
                double v[3] = {0.0, 0.0, 0.0};
                for (int gi : run->set()) {
                    const int64_t k = plan.sched[(size_t)gi][(size_t)s];
                    known = known && k >= h.start;
                    all = all && k > h.start;
                }
                if (known && !all)
                    for (const int64_t p : slots) {
                        if (p < 0) continue;
                        const int64_t m = plan.member_of[(size_t)p];
                        if (plan.sched[(size_t)plan.group_of[(size_t)m]][(size_t)s] > h.start)
                            continue;
                        const double w = h.ms[(size_t)m];
                        for (int d = 0; d < 3; ++d) v[d] += h.m0[(size_t)p * 3 + d] * w;
                    }
                const bool recorded = all || run->set().size() > 1;
                for (int d = 0; d < 3; ++d)
                    ens[(size_t)s * 3 + d] +=
                        !known ? nan : v[d] + (recorded ? o.ens[(size_t)s * 3 + d] : 0.0);
            }
    }

    // ---- results in SI units (lib/simulation.cpp:610-621)
    auto fill_time_field = [&](int64_t m, double *time, double *field) {
        const simulation::ReducedMember &r = plan.red[(size_t)m];
        const double ts = S > 1 ? r.end_time / (double)(S - 1) : 0.0;
        for (int64_t s = 0; s < S; ++s) {
            const double tr = s == 0 ? 0.0 : (double)s * ts;
            if (time) time[s] = tr / r.time_factor;
            if (field)
                field[s] = applied_host(h.shape[(size_t)m], r.happ, r.fapp, tr) * r.anisotropy_field;
        }
    };
    fill_time_field(0, out.time, out.field);
    if (out.member_time || out.member_field)
        for (int64_t m = 0; m < h.M; ++m)
            fill_time_field(m, out.member_time ? out.member_time + m * S : nullptr,
                            out.member_field ? out.member_field + m * S : nullptr);
    if (out.ens_m && !ens.empty()) std::memcpy(out.ens_m, ens.data(), ens.size() * sizeof(double));
    out.n_steps = plan.group_steps[0];
    out.newton_iters = newton_iters;
    out.newton_failures = newton_fail;
    out.kernel_ms = ss->kernel_ms;
}

}  // namespace

namespace simulation {

void ensemble_run(const EnsembleSpec &sp, EnsembleResult &out)
{
    std::unique_ptr<mp_session> ss(
        session_create(sp, out.mx || out.my || out.mz, out.ens_m != nullptr));
    session_finish(ss.get(), out);
}

}  // namespace simulation

// ============================================ fixed scratch (no allocation)
// Device memory of mp_ensemble_run_noalloc: one array per GPU, placed when
// the library's code object loads on that GPU and held until the process
// ends.  Host code never uses the name `scratch` as an address (on the host
// it is only a stand-in for the symbol): the device address comes from
// hipGetSymbolAddress, once per device, with that device current.
constexpr size_t kScratchBytes = (size_t)64 << 20;
static __device__ __align__(256) unsigned char scratch[kScratchBytes];

namespace {

constexpr int kMaxDevices = 64;
std::mutex g_scratch_mutex;
void *g_scratch_ptr[kMaxDevices] = {};

// The calling thread's current device's copy of `scratch`.
void *scratch_on(int device)
{
    require(device >= 0 && device < kMaxDevices, "device ordinal out of range");
    std::lock_guard<std::mutex> lock(g_scratch_mutex);
    if (g_scratch_ptr[device] == nullptr) {
        void *ptr = nullptr;
        MP_HIP(hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch)));
        require(ptr != nullptr, "no device address for the scratch array");
        g_scratch_ptr[device] = ptr;
    }
    return g_scratch_ptr[device];
}

}  // namespace

// ====================================================================== C ABI
extern "C" {

int mp_ensemble_run(const mp_ensemble_spec *spec, mp_ensemble_out *out)
{
    return guarded([&] {
        if (!spec || !out) throw simulation::Error(MP_ERR_ARG, "spec and out are required");
        simulation::ensemble_run(*spec, *out);
    });
}

int mp_ensemble_run_noalloc(const mp_ensemble_spec *spec, mp_ensemble_out *out)
{
    return guarded([&] {
        if (!spec || !out) throw simulation::Error(MP_ERR_ARG, "spec and out are required");
        int ndev = 0;
        if (hipGetDeviceCount(&ndev) != hipSuccess || ndev == 0)
            throw simulation::Error(MP_ERR_NODEV, "no HIP device visible");
        require(spec->device >= 0 && spec->device < ndev, "device ordinal out of range");
        MP_HIP(hipSetDevice(spec->device));
        Arena arena;
        arena.base = static_cast<char *>(scratch_on(spec->device));
        arena.cap = kScratchBytes;
        arena.who = "mp_ensemble_run_noalloc";
        ArenaScope scope(&arena);
        simulation::ensemble_run(*spec, *out);
    });
}

int mp_full_dynamics(const double *radius, const double *anisotropy,
                     const double *anisotropy_axis, const double *magnetisation_direction,
                     const double *location, size_t n_particles, double magnetisation,
                     double damping, double temperature, int renorm, int interactions,
                     int use_implicit, double eps, double time_step, double end_time,
                     size_t max_samples, long seed, int field_shape, double field_amplitude,
                     double field_frequency, int precision, double *time, double *field,
                     double *mx, double *my, double *mz)
{
    int64_t offs[2] = {0, (int64_t)n_particles};
    int32_t shape = field_shape;
    int64_t sd = seed;
    mp_ensemble_spec sp{};
    sp.n_members = 1;
    sp.member_offsets = offs;
    sp.radius = radius;
    sp.anisotropy = anisotropy;
    sp.anisotropy_axis = anisotropy_axis;
    sp.magnetisation_direction = magnetisation_direction;
    sp.location = location;
    sp.magnetisation = &magnetisation;
    sp.damping = &damping;
    sp.temperature = &temperature;
    sp.field_shape = &shape;
    sp.field_amplitude = &field_amplitude;
    sp.field_frequency = &field_frequency;
    sp.seed = &sd;
    sp.time_step = time_step;
    sp.end_time = end_time;
    sp.max_samples = (int64_t)max_samples;
    sp.renorm = renorm;
    sp.interactions = interactions;
    sp.scheme = use_implicit ? MP_SCHEME_IMPLICIT_MIDPOINT : MP_SCHEME_HEUN;
    sp.precision = precision;
    sp.implicit_tol = eps;
    sp.implicit_max_iter = 1000;
    sp.noise = MP_NOISE_PHILOX;
    mp_ensemble_out o{};
    o.time = time;
    o.field = field;
    o.mx = mx;
    o.my = my;
    o.mz = mz;
    return mp_ensemble_run(&sp, &o);
}

int mp_session_create(const mp_ensemble_spec *spec, int want_trajectories, int want_ensemble,
                      mp_session **session)
{
    return guarded([&] {
        if (!spec || !session) throw simulation::Error(MP_ERR_ARG, "spec and session are required");
        *session = session_create(*spec, want_trajectories != 0, want_ensemble != 0);
    });
}

int mp_session_advance(mp_session *session, int64_t n_steps, int64_t *steps_done)
{
    return guarded([&] {
        if (!session || n_steps < 0) throw simulation::Error(MP_ERR_ARG, "bad session arguments");
        session_advance(session, n_steps);
        if (steps_done) *steps_done = session->groups[0]->n_done;
    });
}

int mp_session_info(mp_session *session, int64_t *n_steps_total, int64_t *launches,
                    double *kernel_ms, int32_t *cluster_block, int32_t *dipolar,
                    int32_t *cluster_lanes)
{
    return guarded([&] {
        if (!session) throw simulation::Error(MP_ERR_ARG, "session is required");
        int64_t tot = 0, l = 0;
        for (auto &g : session->groups) {
            tot = std::max(tot, g->n_total);
            l += g->launches;
        }
        if (n_steps_total) *n_steps_total = tot;
        if (launches) *launches = l;
        if (kernel_ms) *kernel_ms = session->kernel_ms;
        if (cluster_block) *cluster_block = session->cluster_block;
        if (dipolar) *dipolar = session->dipolar;
        if (cluster_lanes) *cluster_lanes = session->cluster_lanes;
    });
}

int mp_session_state(mp_session *session, double *state, int64_t *step)
{
    return guarded([&] {
        if (!session || !state) throw simulation::Error(MP_ERR_ARG, "session and state are required");
        MP_HIP(hipSetDevice(session->device));
        MP_HIP(hipStreamSynchronize(session->sg.s));
        for (auto &g : session->groups) g->state(state);
        if (step) *step = session->groups[0]->n_done;
    });
}

int mp_session_finish(mp_session *session, mp_ensemble_out *out)
{
    return guarded([&] {
        if (!session || !out) throw simulation::Error(MP_ERR_ARG, "session and out are required");
        session_finish(session, *out);
    });
}

void mp_session_destroy(mp_session *session) { delete session; }

int mp_sample_schedule(double dt_reduced, double end_reduced, int64_t max_samples, int64_t *k,
                       int64_t *n_steps)
{
    return guarded([&] {
        if (max_samples < 1 || !k || !n_steps || !(dt_reduced > 0))
            throw simulation::Error(MP_ERR_ARG, "invalid schedule arguments");
        std::vector<int64_t> v;
        *n_steps = simulation::sample_schedule(dt_reduced, end_reduced, max_samples, v);
        std::memcpy(k, v.data(), v.size() * sizeof(int64_t));
    });
}

int mp_dipolar_field(const double *location, const double *radius, const double *anisotropy,
                     size_t n_particles, double magnetisation, const double *m, size_t reps,
                     int mode, double *h, int device)
{
    return guarded([&] {
        if (!location || !radius || !anisotropy || !m || !h || n_particles == 0 || reps == 0 ||
            !(magnetisation > 0))
            throw simulation::Error(MP_ERR_ARG, "invalid dipolar field arguments");
        if (mode != MP_DIPOLAR_PAIRS && mode != MP_DIPOLAR_GEMM_BF16X3 && mode != MP_DIPOLAR_GEMM_F32)
            throw simulation::Error(MP_ERR_ARG, "unknown dipolar mode");
        int ndev = 0;
        if (hipGetDeviceCount(&ndev) != hipSuccess || ndev == 0)
            throw simulation::Error(MP_ERR_NODEV, "no HIP device visible");
        if (device < 0 || device >= ndev) throw simulation::Error(MP_ERR_ARG, "bad device");
        MP_HIP(hipSetDevice(device));
        const simulation::ReducedMember r = simulation::reduce_member(
            radius, anisotropy, n_particles, magnetisation, 0.1, 0.0, 1.0, 1.0, 0.0, 0.0);
        const int ld = replica_ld((int64_t)n_particles);
        const int rows = replica_rows((int64_t)reps);
        std::vector<double> D;
        dipole_tensor(r, location, magnetisation, n_particles, ld, D);
        std::vector<double> ma((size_t)rows * ld, 0.0);
        for (size_t rr = 0; rr < reps; ++rr)
            for (size_t p = 0; p < n_particles; ++p)
                for (int c = 0; c < 3; ++c)
                    ma[rr * ld + mp::replica_col((int)p, c)] = m[(rr * n_particles + p) * 3 + c];
        std::vector<double> out((size_t)rows * ld);
        if (mode == MP_DIPOLAR_PAIRS) {
            DevBuf<double> da, db, dc((size_t)rows * ld);
            da.upload(ma);
            db.upload(D);
            const int tot = rows * ld;
            hipLaunchKernelGGL(mp::gemm_f64_kernel, dim3((unsigned)((tot + 255) / 256)), dim3(256),
                               0, 0, da.p, db.p, dc.p, rows, ld, ld);
            MP_HIP(hipGetLastError());
            MP_HIP(hipMemcpy(out.data(), dc.p, out.size() * sizeof(double), hipMemcpyDeviceToHost));
        } else {
            std::vector<float> tiled((size_t)rows * ld);
            for (int rr = 0; rr < rows; ++rr)
                for (int c = 0; c < ld; ++c)
                    tiled[mp::replica_at(ld, rr, c)] = (float)ma[(size_t)rr * ld + c];
            DevBuf<float> a32, tensor, c32((size_t)rows * ld);
            a32.upload(tiled);
            tensor.upload(tensor_fragments(D, ld, mode));
            mp::ReplicaArgs a{};
            a.ld = ld;
            a.h = c32.p;
            launch_product(mode, 0, a32.p, tensor.p, a, rows, device_cus(), 0, 0.f, 0, 0, 0);
            MP_HIP(hipMemcpy(tiled.data(), c32.p, tiled.size() * sizeof(float), hipMemcpyDeviceToHost));
            for (int rr = 0; rr < rows; ++rr)
                for (int c = 0; c < ld; ++c)
                    out[(size_t)rr * ld + c] = (double)tiled[mp::replica_at(ld, rr, c)];
        }
        for (size_t rr = 0; rr < reps; ++rr)
            for (size_t p = 0; p < n_particles; ++p)
                for (int c = 0; c < 3; ++c)
                    h[(rr * n_particles + p) * 3 + c] = out[rr * ld + mp::replica_col((int)p, c)];
    });
}

int mp_wiener_normals(uint64_t seed, uint32_t particle, uint32_t tag, uint64_t j0, size_t n,
                      int precision, double *out, int device)
{
    return guarded([&] {
        if (!out) throw simulation::Error(MP_ERR_ARG, "out is required");
        if (n == 0) return;
        int ndev = 0;
        if (hipGetDeviceCount(&ndev) != hipSuccess || ndev == 0)
            throw simulation::Error(MP_ERR_NODEV, "no HIP device visible");
        if (device < 0 || device >= ndev) throw simulation::Error(MP_ERR_ARG, "bad device");
        MP_HIP(hipSetDevice(device));
        DevBuf<double> d(n);
        const unsigned grid = (unsigned)((n + 255) / 256);
        if (precision == MP_PRECISION_FP32)
            hipLaunchKernelGGL(mp::wiener_kernel<float>, dim3(grid), dim3(256), 0, 0,
                               (uint32_t)seed, (uint32_t)(seed >> 32), particle, tag, j0,
                               (int64_t)n, d.p);
        else
            hipLaunchKernelGGL(mp::wiener_kernel<double>, dim3(grid), dim3(256), 0, 0,
                               (uint32_t)seed, (uint32_t)(seed >> 32), particle, tag, j0,
                               (int64_t)n, d.p);
        MP_HIP(hipGetLastError());
        MP_HIP(hipMemcpy(out, d.p, n * sizeof(double), hipMemcpyDeviceToHost));
    });
}

void mp_constants(double *kb, double *mu0, double *gamma)
{
    if (kb) *kb = kKB;
    if (mu0) *mu0 = kMU0;
    if (gamma) *gamma = kGYROMAG;
}

int mp_save_results(const char *prefix, const double *mx, const double *my, const double *mz,
                    const double *field, const double *time, size_t n_samples)
{
    return guarded([&] {
        require(prefix && mx && my && mz && field && time, "prefix and all five arrays are required");
        const char *ext[5] = {".mx", ".my", ".mz", ".field", ".time"};
        const double *arr[5] = {mx, my, mz, field, time};
        for (int i = 0; i < 5; ++i) {
            const std::string name = std::string(prefix) + ext[i];
            FILE *f = std::fopen(name.c_str(), "wb");
            if (!f) throw simulation::Error(MP_ERR_ARG, "cannot open " + name + " for writing");
            const size_t w = n_samples ? std::fwrite(arr[i], sizeof(double), n_samples, f) : 0;
            const bool ok = std::fclose(f) == 0 && w == n_samples;
            if (!ok) throw simulation::Error(MP_ERR_ARG, "failed to write " + name);
        }
    });
}

const char *mp_last_error(void) { return last_error().c_str(); }

const char *mp_version(void) { return "magpy_amd 0.1 (abi 1, gfx950)"; }

int mp_device_info(int device, char *buf, size_t len)
{
    hipDeviceProp_t prop;
    hipError_t e = hipGetDeviceProperties(&prop, device);
    if (e != hipSuccess) {
        last_error() = hipGetErrorString(e);
        return MP_ERR_NODEV;
    }
    if (buf && len)
        std::snprintf(buf, len, "%s (%s), %d CUs, %d MHz, %.1f GiB", prop.name, prop.gcnArchName,
                      prop.multiProcessorCount, prop.clockRate / 1000,
                      (double)prop.totalGlobalMem / (1024.0 * 1024.0 * 1024.0));
    return MP_OK;
}

}  // extern "C"
