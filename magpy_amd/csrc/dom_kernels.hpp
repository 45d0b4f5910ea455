// dom_kernels.hpp -- discrete orientation model of independent particles.
//
// Each particle is a two-state system (up, down) whose probabilities obey
// the master equation dp/dt = W(h(t)) p with the Neel-Brown rates of
// dom::transition_matrix (lib/dom.cpp:30-56); the reference integrates it
// per particle with the adaptive Cash-Karp RK45 of integrator::rk45
// (lib/integrators.cpp:152-251) inside simulation::dom_ensemble_dynamics
// (lib/simulation.cpp:659-767), sampling mz = p_up - p_down by first-order
// hold.  Here one lane integrates one particle in FP64, all particles of an
// ensemble in one launch; samples are written [sample][particle].
//
// The reference loops until a step is accepted and until time passes each
// sample; a NaN error estimate or a vanishing step would spin forever.
// Each lane bounds both (kDomMaxRetries per step, max_steps per lane) and
// flags the particle instead, so every wave finishes.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace mp {

constexpr int kDomMaxRetries = 200;

struct DomArgs {
    int n;
    const double *k, *v, *temp, *ms, *alpha;   // per particle, SI
    const double *happ;                       // per particle: field amplitude / H_k
    const double *p_up, *p_down;              // initial probabilities
    int shape;                                // 0 sine, 1 square, 2 constant, 3 square Fourier
    double freq;
    int64_t n_components;
    double time_step, end_time;
    int64_t S;
    int64_t max_steps;
    double *mz;                               // [S][n]
    uint32_t *status;                         // bit 0: gave up (non-finite or no progress)
    int64_t *steps;                           // accepted steps per particle
    // Particles integrated by kDomLanes lanes each: the first wide_blocks
    // workgroups take kDomPerWave of them each, from wide_list[0 .. *wide_count),
    // or, without a list, all n particles.
    int wide_blocks;
    const int *wide_list, *wide_count;
    const int *wide;                          // 1: the particle is in the list
};

constexpr int kDomLanes = 16, kDomPerWave = 64 / kDomLanes;

__device__ inline double dom_field(const DomArgs &a, double h, double t)
{
#pragma clang fp contract(off)
    const double pi = 3.14159265358979323846;
    switch (a.shape) {
    case 0: return h * sin(2 * pi * a.freq * t);                       // lib/field.cpp:37-40
    case 1: return h * ((long long)(t * a.freq * 2) % 2 ? -1.0 : 1.0);  // lib/field.cpp:51-54
    case 3: {                                                          // lib/field.cpp:67-78
        double f = 0.0;
        for (int64_t k = 1; k < a.n_components + 1; ++k) {
            const double odd = (double)(2 * k - 1);
            f += sin(2 * pi * odd * a.freq * t) / odd;
        }
        return f * (4 / pi * h);
    }
    default: return h;
    }
}

// The particle's constants of dom::transition_matrix (lib/dom.cpp:30-56):
// sigma = K V / kT and the field-free part tau_N sqrt(pi) / sigma^1.5 of the
// prefactor, in the reference's order of operations.
struct DomParticle {
    double happ, sigma, c0;
};

__device__ inline DomParticle dom_particle(double k, double v, double temp, double ms, double al,
                                           double happ)
{
#pragma clang fp contract(off)
    const double kb = 1.38064852e-23, gamma = 1.76086e11, pi = 3.14159265358979323846;
    const double sigma = k * v / kb / temp;
    const double taun = v * ms * (1 + al * al) / 2.0 / gamma / al / kb / temp;
    return DomParticle{happ, sigma, taun * sqrt(pi) / pow(sigma, 1.5)};
}

// The rates in the field h: W = [[-r2, r1], [r2, -r1]], pre = c0 / (1 - h^2)
// (the reference's taun sqrt(pi) / pow(sigma, 1.5) / (1 - h h), left to
// right).  They depend on t (through the field) and the particle, not on the
// probabilities.  dom_rate forms r1 from w = 1 - h or r2 from w = 1 + h.
__device__ inline double dom_rate(const DomParticle &q, double h, double w)
{
#pragma clang fp contract(off)
    const double pre = q.c0 / (1 - h * h);
    return 1.0 / pre * w * exp(-(q.sigma * w * w));
}

__device__ inline void dom_rates(const DomArgs &a, const DomParticle &q, double t, double &r1,
                                 double &r2)
{
#pragma clang fp contract(off)
    const double h = dom_field(a, q.happ, t);
    r1 = dom_rate(q, h, 1 - h);
    r2 = dom_rate(q, h, 1 + h);
}

// dp = W p
__device__ inline void dom_apply(double r1, double r2, const double *p, double *dp)
{
#pragma clang fp contract(off)
    dp[0] = -r2 * p[0] + r1 * p[1];
    dp[1] = r2 * p[0] + -r1 * p[1];
}

// integrator::rk45 (lib/integrators.cpp:152-251) with the Cash-Karp tableau
// of include/integrators.hpp:128-160; returns false if no step was accepted
// within kDomMaxRetries attempts.  The rates of an attempt's six stage times
// are formed before its stages (they do not depend on the stage values), so
// their FP64 sin/exp evaluations can overlap instead of alternating with
// the stage arithmetic; (r1t, r2t) are the rates at t, which do not change
// between attempts and on return hold the rates at the new t (the accepted
// attempt's fifth stage time, t + h * 1.0 = t + h).  The same values, in
// the same expressions, as evaluating each stage's rates in turn.
__device__ inline bool dom_rk45(const DomArgs &a, const DomParticle &q, double *next,
                                const double *x, double *h_ptr, double *t_ptr, double tol,
                                double &r1t, double &r2t)
{
#pragma clang fp contract(off)
    double k1[2], k2[2], k3[2], k4[2], k5[2], k6[2], y[2], x5[2];
    double h = *h_ptr, t = *t_ptr, err = 0.0;
    double r1[5], r2[5];     // stages 2..6
    bool ok = false;
    dom_apply(r1t, r2t, x, k1);
    for (int attempt = 0; attempt < kDomMaxRetries && !ok; ++attempt) {
        const double ts[5] = {t + h * 0.2, t + h * 0.3, t + h * 0.6, t + h * 1.0,
                              t + h * (7.0 / 8.0)};
#pragma unroll
        for (int st = 0; st < 5; ++st) dom_rates(a, q, ts[st], r1[st], r2[st]);
        for (int i = 0; i < 2; ++i) y[i] = k1[i] * h * 0.2 + x[i];
        dom_apply(r1[0], r2[0], y, k2);
        for (int i = 0; i < 2; ++i) y[i] = x[i] + h * (3.0 / 40.0 * k1[i] + 9.0 / 40.0 * k2[i]);
        dom_apply(r1[1], r2[1], y, k3);
        for (int i = 0; i < 2; ++i)
            y[i] = x[i] + h * (3.0 / 10.0 * k1[i] + -9.0 / 10.0 * k2[i] + 6.0 / 5.0 * k3[i]);
        dom_apply(r1[2], r2[2], y, k4);
        for (int i = 0; i < 2; ++i)
            y[i] = x[i] + h * (-11.0 / 54.0 * k1[i] + 2.5 * k2[i] + -70.0 / 27.0 * k3[i] +
                               35.0 / 27.0 * k4[i]);
        dom_apply(r1[3], r2[3], y, k5);
        for (int i = 0; i < 2; ++i)
            y[i] = x[i] + h * (1631.0 / 55296.0 * k1[i] + 175.0 / 512.0 * k2[i] +
                               575.0 / 13824.0 * k3[i] + 44275.0 / 110592.0 * k4[i] +
                               253.0 / 4096.0 * k5[i]);
        dom_apply(r1[4], r2[4], y, k6);
        for (int i = 0; i < 2; ++i)
            x5[i] = x[i] + h * (37.0 / 378.0 * k1[i] + 250.0 / 621.0 * k3[i] +
                                125.0 / 594.0 * k4[i] + 512.0 / 1771.0 * k6[i]);
        for (int i = 0; i < 2; ++i)
            next[i] = x[i] + h * (2825.0 / 27648.0 * k1[i] + 18575.0 / 48384.0 * k3[i] +
                                  13525.0 / 55296.0 * k4[i] + 277.0 / 14336.0 * k5[i] +
                                  0.25 * k6[i]);
        // the reference's pow(., 2) and pow(., 0.5) of these norms as a square
        // and a square root: x * x is pow(x, 2) exactly, and sqrt, correctly
        // rounded, is what an accurate pow(x, 0.5) returns; a general FP64
        // pow is a long dependent chain, and these were five of the six per
        // attempt
        const double mag = sqrt(x[0] * x[0] + x[1] * x[1]);
        const double d0 = fabs(x5[0] - next[0]), d1 = fabs(x5[1] - next[1]);
        err = sqrt(d0 * d0 + d1 * d1);
        err /= (2.0 * tol * (1 + mag));
        if (err < 1.0) {
            ok = true;
        } else {
            double f = 0.84 * pow(err, -0.2);
            f = fabs(f) < 0.1 ? 0.1 : f;
            h *= f;
        }
    }
    if (!ok) return false;
    *t_ptr = t + h;
    r1t = r1[3];
    r2t = r2[3];
    double f = err == 0.0 ? 5.0 : 0.84 * pow(err, -0.2);
    f = f > 5 ? 5.0 : f;
    *h_ptr = f * h;
    return true;
}

// The value of lane ^ 1
__device__ inline double dom_swap(double v)
{
    return __hiloint2double(__builtin_amdgcn_mov_dpp(__double2hiint(v), 0xb1, 0xf, 0xf, true),
                            __builtin_amdgcn_mov_dpp(__double2loint(v), 0xb1, 0xf, 0xf, true));
}

// simulation::dom_ensemble_dynamics (lib/simulation.cpp:659-767) by dom_rk45,
// one lane per particle.
__device__ inline void dom_narrow(const DomArgs &a, int p)
{
#pragma clang fp contract(off)
    const double k = a.k[p], v = a.v[p], temp = a.temp[p], ms = a.ms[p], al = a.alpha[p];
    const double happ = a.happ[p];
    double next[2] = {a.p_up[p], a.p_down[p]}, last[2];
    a.mz[p] = next[0] - next[1];
    const double ts = a.end_time / (double)(a.S - 1);
    const double max_dt = a.end_time / 1000.0;
    double t = 0.0, t_last = 0.0, dt = 0.01 * a.time_step;
    const DomParticle q = dom_particle(k, v, temp, ms, al, happ);
    double r1t, r2t;     // rates at t
    dom_rates(a, q, t, r1t, r2t);
    int64_t steps = 0;
    bool alive = true;
    for (int64_t s = 1; s < a.S; ++s) {
        while (alive && t <= (double)s * ts) {
            last[0] = next[0];
            last[1] = next[1];
            t_last = t;
            if (++steps > a.max_steps ||
                !dom_rk45(a, q, next, last, &dt, &t, a.time_step, r1t, r2t)) {
                alive = false;
                break;
            }
            dt = dt > max_dt ? max_dt : dt;
        }
        double out;
        if (alive) {
            const double mz_last = last[0] - last[1], mz_next = next[0] - next[1];
            const double beta = (mz_next - mz_last) / (t - t_last);
            out = mz_last + beta * ((double)s * ts - t_last);
        } else {
            out = __builtin_nan("");
        }
        a.mz[(size_t)s * a.n + p] = out;
    }
    a.status[p] = alive ? 0u : 1u;
    a.steps[p] = steps;
}

// The same run by kDomLanes lanes: of an attempt's ten rates (five stage times,
// two directions) a lane forms one, and they meet in LDS (rates[2 s + u]); an
// even lane carries the up probability through the tableau, an odd lane the down
// one.  Every value is formed by dom_rk45's expressions, sums of two terms at
// most in the other order, so the bits are the same.  A lone wave issues one
// instruction every ~5.5 cycles, so a particle's time is its instructions: 2.7 ->
// 1.2 us per attempt; 65,536 particles, five field cycles, 11.8 -> 6.5 ms, the
// 3,767 steps of the fastest relaxing one bounding both.
__device__ inline void dom_wide(const DomArgs &a, int p, double *rates)
{
#pragma clang fp contract(off)
    const int l = threadIdx.x % kDomLanes, c = l & 1;
    const int job = l < 10 ? l : l - 10, stage = job >> 1;
    const bool up = (job & 1) == 0;   // r1
    const double when = stage == 0 ? 0.2 : stage == 1 ? 0.3 : stage == 2 ? 0.6 : stage == 3 ? 1.0
                                                                                       : 7.0 / 8.0;
    const DomParticle q = dom_particle(a.k[p], a.v[p], a.temp[p], a.ms[p], a.alpha[p], a.happ[p]);
    double next = c == 0 ? a.p_up[p] : a.p_down[p], last = next;
    double mz_next = next - dom_swap(next);   // (of the even lanes)
    if (l == 0) a.mz[p] = mz_next;
    const double ts = a.end_time / (double)(a.S - 1);
    const double max_dt = a.end_time / 1000.0, tol = a.time_step;
    double t = 0.0, t_last = 0.0, dt = 0.01 * a.time_step;
    // rates out of and into this lane's state: c = 0: r2, r1; c = 1: r1, r2
    double out_t, in_t;
    {
        double r1, r2;
        dom_rates(a, q, t, r1, r2);
        out_t = c == 0 ? r2 : r1;
        in_t = c == 0 ? r1 : r2;
    }
    // dp = W p
    auto apply = [](double out, double in, double own) {
        return -out * own + in * dom_swap(own);
    };
    int64_t steps = 0;
    bool alive = true;
    for (int64_t s = 1; s < a.S; ++s) {
        while (alive && t <= (double)s * ts) {
            last = next;
            t_last = t;
            if (++steps > a.max_steps) {
                alive = false;
                break;
            }
            const double x = last;
            double h = dt, err = 0.0;
            bool ok = false;
            const double k1 = apply(out_t, in_t, x);
            const double x_other = dom_swap(x);
            const double mag = sqrt(x * x + x_other * x_other);
            double out4 = 0.0, in4 = 0.0;
            for (int attempt = 0; attempt < kDomMaxRetries && !ok; ++attempt) {
                const double f = dom_field(a, q.happ, t + h * when);
                rates[job] = dom_rate(q, f, up ? 1 - f : 1 + f);
                __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
                __builtin_amdgcn_wave_barrier();
                __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
                double ro[5], ri[5];
#pragma unroll
                for (int st = 0; st < 5; ++st) {
                    ro[st] = rates[2 * st + 1 - c];
                    ri[st] = rates[2 * st + c];
                }
                const double k2 = apply(ro[0], ri[0], k1 * h * 0.2 + x);
                const double k3 =
                    apply(ro[1], ri[1], x + h * (3.0 / 40.0 * k1 + 9.0 / 40.0 * k2));
                const double k4 = apply(
                    ro[2], ri[2], x + h * (3.0 / 10.0 * k1 + -9.0 / 10.0 * k2 + 6.0 / 5.0 * k3));
                const double k5 =
                    apply(ro[3], ri[3], x + h * (-11.0 / 54.0 * k1 + 2.5 * k2 + -70.0 / 27.0 * k3 +
                                                 35.0 / 27.0 * k4));
                const double k6 = apply(
                    ro[4], ri[4],
                    x + h * (1631.0 / 55296.0 * k1 + 175.0 / 512.0 * k2 + 575.0 / 13824.0 * k3 +
                             44275.0 / 110592.0 * k4 + 253.0 / 4096.0 * k5));
                const double x5 = x + h * (37.0 / 378.0 * k1 + 250.0 / 621.0 * k3 +
                                           125.0 / 594.0 * k4 + 512.0 / 1771.0 * k6);
                next = x + h * (2825.0 / 27648.0 * k1 + 18575.0 / 48384.0 * k3 +
                                13525.0 / 55296.0 * k4 + 277.0 / 14336.0 * k5 + 0.25 * k6);
                const double d = fabs(x5 - next), d_other = dom_swap(d);
                err = sqrt(d * d + d_other * d_other);
                err /= (2.0 * tol * (1 + mag));
                if (err < 1.0) {
                    ok = true;
                    out4 = ro[3];
                    in4 = ri[3];
                } else {
                    double g = 0.84 * pow(err, -0.2);
                    g = fabs(g) < 0.1 ? 0.1 : g;
                    h *= g;
                }
            }
            if (!ok) {
                alive = false;
                break;
            }
            t = t + h;
            out_t = out4;
            in_t = in4;
            double g = err == 0.0 ? 5.0 : 0.84 * pow(err, -0.2);
            g = g > 5 ? 5.0 : g;
            dt = g * h;
            dt = dt > max_dt ? max_dt : dt;
        }
        double out;
        if (alive) {
            const double mz_last = last - dom_swap(last);
            mz_next = next - dom_swap(next);
            const double beta = (mz_next - mz_last) / (t - t_last);
            out = mz_last + beta * ((double)s * ts - t_last);
        } else {
            out = __builtin_nan("");
        }
        if (l == 0) a.mz[(size_t)s * a.n + p] = out;
    }
    if (l == 0) {
        a.status[p] = alive ? 0u : 1u;
        a.steps[p] = steps;
    }
}

__global__ __launch_bounds__(64) void dom_kernel(DomArgs a)
{
    __shared__ double rates[kDomPerWave][10];
    if ((int)blockIdx.x < a.wide_blocks) {
        const int i = blockIdx.x * kDomPerWave + threadIdx.x / kDomLanes;
        if (i >= (a.wide_list != nullptr ? *a.wide_count : a.n)) return;
        dom_wide(a, a.wide_list != nullptr ? a.wide_list[i] : i, rates[threadIdx.x / kDomLanes]);
    } else {
        const int p = (blockIdx.x - a.wide_blocks) * 64 + threadIdx.x;
        if (p >= a.n || (a.wide != nullptr && a.wide[p] != 0)) return;
        dom_narrow(a, p);
    }
}

// Which particles are integrated wide: those of the largest relaxation rate.
// Most take the 1,000 steps that the step limit asks for, while error control
// gives the fastest relaxing up to four times as many (a particle's steps grow
// with its peak rate), and a launch lasts as long as its longest particle.
// dom_rank bins every particle by the larger of its rates in no field and in the
// peak field (four bins a factor of two), dom_pick takes the top bins that hold
// at most `most` particles together.
constexpr int kDomBins = 1024;

__device__ inline int dom_bin(float rate)
{
    return (int)((__float_as_uint(rate) & 0x7fffffffu) >> 21);   // exponent, two mantissa bits
}

static __global__ __launch_bounds__(256) void dom_rank(DomArgs a, int *bin, int *hist)
{
    const int p = blockIdx.x * 256 + threadIdx.x;
    if (p >= a.n) return;
    const DomParticle q = dom_particle(a.k[p], a.v[p], a.temp[p], a.ms[p], a.alpha[p], a.happ[p]);
    // a square wave's Fourier sum overshoots by a fifth
    const double h = a.shape == 3 ? 1.2 * fabs(q.happ) : fabs(q.happ);
    const double still = 2 * dom_rate(q, 0.0, 1.0);
    const double peak = fabs(dom_rate(q, h, 1 - h)) + fabs(dom_rate(q, h, 1 + h));
    const int b = dom_bin((float)fmax(still, peak));
    bin[p] = b;
    atomicAdd(hist + b, 1);
}

static __global__ __launch_bounds__(256) void dom_pick(const int *bin, const int *hist, int n,
                                                       int most, int *wide, int *list, int *count)
{
    // above[i]: particles in bins >= 4 i
    __shared__ int above[kDomBins / 4 + 1];
    __shared__ int first;
    const int i = threadIdx.x;
    int own = 0;
    for (int b = 0; b < 4; ++b) own += hist[4 * i + b];
    above[i] = own;
    if (i == 0) {
        above[kDomBins / 4] = 0;
        first = kDomBins;
    }
    __syncthreads();
    for (int d = 1; d < kDomBins / 4; d *= 2) {
        const int x = i + d < kDomBins / 4 ? above[i + d] : 0;
        __syncthreads();
        above[i] += x;
        __syncthreads();
    }
    // the lowest bin that, with those above it, holds at most `most`
    int sum = above[i + 1];
    for (int b = 3; b >= 0; --b) {
        sum += hist[4 * i + b];
        if (sum <= most) atomicMin(&first, 4 * i + b);
    }
    __syncthreads();
    const int p = blockIdx.x * 256 + i;
    if (p >= n) return;
    const bool w = bin[p] >= first;
    wide[p] = w ? 1 : 0;
    if (w) list[atomicAdd(count, 1)] = p;
}

}  // namespace mp
