// krylov.h -- Krylov acceleration of the FP32 correction solves of the
// FP64 refinement: device state and per-point arithmetic shared by the
// single-system (msi9.hip) and the batched (batch.hip) kernels.
//
// A correction solve A c = -r0 runs MSI iterations.  Plain MSI takes each
// sweep result z = -(LU)^-1 r as it is, c += z, r += A z, and needs some
// hundred iterations on a large grid for ten decades.  Here z is the next
// direction of Orthomin (generalized conjugate residuals with a short
// window): q = A z is made orthogonal to the last `win` directions q_m,
//     q' = q - sum beta_m q_m,  z' = z - sum beta_m p_m,
//     beta_m = (q, q_m) / (q_m, q_m),
// and the step along it minimises the residual norm,
//     c += alpha z',  r += alpha q',  alpha = -(q', r) / (q', q').
// Same sweeps, same stopping rule; the pressure systems take five to seven
// times fewer of them for a 1e-10 drop (258x130: 411 -> 69, 515x259: 514 ->
// 71, 1026x514: 646 -> 100), and a window of 2 to 25 mostly needs the same
// number within a few; 4 leaves a margin for systems further from symmetry
// (upwind convection in a recirculating field, 130x66: 250 iterations with
// 4, 350 with 2, 550 plain).  Dot products are FP64 sums of products taken
// in FP64; vectors are FP32 like the sweeps.  Solve times: 1026x514 133.3 ->
// 21.4 ms, 515x259 52.4 -> 8.2 ms, 256 uneven systems 242.6 -> 43.1 ms; the
// solutions' errors against 64 bits 4.5e-9 -> 0.4e-9 and 6.2e-9 -> 2.7e-9.
//
// Where r is nearly orthogonal to the new q' (cosine below 0.1), r hardly
// changes and the next sweep of it would give the same direction again, the
// stagnation short windows are known for; the sweep then takes q' instead
// (Orthodir's choice), which extends the same Krylov space.  Most pressure
// systems never need it; one of ten (130x60, aspect 1e3, smooth right-hand
// side) stalls at 2e-3 and takes 275 iterations without it, 66 with one such
// step, and the recirculating one 325 and 250.
//
// win = 0 is the minimal-residual step along z alone; `plain` takes z as it
// is (beta = 0, alpha = 1: plain MSI with its residual carried along).
#pragma once

#include <hip/hip_runtime.h>

#include <math.h>

#include "m2d_internal.h"
#include "msi_stencil.h"
#include "skew.h"

namespace m2d {

constexpr int kKryWin = 4;             // directions kept
constexpr int kKrySums = 2 + kKryWin;  // (q,q), (q,r), (q,q_m)

// The recurrence's scalars of one system (device memory).
struct KrylovCoef {
    double nn[kKryWin + 1];  // (q', q') of the direction in each q slot
    float beta[kKryWin];
    float alpha;
    float turn;  // 0: the next sweep takes r; else turn * q'
};

// Vectors of one system, reference layout, n = nx * ny values each: p holds
// win slots, q win + 1 (the direction being made takes a slot of its own), r
// the residual.  The sweeps read a skewed copy of r, or of q'.
struct KrylovVec {
    float *p, *q, *r;
    KrylovCoef *c;
    long n;
    int win, plain;
};

// The slots at iteration `it` (iterations done in this solve): q slot of the
// new direction, of the m-th latest one (m = 1..kept), and p slots alike.
struct KrylovSlots {
    int it, win, kept;
    __device__ KrylovSlots(const KrylovVec &v, int iter)
        : it(iter), win(v.win), kept(v.plain ? 0 : (iter < v.win ? iter : v.win))
    {
    }
    __device__ int q(int m) const { return (it - m) % (win + 1); }
    __device__ int p(int m) const { return (it - m) % win; }
};

// q = A z at (i, j), z skewed; ra: A in the reference layout.
template <int ND>
__device__ __forceinline__ float krylov_apply(const float *ra, const float *z, const Skew &sk,
                                              int i, int j)
{
    const long N = (long)sk.nx * sk.ny;
    auto zv = [&](int ii, int jj, long) { return z[sk.template of_point_c<16>(ii, jj)]; };
    return ND == 5 ? residual_point5_f<float, float>(ra, N, zv, 0.f, i, j, sk.nx, sk.ny)
                   : residual_point_f<float, float>(ra, N, zv, 0.f, i, j, sk.nx, sk.ny);
}

// Adds the new direction's products at a point to the sums: s[0] (q,q), s[1]
// (q,r), s[1 + m] (q,q_m).
struct KrylovKept {
    float q[kKryWin];
    __device__ void load(const KrylovVec &v, const KrylovSlots &k, long e)
    {
#pragma unroll
        for (int m = 1; m <= kKryWin; ++m) q[m - 1] = m <= k.kept ? v.q[k.q(m) * v.n + e] : 0.f;
    }
    __device__ void dots(float qn, float r, double *s) const
    {
        s[0] += (double)qn * (double)qn;
        s[1] += (double)qn * (double)r;
#pragma unroll
        for (int m = 0; m < kKryWin; ++m) s[2 + m] += (double)qn * (double)q[m];
    }
};

// beta and alpha from the sums (one thread).  (q', q') = (q,q) - sum beta_m
// (q,q_m); where less than 1e-5 of (q,q) is left, the difference of FP32
// directions is mostly their rounding: the step is then taken along z alone.
// (q, r) needs no correction, r being orthogonal to every kept direction.
// rn: the residual norm before the step.
__device__ inline void krylov_coef(const KrylovVec &v, const KrylovSlots &k, const double *s,
                                   double rn)
{
    KrylovCoef &c = *v.c;
    double b[kKryWin], n2 = s[0];
#pragma unroll
    for (int m = 1; m <= kKryWin; ++m) {
        const double nm = m <= k.kept ? c.nn[k.q(m)] : 0.0;
        b[m - 1] = nm > 0.0 ? s[1 + m] / nm : 0.0;
        n2 -= b[m - 1] * s[1 + m];
    }
    if (!(n2 > 1e-5 * s[0])) {
        n2 = s[0];
        for (int m = 0; m < kKryWin; ++m) b[m] = 0.0;
    }
    c.nn[k.q(0)] = n2;
    for (int m = 0; m < kKryWin; ++m) c.beta[m] = (float)b[m];
    // q = 0: nothing to gain along z; not finite: let it show in r
    c.alpha = v.plain ? 1.f : (n2 == 0.0 ? 0.f : (float)(-s[1] / n2));
    const bool turn = !v.plain && v.win && n2 > 0.0 && s[1] * s[1] < 0.01 * n2 * (rn * rn);
    c.turn = turn ? (float)(rn / sqrt(n2)) : 0.f;
}

// The direction and the step at a point, in two parts so that the loads of
// several points can be in flight together: load, then finish, which writes
// the direction, c and r and returns the new residual; in gets the next
// sweep's input.
struct KrylovStep {
    float q, z, r, c, op[kKryWin], oq[kKryWin];
    __device__ void load(const KrylovVec &v, const KrylovSlots &k, long e, float z_,
                         const float *cv)
    {
        z = z_;
        r = v.r[e];
        c = cv[e];
        q = v.q[k.q(0) * v.n + e];
#pragma unroll
        for (int m = 1; m <= kKryWin; ++m) {
            const bool on = m <= k.kept;
            op[m - 1] = on ? v.p[k.p(m) * v.n + e] : 0.f;
            oq[m - 1] = on ? v.q[k.q(m) * v.n + e] : 0.f;
        }
    }
    __device__ float finish(const KrylovVec &v, const KrylovSlots &k, const KrylovCoef &f, long e,
                            float *cv, float &in)
    {
#pragma unroll
        for (int m = 0; m < kKryWin; ++m) {
            z = fmaf(-f.beta[m], op[m], z);
            q = fmaf(-f.beta[m], oq[m], q);
        }
        if (k.win && !v.plain) {
            v.p[k.p(0) * v.n + e] = z;
            v.q[k.q(0) * v.n + e] = q;
        }
        cv[e] = fmaf(f.alpha, z, c);
        r = fmaf(f.alpha, q, r);
        v.r[e] = r;
        in = f.turn != 0.f ? f.turn * q : r;
        return r;
    }
};

// Sums of K values over a workgroup of 256 threads, in a fixed order; the
// result is valid in thread 0.
template <int K>
__device__ __forceinline__ void block_sums(double (&s)[K])
{
    __shared__ double red[K][4];
#pragma unroll
    for (int k = 0; k < K; ++k) {
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) s[k] += __shfl_down(s[k], o, 64);
        if ((threadIdx.x & 63u) == 0) red[k][threadIdx.x >> 6] = s[k];
    }
    __syncthreads();
    if (threadIdx.x == 0)
#pragma unroll
        for (int k = 0; k < K; ++k) s[k] = ((red[k][0] + red[k][1]) + red[k][2]) + red[k][3];
}

// Which kind of step the next correction solve takes.  A solve's rate is its
// residual drop per iteration; the accelerated steps are kept while theirs
// is below 0.9 (ten decades in 220 iterations), else plain ones are tried
// once and from then on the kind with the better last rate runs: no system
// plain MSI converges on is left with steps that stagnate.
struct KrylovChoice {
    double rate[2] = {0.0, 0.0};  // [accelerated, plain], 0: not run yet
    int plain = 0;
    void after(double before, double now, int its)
    {
        if (its < 1 || !(before > 0.0)) return;
        const double d = pow(now / before, 1.0 / its);
        rate[plain] = d > 0.0 ? d : (d == 0.0 ? 1e-300 : 1e300);
        if (!plain && rate[0] <= 0.9) return;
        plain = rate[1] == 0.0 ? 1 : (rate[1] < rate[0] ? 1 : 0);
    }
};

// The residual drop a correction solve is run to: inner_gamma, or ten times
// what the outer stopping rule still asks for where that is less of a drop.
// Ten times, because the steps lower the residual of the fast components as
// far as that of the slow ones, so that a solution that only just passes the
// rule can be as far off as a plain MSI one; it costs about 5 iterations.
inline double correction_drop(double inner_gamma, const SolveState &outer)
{
    const double need = outer.rn > 0.0 ? 0.1 * outer.gammarp / outer.rn : 0.0;
    return need > inner_gamma && need < 1.0 ? need : inner_gamma;
}

}  // namespace m2d
