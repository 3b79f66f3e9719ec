// tstep.hip -- the Scarborough time-step statistics of
// src/tstepper/mod_tstepper_scarborough.f90 on the GPU: the mean convergence
// coefficient of a 9- or 5-diagonal system (get_mean_cc_9d / _5d,
// :260-320), the first time step (tstepper_dt0_scarborough, :40-76) and the
// next one (tstepper_dt_scarborough, :80-123).
//
// The per-point coefficients (sum of |a_nb| over |a_P|, the sums left to
// right as the reference's SUM intrinsic adds them) are computed in parallel
// into a scratch array in the reference's loop order (i outer, j inner), whose
// sum is the left-to-right loop's bit for bit (seqsum.hip), so the mean is the
// reference's; tstepper_dt runs its four means in the same launches.  The
// minimum of dt0 does not depend on the order and is a parallel reduction.  Entries take host or device arrays (all of one kind); they
// return the value, so they synchronise.
#include <math.h>

#include <vector>

#include "m2d_internal.h"

using namespace m2d;

namespace {

constexpr int kT = 256;

// terms of interior points (i, j) (1-based) -> t[(i-2)*(ny-2) + (j-2)].  The
// diagonals are read along i and the terms written along j: a 64 x 16 tile
// goes through LDS, so both are whole cache lines (row width 65: no bank
// conflicts either way).  Grid row z: array z.
constexpr int kTi = 64, kTj = 16;
struct CcArrays {
    const double *a[4];
    int nd[4];
};
__global__ __launch_bounds__(kT) void k_cc_terms(CcArrays A, int nx, int ny,
                                                double *__restrict__ t)
{
    __shared__ double tile[kTj][kTi + 1];
    const double *__restrict__ a = A.a[blockIdx.z];
    const int nd = A.nd[blockIdx.z];
    t += (long)blockIdx.z * ((long)(nx - 2) * (ny - 2));
    const long N = (long)nx * ny;
    const int i0 = blockIdx.x * kTi + 2, j0 = blockIdx.y * kTj + 2;
    const int i = i0 + (threadIdx.x & (kTi - 1));
#pragma unroll
    for (int r = threadIdx.x / kTi; r < kTj; r += kT / kTi) {
        const int j = j0 + r;
        if (i > nx - 1 || j > ny - 1) continue;
        const long np = (long)nx * (j - 1) + i - 1;
        double s1, s2, ap;
        if (nd == 9) {
            s1 = fabs(a[np]) + fabs(a[N + np]) + fabs(a[2 * N + np]) + fabs(a[3 * N + np]);
            s2 = fabs(a[5 * N + np]) + fabs(a[6 * N + np]) + fabs(a[7 * N + np]) +
                 fabs(a[8 * N + np]);
            ap = fabs(a[4 * N + np]);
        } else {
            s1 = fabs(a[np]) + fabs(a[N + np]);
            s2 = fabs(a[3 * N + np]) + fabs(a[4 * N + np]);
            ap = fabs(a[2 * N + np]);
        }
        tile[r][threadIdx.x & (kTi - 1)] = (s1 + s2) / ap;
    }
    __syncthreads();
    const int j = j0 + (threadIdx.x & (kTj - 1));
    if (j > ny - 1) return;
    for (int c = threadIdx.x / kTj; c < kTi && i0 + c <= nx - 1; c += kT / kTj)
        t[(long)(i0 + c - 2) * (ny - 2) + (j - 2)] = tile[threadIdx.x & (kTj - 1)][c];
}

// per-block minimum of 1/sqrt(Jp (u^2 + v^2)) over interior points
__global__ __launch_bounds__(kT) void k_dt0_partial(const double *__restrict__ Jp,
                                                   const double *__restrict__ u,
                                                   const double *__restrict__ v, int nx, int ny,
                                                   double *__restrict__ part)
{
    const int i = blockIdx.x * kT + threadIdx.x + 2, j = blockIdx.y + 2;
    double m = 1.0e10;
    if (i <= nx - 1) {
        const long np = (long)nx * (j - 1) + i - 1;
        const double aux = 1.0 / sqrt(Jp[np] * (u[np] * u[np] + v[np] * v[np]));
        if (m > aux) m = aux;
    }
    __shared__ double red[kT];
    red[threadIdx.x] = m;
    __syncthreads();
    for (int o = kT / 2; o > 0; o >>= 1) {
        if ((int)threadIdx.x < o && red[threadIdx.x] > red[threadIdx.x + o])
            red[threadIdx.x] = red[threadIdx.x + o];
        __syncthreads();
    }
    if (threadIdx.x == 0) part[blockIdx.y * gridDim.x + blockIdx.x] = red[0];
}

__global__ __launch_bounds__(kT) void k_min(const double *__restrict__ part, long n,
                                           double *__restrict__ out)
{
    __shared__ double red[kT];
    double m = 1.0e10;
    for (long q = threadIdx.x; q < n; q += kT)
        if (m > part[q]) m = part[q];
    red[threadIdx.x] = m;
    __syncthreads();
    for (int o = kT / 2; o > 0; o >>= 1) {
        if ((int)threadIdx.x < o && red[threadIdx.x] > red[threadIdx.x + o])
            red[threadIdx.x] = red[threadIdx.x + o];
        __syncthreads();
    }
    if (threadIdx.x == 0) out[0] = red[0] * 0.25;
}

// device copies of host inputs (or the inputs themselves), plus scratch
struct Staged {
    std::vector<const double *> in;
    Scratch buf;
};

int stage(Staged &S, const std::vector<const double *> &ptrs, const std::vector<long> &lens,
          long scratch, double **scratch_out, hipStream_t s)
{
    bool dev = is_device_array(ptrs[0]);
    for (const double *p : ptrs)
        if (!p || is_device_array(p) != dev) return M2D_ERR_ARG;
    long tot = scratch;
    if (!dev)
        for (long n : lens) tot += n;
    double *const buf = S.buf.get((size_t)(tot > 0 ? tot : 1));
    if (!buf) return M2D_ERR_HIP;
    long off = 0;
    for (size_t k = 0; k < ptrs.size(); ++k) {
        if (dev) {
            S.in.push_back(ptrs[k]);
            continue;
        }
        if (hipMemcpyAsync(buf + off, ptrs[k], sizeof(double) * lens[k], hipMemcpyHostToDevice,
                           s) != hipSuccess)
            return M2D_ERR_HIP;
        S.in.push_back(buf + off);
        off += lens[k];
    }
    *scratch_out = buf + off;
    return M2D_OK;
}

// means of K <= 4 coefficient arrays (nd[k] diagonals each): the terms of all
// K into one scratch, then K concurrent in-order sums
int mean_cc(int nx, int ny, int K, const double *const *a, const int *nd, double *out)
{
    if (nx < 3 || ny < 3 || !out) return M2D_ERR_ARG;
    const hipStream_t s = assembly_stream_current();
    const long N = (long)nx * ny, n = (long)(nx - 2) * (ny - 2);
    std::vector<const double *> ptrs(a, a + K);
    std::vector<long> lens;
    for (int k = 0; k < K; ++k) lens.push_back(nd[k] * N);
    Staged S;
    double *t = nullptr;
    int rc = stage(S, ptrs, lens, K * n + seq_scratch(n, K), &t, s);
    if (rc) return rc;
    double *const res = Scratch::results();
    if (!res) return M2D_ERR_HIP;
    cc_terms_enqueue(nx, ny, K, S.in.data(), nd, t, s);
    seq_sums_enqueue(t, n, K, res, true, t + K * n, s);
    if (hipGetLastError() != hipSuccess || hipStreamSynchronize(s) != hipSuccess)
        return M2D_ERR_HIP;
    S.buf.done();
    for (int k = 0; k < K; ++k) out[k] = res[k];
    return M2D_OK;
}

}  // namespace

void m2d::cc_terms_enqueue(int nx, int ny, int K, const double *const *a, const int *nd,
                           double *t, hipStream_t s)
{
    CcArrays A;
    for (int k = 0; k < 4; ++k) {
        A.a[k] = a[k < K ? k : 0];
        A.nd[k] = nd[k < K ? k : 0];
    }
    const dim3 grid((unsigned)((nx - 2 + kTi - 1) / kTi), (unsigned)((ny - 2 + kTj - 1) / kTj),
                    (unsigned)K);
    hipLaunchKernelGGL(k_cc_terms, grid, dim3(kT), 0, s, A, nx, ny, t);
}

// tstepper_dt_scarborough's rule (mod_tstepper_scarborough.f90:80-123) on
// the four means: the largest against mincc and maxcc
double m2d::scarborough_dt(double dt, const double *cc, double h0, double mincc, double maxcc)
{
    double c = cc[0];
    for (int k = 1; k < 4; ++k)
        if (cc[k] > c) c = cc[k];
    double h;
    if (c < mincc)
        h = h0 * sqrt(1.0 - c / mincc);
    else if (maxcc < c)
        h = -h0 * sqrt(c / maxcc - 1.0);
    else
        h = 0.0;
    return dt * (1.0 + h);
}

// The scratch a host thread keeps between calls (m2d::Scratch).
namespace {
struct Kept {
    double *p = nullptr;
    size_t n = 0;
    int dev = -1;
    bool used = false;
    ~Kept()
    {
        if (p) (void)hipFree(p);
    }
};
thread_local Kept g_kept;
constexpr size_t kKeepDoubles = (size_t)64 << 17;  // 64 MiB
}  // namespace

double *m2d::Scratch::get(size_t n)
{
    Kept &k = g_kept;
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess) return nullptr;
    if (k.used || n > kKeepDoubles)
        return hipMalloc((void **)&p_, sizeof(double) * n) == hipSuccess ? p_ : nullptr;
    if (!k.p || k.n < n || k.dev != dev) {
        if (k.p) (void)hipFree(k.p);
        k.p = nullptr;
        k.n = 0;
        if (hipMalloc((void **)&k.p, sizeof(double) * n) != hipSuccess) {
            k.p = nullptr;
            return nullptr;
        }
        k.n = n;
        k.dev = dev;
    }
    k.used = kept_ = true;
    return p_ = k.p;
}

double *m2d::Scratch::results()
{
    struct Pinned {
        double *p = nullptr;
        ~Pinned()
        {
            if (p) (void)hipHostFree(p);
        }
    };
    thread_local Pinned r;
    if (!r.p && hipHostMalloc((void **)&r.p, sizeof(double) * kResults, hipHostMallocPortable) !=
                    hipSuccess)
        r.p = nullptr;
    return r.p;
}

m2d::Scratch::~Scratch()
{
    if (!p_) return;
    if (kept_) g_kept.used = false;
    if (kept_ && done_) return;
    (void)hipFree(p_);
    if (kept_) {
        g_kept.p = nullptr;
        g_kept.n = 0;
    }
}

void m2d_set_last_status_code(int status);

// get_mean_cc_9d (mod_tstepper_scarborough.f90:260-288)
extern "C" double m2d_get_mean_cc_9d(const int *nx, const int *ny, const double *a)
{
    double v = 0.0;
    const int nd = 9;
    const int rc = (!nx || !ny) ? M2D_ERR_ARG : mean_cc(*nx, *ny, 1, &a, &nd, &v);
    m2d_set_last_status_code(rc);
    return v;
}

// get_mean_cc_5d (:292-320)
extern "C" double m2d_get_mean_cc_5d(const int *nx, const int *ny, const double *a)
{
    double v = 0.0;
    const int nd = 5;
    const int rc = (!nx || !ny) ? M2D_ERR_ARG : mean_cc(*nx, *ny, 1, &a, &nd, &v);
    m2d_set_last_status_code(rc);
    return v;
}

// tstepper_dt0_scarborough (:40-76)
extern "C" double m2d_tstepper_dt0_scarborough(const int *nx_, const int *ny_, const double *Jp,
                                               const double *u, const double *v)
{
    double dt = 0.0;
    int rc = M2D_OK;
    if (!nx_ || !ny_ || *nx_ < 3 || *ny_ < 3 || !Jp || !u || !v) rc = M2D_ERR_ARG;
    if (!rc) {
        const int nx = *nx_, ny = *ny_;
        const long N = (long)nx * ny;
        const hipStream_t s = assembly_stream_current();
        const dim3 grid((unsigned)((nx - 2 + kT - 1) / kT), (unsigned)(ny - 2));
        const long np = (long)grid.x * grid.y;
        Staged S;
        double *part = nullptr;
        rc = stage(S, {Jp, u, v}, {N, N, N}, np + 1, &part, s);
        if (!rc) {
            hipLaunchKernelGGL(k_dt0_partial, grid, dim3(kT), 0, s, S.in[0], S.in[1], S.in[2],
                               nx, ny, part);
            hipLaunchKernelGGL(k_min, dim3(1), dim3(kT), 0, s, part, np, part + np);
            if (hipGetLastError() != hipSuccess ||
                hipMemcpyAsync(&dt, part + np, sizeof(double), hipMemcpyDeviceToHost, s) !=
                    hipSuccess ||
                hipStreamSynchronize(s) != hipSuccess)
                rc = M2D_ERR_HIP;
            else
                S.buf.done();
        }
    }
    m2d_set_last_status_code(rc);
    return dt;
}

// tstepper_dt_scarborough (:80-123); h0, mincc and maxcc are the module
// variables tstepper_scarborough_init reads from the parameter file.
extern "C" double m2d_tstepper_dt_scarborough(const int *nx, const int *ny, const double *dt,
                                              const double *au, const double *av,
                                              const double *at, const double *ap,
                                              const double *h0, const double *mincc,
                                              const double *maxcc)
{
    if (!nx || !ny || !dt || !h0 || !mincc || !maxcc) {
        m2d_set_last_status_code(M2D_ERR_ARG);
        return 0.0;
    }
    const double *a[4] = {au, av, at, ap};
    const int nd[4] = {9, 9, 9, 5};
    double cc[4] = {0.0, 0.0, 0.0, 0.0};
    const int rc = mean_cc(*nx, *ny, 4, a, nd, cc);
    m2d_set_last_status_code(rc);
    if (rc) return 0.0;
    return scarborough_dt(*dt, cc, *h0, *mincc, *maxcc);
}
