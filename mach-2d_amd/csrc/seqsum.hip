// seqsum.hip -- sums that equal a sequential left-to-right loop bit for bit,
// computed in parallel.
//
// While the running sum s stays in one binade [2^e, 2^(e+1)), with u =
// 2^(e-52) its spacing, s = S u for a whole number S and adding a term t >= 0
// rounds S + t/u to the nearest whole number, ties to even.  So a term adds
// q = rint(t/u), whatever S is, unless the fraction of t/u is exactly one
// half: then S + floor(t/u) is rounded to even, which depends on S's parity
// alone.  A run of terms is therefore a map from S's parity to the whole
// number it adds; maps of neighbouring runs compose associatively, and all
// their numbers are exact in FP64 while the result stays below 2^53, i.e. in
// the binade.  (A map whose number reaches 2^53 only has to stay that large.)
// The additions that leave the binade, about log2 of the sum over the first
// term of them, are made as they are.
//
//   k_seq_part  (n > kSeqDirect) one wave per segment of kSeqSeg terms: its
//               sum in any order
//   k_seq_map   one wave per segment: the sum of the segments before it tells
//               the binade (up to the rounding, which the next kernel
//               checks), then the segment's map in it; where the sum moves
//               into the next binade inside the segment, the term that takes
//               it there and a map on either side
//   k_seq_final one workgroup per sum.  The first segment, whose first terms
//               move the sum through most of its binades, one by one
//               (seq_add_chunk); then 64 maps at a time by a scan over the
//               lanes as far as they stay in the binade; the two maps and the
//               term of a segment that leaves it; and a segment whose binade
//               was guessed wrong from its terms by the same scan
//
// From the first segment with a negative or non-finite term on, the rest is
// added one by one (seq_sum): the reference's sums are of absolute values, of
// ratios of them and of a pressure, so that path is for other callers' data.
//
// What bounds it: the sequential chain took 4.2 ns (10 cycles) per term, 2.2
// ms for the 524288 terms of a 1026x514 grid; now the last kernel's chain of
// scans (about 900 cycles each) and the launches.  Measured on MI355X, the
// kernels of one sum: 524288 terms 2222 -> 28 us, 32768 terms 141 ->
// 16 us.  A sum that stays zero has no binade, so its segments are taken from
// their terms one after the other, about 1 us each: 32768 zeros (the T
// system's neighbours in an Euler step) 141 -> 70 us.
#include <hip/hip_runtime.h>

#include "m2d_internal.h"
#include "seqsum.h"

namespace m2d {

namespace {

constexpr int kSeqLaneTerms = 8;     // terms per lane of the scans over terms
constexpr int kSeqGroup = 64 * kSeqLaneTerms;
constexpr double kTwo53 = 9007199254740992.0;

struct Seg {
    double part;        // sum, any order
    double inc0, inc1;  // the map: what an even / odd S gains in the binade e
    double term;        // kTwo: the term that moves the sum into e + 1 ...
    double jnc0, jnc1;  // ... and the map of the terms after it there
    int e;
    int kind;
};
enum { kTerms = 0, kOne = 1, kTwo = 2 };  // from its terms; one map; two
static_assert(kSeqGroup == kSeqSeg && kSeqSeg == kSeqChunk, "a segment is one scan");
static_assert(sizeof(Seg) == 8 * kSeqSegDoubles, "seq_scratch counts it");
constexpr int kNoBinade = 1 << 20;

// exponent of a positive v in [2^-960, inf), where 2^(52 - e) is a normal
// number too; kNoBinade for the others
__device__ __forceinline__ int binade(double v)
{
    const int b = (int)((unsigned long long)__double_as_longlong(v) >> 52);  // sign 0
    return b >= 63 && b <= 2046 ? b - 1023 : kNoBinade;
}
__device__ __forceinline__ double two_to(int k)  // -1022 <= k <= 1023
{
    return __longlong_as_double((long long)(k + 1023) << 52);
}
__device__ __forceinline__ bool odd(double whole)
{
    const double h = whole * 0.5;
    return h != floor(h);
}
// negative (also -0.0) or not finite
__device__ __forceinline__ bool bad_term(double t)
{
    return (unsigned)(__double_as_longlong(t) >> 32) >= 0x7ff00000u;
}

// What V terms (t >= 0, finite) in order gain in the binade e without ties;
// tie: one of them is exactly half way between two sums.
template <int V>
__device__ __forceinline__ double gain_of(const double (&t)[V], int e, bool &tie)
{
    const double sc = two_to(52 - e);
    double i0 = 0.0;
    tie = false;
#pragma unroll
    for (int v = 0; v < V; ++v) {
        const double x = t[v] * sc, q = rint(x);
        tie = tie || fabs(x - q) == 0.5;
        i0 += q;
    }
    return i0;
}

// The map (i0, i1) of V terms with ties among them.
template <int V>
__device__ __forceinline__ void map_of(const double (&t)[V], int e, double &i0, double &i1)
{
    const double sc = two_to(52 - e);
    i0 = i1 = 0.0;
#pragma unroll
    for (int v = 0; v < V; ++v) {
        const double x = fmin(t[v] * sc, kTwo53), f = floor(x);
        if (x - f != 0.5) {
            const double q = rint(x);
            i0 += q;
            i1 += q;
        } else {
            const double a = i0 + f, b = i1 + f;
            i0 = odd(a) ? a + 1.0 : a;  // S even: S + a rounded to even
            i1 = odd(b) ? b : b + 1.0;  // S odd
        }
    }
}

// (a0, a1) = the map a, then the map b
__device__ __forceinline__ void map_then(double &a0, double &a1, double b0, double b1)
{
    a0 += odd(a0) ? b1 : b0;
    a1 += odd(a1) ? b0 : b1;
}

template <int CTRL, int ROWS>
__device__ __forceinline__ double dpp_or_zero(double v)
{
    const long long b = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_update_dpp(0, (int)b, CTRL, ROWS, 0xf, false);
    const int hi = __builtin_amdgcn_update_dpp(0, (int)(b >> 32), CTRL, ROWS, 0xf, false);
    return __longlong_as_double((long long)(((unsigned long long)(unsigned)hi << 32) |
                                            (unsigned)lo));
}

// inclusive sum over the lanes (lanes outside the masked rows add zero)
__device__ __forceinline__ double lane_scan(double v)
{
    v += dpp_or_zero<0x111, 0xf>(v);  // row_shr:1
    v += dpp_or_zero<0x112, 0xf>(v);  // row_shr:2
    v += dpp_or_zero<0x114, 0xf>(v);  // row_shr:4
    v += dpp_or_zero<0x118, 0xf>(v);  // row_shr:8
    v += dpp_or_zero<0x142, 0xa>(v);  // row_bcast:15 into rows 1 and 3
    v += dpp_or_zero<0x143, 0xc>(v);  // row_bcast:31 into rows 2 and 3
    return v;
}

__device__ __forceinline__ double lane_value(double v, int lane)
{
    const long long b = __double_as_longlong(v);
    const unsigned lo = (unsigned)__builtin_amdgcn_readlane((int)b, lane);
    const unsigned hi = (unsigned)__builtin_amdgcn_readlane((int)(b >> 32), lane);
    return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}

// s (binade e) plus the lanes' maps in order, as far as the sum stays in the
// binade: returns the number of lanes taken
__device__ __forceinline__ int take_maps(double &s, int e, double i0, double i1)
{
    const double S = s * two_to(52 - e);
    double c;
    if (__ballot(i0 != i1) == 0) {
        c = lane_scan(i0);
    } else {
        const int lane = threadIdx.x & 63;
        for (int d = 1; d < 64; d <<= 1) {
            double a0 = __shfl_up(i0, d), a1 = __shfl_up(i1, d);
            map_then(a0, a1, i0, i1);
            if (lane >= d) {
                i0 = a0;
                i1 = a1;
            }
        }
        c = odd(S) ? i1 : i0;
    }
    // every addend is >= 0: the lanes below 2^53 are the first ones
    const unsigned long long over = __ballot(!(S + c < kTwo53));
    const int L = over ? __ffsll(over) - 1 : 64;
    if (L) s = (S + lane_value(c, L - 1)) * two_to(e - 52);
    return L;
}

// the V terms of one lane, added one by one
template <int V>
__device__ __forceinline__ void take_lane(double &s, const double (&t)[V], int lane)
{
#pragma unroll
    for (int v = 0; v < V; ++v) s = lane_value(t[v], lane) + s;
}

// s plus 64 V terms, lane l holding terms V l .. V l + V - 1, none bad
template <int V>
__device__ __forceinline__ void take_terms(double &s, const double (&t)[V])
{
    const int lane = threadIdx.x & 63;
    int from = 0;
    while (from < 64) {
        const int e = binade(s);
        int L = from;
        if (e != kNoBinade) {
            const bool on = lane >= from;
            bool tie;
            double i0 = gain_of(t, e, tie), i1;
            const unsigned long long ties = __ballot(on && tie);
            i0 = i1 = on ? i0 : 0.0;
            // one or two lanes with ties: the scan stops there and the lane
            // is added as it is; with more the maps are cheaper
            if (__popcll(ties) > 2) {
                if (on && tie) map_of(t, e, i0, i1);
            } else if (on && tie) {
                i0 = i1 = kTwo53;
            }
            L = take_maps(s, e, i0, i1);
        } else if (s == 0.0) {  // zeros leave it zero
            bool z = true;
#pragma unroll
            for (int v = 0; v < V; ++v) z = z && t[v] == 0.0;
            const unsigned long long nz = __ballot(!z && lane >= from);
            L = nz ? __ffsll(nz) - 1 : 64;
        }
        if (L < 64) take_lane(s, t, L);
        from = L + 1;
    }
}

// s plus terms [0, m) of t, 512 at a time; at counts them.  False, with s and
// at where it stopped, at a group with a bad term.
__device__ __forceinline__ bool take_range(double &s, const double *__restrict__ t, long m,
                                           long &at)
{
    auto load = [&](long p, double(&v)[kSeqLaneTerms]) {
        const long b = p + (long)(threadIdx.x & 63) * kSeqLaneTerms;
#pragma unroll
        for (int k = 0; k < kSeqLaneTerms; ++k) v[k] = b + k < m ? t[b + k] : 0.0;
    };
    double v[kSeqLaneTerms], w[kSeqLaneTerms];
    load(0, v);
    for (long p = 0; p < m; p += kSeqGroup) {
        load(p + kSeqGroup, w);
        bool b = false;
#pragma unroll
        for (int k = 0; k < kSeqLaneTerms; ++k) b = b || bad_term(v[k]);
        if (__ballot(b)) return false;
        take_terms(s, v);
#pragma unroll
        for (int k = 0; k < kSeqLaneTerms; ++k) v[k] = w[k];
        at += kSeqGroup;
    }
    return true;
}

// the map of the terms of the wave's lanes in order, on every lane
template <int V>
__device__ __forceinline__ void wave_map(const double (&t)[V], int e, double &i0, double &i1)
{
    bool tie;
    i0 = i1 = gain_of(t, e, tie);
    if (tie) map_of(t, e, i0, i1);
    if (__ballot(tie) == 0) {
        i0 = i1 = lane_value(lane_scan(i0), 63);
    } else {
        for (int d = 1; d < 64; d <<= 1) {  // lane l: lanes l .. l + 2d - 1
            const double b0 = __shfl_down(i0, d), b1 = __shfl_down(i1, d);
            map_then(i0, i1, b0, b1);
        }
        i0 = lane_value(i0, 0);
        i1 = lane_value(i1, 0);
    }
    i0 = fmin(i0, kTwo53);
    i1 = fmin(i1, kTwo53);
}

constexpr int kSegWaves = 4;  // segments per workgroup
constexpr int kLaneTerms = kSeqSeg / 64;

__global__ __launch_bounds__(64 * kSegWaves) void k_seq_part(const double *__restrict__ t,
                                                             long n, Seg *__restrict__ segs,
                                                             int nseg)
{
    const int lane = threadIdx.x & 63, q = blockIdx.x * kSegWaves + (threadIdx.x >> 6);
    if (q >= nseg) return;
    t += (long)blockIdx.y * n;
    const long at = (long)q * kSeqSeg;
    double s = 0.0;
#pragma unroll
    for (int k = 0; k < kLaneTerms; ++k) {
        const long p = at + 64 * k + lane;
        s += p < n ? t[p] : 0.0;
    }
    s = lane_value(lane_scan(s), 63);
    if (lane == 0) segs[(long)blockIdx.y * nseg + q].part = s;
}

__global__ __launch_bounds__(64 * kSegWaves) void k_seq_map(const double *__restrict__ t, long n,
                                                            Seg *__restrict__ segs, int nseg)
{
    const int lane = threadIdx.x & 63, q = blockIdx.x * kSegWaves + (threadIdx.x >> 6);
    if (q >= nseg) return;
    t += (long)blockIdx.y * n;
    segs += (long)blockIdx.y * nseg;
    double v[kLaneTerms];
    const long at = (long)q * kSeqSeg + lane * kLaneTerms;
    bool bad = false;
#pragma unroll
    for (int k = 0; k < kLaneTerms; ++k) {
        v[k] = at + k < n ? t[at + k] : 0.0;
        bad = bad || bad_term(v[k]);
    }
    double before = 0.0;
#pragma unroll 8
    for (int k = lane; k < q; k += 64) before += segs[k].part;
    before = lane_value(lane_scan(before), 63);
    // the binades at both ends, with a margin for the rounding of both sums
    // (below n 2^-53)
    const int lo = binade(before * (1.0 - 1e-9));
    int hi = binade((before + segs[q].part) * (1.0 + 1e-9));
    Seg g = {segs[q].part, 0.0, 0.0, 0.0, 0.0, 0.0, lo, kTerms};
    if (__ballot(bad) == 0 && lo != kNoBinade && hi - lo <= 1) {
        if (hi > lo) {
            // the first term whose approximate sum reaches the next binade
            const double edge = two_to(hi);
            double sum = 0.0;
#pragma unroll
            for (int k = 0; k < kLaneTerms; ++k) sum += v[k];
            double run = before + (lane_scan(sum) - sum);
            int c = kLaneTerms;
#pragma unroll
            for (int k = 0; k < kLaneTerms; ++k) {
                run += v[k];
                if (run >= edge && c == kLaneTerms) c = k;
            }
            const unsigned long long over = __ballot(c < kLaneTerms);
            if (over) {
                const int L = __ffsll(over) - 1;
                double w[kLaneTerms], x = 0.0;
#pragma unroll
                for (int k = 0; k < kLaneTerms; ++k) {
                    const bool after = lane > L || (lane == L && k > c);
                    x = lane == L && k == c ? v[k] : x;
                    w[k] = after ? v[k] : 0.0;
                    v[k] = lane < L || (lane == L && k < c) ? v[k] : 0.0;
                }
                g.term = lane_value(x, L);
                wave_map(w, hi, g.jnc0, g.jnc1);
            } else {
                hi = lo;  // only the margin reaches it
            }
        }
        wave_map(v, lo, g.inc0, g.inc1);
        g.kind = hi > lo ? kTwo : kOne;
    }
    if (lane == 0) segs[q] = g;
}

// s (binade e) plus the map (i0, i1); false, s unchanged, where that leaves it
__device__ __forceinline__ bool take_map(double &s, int e, double i0, double i1)
{
    const double S = s * two_to(52 - e), R = S + (odd(S) ? i1 : i0);
    if (!(R < kTwo53)) return false;
    s = R * two_to(e - 52);
    return true;
}

// out[y] = the sum of t[y n .. y n + n) left to right, over n if mean.  Wave
// 0 walks; the whole workgroup first brings kStageSegs maps and the first
// segment's terms into LDS at once, so the walk does not wait for memory map
// by map.
constexpr int kFinalThreads = 256, kStageSegs = 1024;

__global__ __launch_bounds__(kFinalThreads) void k_seq_final(const double *__restrict__ t,
                                                             long n,
                                                             const Seg *__restrict__ segs,
                                                             int nseg, double *__restrict__ out,
                                                             int mean)
{
    __shared__ Seg maps[kStageSegs];
    __shared__ __align__(16) double terms[kSeqSlots * kSeqChunk];  // seq_sum's ring
    __shared__ int stopped;
    const int lane = threadIdx.x & 63;
    const bool walker = threadIdx.x < 64;
    t += (long)blockIdx.x * n;
    segs += (long)blockIdx.x * nseg;
    double s = 0.0;
    long at = 0;
    bool good = true;
    for (int k = threadIdx.x; k < kSeqSeg; k += kFinalThreads) terms[k] = k < n ? t[k] : 0.0;
    // without maps (nseg = 0) every later segment is taken from its terms
    const int nwalk = (int)((n + kSeqSeg - 1) / kSeqSeg);
    for (int c0 = 0; c0 < nwalk; c0 += kStageSegs) {
        const int mc = nwalk - c0 < kStageSegs ? nwalk - c0 : kStageSegs;
        __syncthreads();
        for (int k = threadIdx.x; k < mc; k += kFinalThreads) {
            if (nseg)
                maps[k] = segs[c0 + k];
            else
                maps[k].kind = kTerms;
        }
        __syncthreads();
        if (walker) {
            // 0 + t is t and t + 0 is t (a sum of zeros stays +0), so the
            // zeros past a short array change nothing
            if (c0 == 0) s = seq_add_chunk(terms, 0.0);
            for (int q0 = 0; q0 < mc && good; q0 += 64) {
                const int q = q0 + lane, m = mc - q0 < 64 ? mc - q0 : 64;
                const int eq = q < mc && maps[q].kind == kOne ? maps[q].e : kNoBinade;
                const double g0 = q < mc ? maps[q].inc0 : 0.0, g1 = q < mc ? maps[q].inc1 : 0.0;
                int from = c0 + q0 == 0 ? 1 : 0;
                while (from < m && good) {
                    const int e = binade(s);
                    int L = from;
                    if (e != kNoBinade)
                        L = take_maps(s, e, lane < from ? 0.0 : eq == e ? g0 : kTwo53,
                                      lane < from ? 0.0 : eq == e ? g1 : kTwo53);
                    if (L < m) {
                        const Seg &g = maps[q0 + L];
                        const int e1 = binade(s);
                        double r = s;
                        bool taken = g.kind == kTwo && g.e == e1 && take_map(r, e1, g.inc0, g.inc1);
                        if (taken) {
                            r = g.term + r;
                            taken = binade(r) == e1 + 1 && take_map(r, e1 + 1, g.jnc0, g.jnc1);
                        }
                        if (taken) {
                            s = r;
                        } else {
                            at = (long)(c0 + q0 + L) * kSeqSeg;
                            good = take_range(s, t + at, n - at < kSeqSeg ? n - at : kSeqSeg, at);
                        }
                    }
                    from = L + 1;
                }
            }
            if (lane == 0) stopped = !good;
        }
        __syncthreads();
        if (stopped) break;
    }
    if (!walker) return;
    if (!good) s = seq_sum(t + at, n - at, terms, s);
    if (lane == 0) out[blockIdx.x] = mean ? s / (double)n : s;
}

}  // namespace

void seq_sums_enqueue(const double *t, long n, int K, double *out, bool mean, double *scratch,
                      hipStream_t s)
{
    const int nseg = seq_segments(n);
    Seg *segs = (Seg *)scratch;
    if (nseg) {
        const dim3 g((unsigned)((nseg + kSegWaves - 1) / kSegWaves), (unsigned)K);
        hipLaunchKernelGGL(k_seq_part, g, dim3(64 * kSegWaves), 0, s, t, n, segs, nseg);
        hipLaunchKernelGGL(k_seq_map, g, dim3(64 * kSegWaves), 0, s, t, n, segs, nseg);
    }
    hipLaunchKernelGGL(k_seq_final, dim3(K), dim3(kFinalThreads), 0, s, t, n, segs, nseg, out,
                       mean ? 1 : 0);
}

}  // namespace m2d
