// vote.hip -- the common-lines voting synchronization matrix on the device:
// the consumer of cryo_clmatrix's clstack in the C1 ab-initio pipeline.
//
// Replaces S = cryo_syncmatrix_vote(clstack, n_theta)
// (abinitio/C1/sync2n/cryo_syncmatrix_vote.m:38-57, called from
// abinitio/C1/cryo_abinitio_C1_worker.m:160) without reference rotations.
// For every pair (k1, k2) with a common line:
//  * every third image k3 with lines to both gives a triangle; its angle
//    phi = acos((c3 - c1 c2) / (sin t1 sin t2)) in degrees, t1 = (l13-l12)2pi/L,
//    t2 = (l21-l23)2pi/L, t3 = (l32-l31)2pi/L, kept when
//    1 + 2c1c2c3 - (c1^2+c2^2+c3^2) > 1e-5            (cryo_voteIJ.m:40-63)
//  * the angles vote in a Gaussian histogram (sigma 3) on 60 points of
//    [0, 180]; the first peak wins; triangles within 6 degrees of it are kept
//    (cryo_voteIJ.m:90-107)
//  * each kept triangle gives a relative rotation (rotratio_eulerangle_vec.m);
//    their top-left 2x2 blocks are averaged into S's block (k1, k2) and its
//    transpose into (k2, k1) (cryo_syncmatrixIJ_vote.m:125-164).
// A pair without a common line, or without voted triangles, gets a zero
// block; the diagonal blocks are the identity.  cos_phi2 and c_alpha are
// clamped to [-1, 1] before acos.
//
// Persistent kernels, one wave per pair, 64 third images at a time, one
// triangle per lane.  peak_kernel adds their Gaussians to the 60 histogram
// points on the FP64 matrix cores and keeps the largest point; terms_kernel
// re-evaluates, term by term, the pairs whose two largest points are too close
// to call; rot_kernel selects and averages.  The cosines and sines of the
// integer line differences come from a table built with the formulas' own
// expression.  The work is FP64 arithmetic per triangle; memory is the
// clstack in two 16-bit orientations (row k1/k2 and column k1/k2 reads are
// contiguous), the per-pair peaks and S.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>

#include "clm_ctx.h"

namespace vote {

constexpr int NT = 60;  // histogram points (ntics)

// M[i*K + j] = clstack(i, j), MT[j*K + i] = clstack(i, j) (1-based lines, 0 = none)
__device__ inline void build(int k1, int K, const int* cl1, const int* cl2, unsigned short* M, unsigned short* MT) {
    const long long e0 = (long long)k1 * K - (long long)k1 * (k1 + 1) / 2;
    for (int j = threadIdx.x; j < K; j += blockDim.x) {
        if (j <= k1) {
            if (j == k1) {
                M[(size_t)k1 * K + k1] = 0;
                MT[(size_t)k1 * K + k1] = 0;
            }
            continue;
        }
        const long long e = e0 + (j - k1 - 1);
        const unsigned short a = (unsigned short)cl1[e], b = (unsigned short)cl2[e];
        M[(size_t)k1 * K + j] = a;   // clstack(k1, k2)
        M[(size_t)j * K + k1] = b;   // clstack(k2, k1)
        MT[(size_t)j * K + k1] = a;
        MT[(size_t)k1 * K + j] = b;
    }
}

// The 2 x 2 identity of image k on S's diagonal.
__device__ inline void diag(int k, int K, double* S) {
    const size_t n2 = 2 * (size_t)K;
    S[(2 * (size_t)k) * n2 + 2 * k] = 1.0;
    S[(2 * (size_t)k + 1) * n2 + 2 * k] = 0.0;
    S[(2 * (size_t)k) * n2 + 2 * k + 1] = 0.0;
    S[(2 * (size_t)k + 1) * n2 + 2 * k + 1] = 1.0;
}

__device__ inline double tick(int d) { return d == NT - 1 ? 180.0 : d * (180.0 / (NT - 1)); }

// Windows of the histogram points: cosines of the angles certainly (by 1e-4
// degree, far beyond the rounding of acos and cos) outside and inside 6
// degrees of point d; those between take the exact test.
struct Window {
    double o_hi, o_lo, i_hi, i_lo;
};

// Tables of one call.  cs[d + n_theta] = (cos, sin) of d * 2 * pi / n_theta
// for the integer line differences d in [-n_theta, n_theta]: the same
// expression, evaluated once, as the angle of a line difference in the
// triangle and rotation formulas (2 * pi * d / L rounds the same way, the
// factor 2 being exact).  ln[l] = (cos, sin) of (l - 1) * 2 * pi / n_theta - pi
// for the lines l <= n_theta: the rotation's third Euler angle, and minus its
// first.  win[d]: the windows.
__device__ inline void tables(int i, int n_theta, double2* cs, double2* ln, Window* win) {
    if (i <= 2 * n_theta) {
        const double d = (double)(i - n_theta);
        const double th = d * 2 * M_PI / (double)n_theta;
        cs[i] = make_double2(cos(th), sin(th));
    }
    if (i <= n_theta) {
        const double th = ((double)i - 1) * 2 * M_PI / (double)n_theta - M_PI;
        ln[i] = make_double2(cos(th), sin(th));
    }
    if (i < NT) {
        const double x = tick(i), w = 360.0 / NT, t = 1e-4;
        auto cosd = [](double v) { return cos(v * M_PI / 180); };
        Window q;
        q.o_hi = x - (w + t) > 0 ? cosd(x - (w + t)) : INFINITY;
        q.o_lo = x + (w + t) < 180 ? cosd(x + (w + t)) : -INFINITY;
        q.i_hi = x - (w - t) > 0 ? cosd(x - (w - t)) : INFINITY;
        q.i_lo = x + (w - t) < 180 ? cosd(x + (w - t)) : -INFINITY;
        win[i] = q;
    }
}

// What the votes need, in one launch: workgroups 0..K-1 build the clstack (and
// write the diagonal of S), the rest the tables.
__global__ __launch_bounds__(256) void setup_kernel(int K, int n_theta, const int* cl1, const int* cl2,
                                                    unsigned short* M, unsigned short* MT, double2* cs, double2* ln,
                                                    Window* win, double* S) {
    const int b = blockIdx.x;
    if (b >= K) return tables((b - K) * 256 + threadIdx.x, n_theta, cs, ln, win);
    if (threadIdx.x == 0) diag(b, K, S);
    build(b, K, cl1, cl2, M, MT);
}

// Entry of line difference d (clamped to the table, so that a malformed
// clstack reads in bounds).
__device__ inline double2 trig(const double2* cs, int nt, int d) {
    const int i = d + nt;
    return cs[i < 0 ? 0 : (i > 2 * nt ? 2 * nt : i)];
}

// Cosine of the angle of triangle (k1, k2, k3), clamped to [-1, 1]; NaN
// when k3 takes no part.
__device__ inline double vote_cos(const unsigned short* r1, const unsigned short* r2, const unsigned short* c1_,
                                  const unsigned short* c2_, int k1, int k3, int l12, int l21,
                                  const double2* cs, int nt) {
    const int l13 = r1[k3], l23 = r2[k3];
    if (k3 == k1 || l13 == 0 || l23 == 0) return NAN;
    const int l31 = c1_[k3], l32 = c2_[k3];
    // theta1 = (l13 - l12) 2pi/L, theta2 = (l21 - l23) 2pi/L, theta3 = (l32 - l31) 2pi/L
    const double2 t1 = trig(cs, nt, l13 - l12), t2 = trig(cs, nt, l21 - l23), t3 = trig(cs, nt, l32 - l31);
    const double c1 = t1.x, c2 = t2.x, c3 = t3.x;
    const double cond = 1 + 2 * c1 * c2 * c3 - (c1 * c1 + c2 * c2 + c3 * c3);
    if (!(cond > 1.0e-5)) return NAN;
    double cp = (c3 - c1 * c2) / (t1.y * t2.y);
    cp = cp > 1 ? 1 : (cp < -1 ? -1 : cp);
    return cp;
}

// Angle (degrees) of triangle (k1, k2, k3), NaN when k3 takes no part.
__device__ inline double vote_angle(const unsigned short* r1, const unsigned short* r2, const unsigned short* c1_,
                                    const unsigned short* c2_, int k1, int k3, int l12, int l21,
                                    const double2* cs, int nt) {
    const double cp = vote_cos(r1, r2, c1_, c2_, k1, k3, l12, l21, cs, nt);
    return isnan(cp) ? cp : acos(cp) * 180 / M_PI;
}

// The (cos, sin) table in LDS when it fits (dynamic LDS of the launch), the
// same values read from global memory otherwise.
__device__ inline const double2* stage_trig(const double2* cs, int nt, int use_lds) {
    extern __shared__ double2 s_cs[];
    if (!use_lds) return cs;
    for (int i = threadIdx.x; i <= 2 * nt; i += blockDim.x) s_cs[i] = cs[i];
    __syncthreads();
    return s_cs;
}

// Pair (k1, k2) of flat index e (k1 < k2, row-major over k1).
__device__ inline void pair_of(long long e, int K, int& k1, int& k2) {
    int a = (int)floor(((2.0 * K - 1.0) - sqrt((2.0 * K - 1.0) * (2.0 * K - 1.0) - 8.0 * (double)e)) / 2.0);
    if (a < 0) a = 0;
    auto first = [&](long long x) { return x * K - x * (x + 1) / 2; };
    while (a > 0 && first(a) > e) a--;
    while (first(a + 1) <= e) a++;
    k1 = a;
    k2 = (int)(e - first(a)) + a + 1;
}

// t / 18 correctly rounded, without the general division sequence.  Let
// q = t/18 lie in [2^e, 2^(e+1)) and u = 2^(e-52) (its ulp).  R = RN(1/18)
// has |R - 1/18| <= 2^-58, so q0 = RN(t R) is within 1.6 u of q; the
// remainder r = t - 18 q0 is a multiple of u (t is a multiple of 16 u, 18 q0
// of 9 u) below 29 u in magnitude, so the FMA computes it exactly; and
// q0 + r R, rounded once by the second FMA, differs from q by
// |r| |R - 1/18| < 29 u 2^-58.  q itself lies at least u/18 from every
// rounding midpoint (t - 18 (2k+1) u/2 is an odd multiple of u), so both
// round to the same double.  t here is 0 or a normal number (a combination
// of angles in degrees), far from the subnormal range.
__device__ inline double div18(double t) {
    constexpr double R = 1.0 / 18.0;
    const double q0 = t * R;
    const double r = fma(-q0, 18.0, t);
    return fma(r, R, q0);
}

// The peak of one pair's histogram evaluated term by term, the lane's point
// against every triangle: chunks of 64 third images are dealt to four partial
// sums, each adding its triangles in k3 order, and those are added in order.
// One exponential per point and triangle.  Called by the whole wave.
__device__ inline int peak_by_terms(int K, int n_theta, const unsigned short* r1, const unsigned short* r2,
                                          const unsigned short* c1, const unsigned short* c2, int k1, int l12,
                                          int l21, const double2* cs, int lane) {
    const double x = lane < NT ? tick(lane) : 0.0;
    double v = 0.0;
    for (int w = 0; w < 4; w++) {
        double h = 0.0;
        for (int base = 64 * w; base < K; base += 256) {
            const int k3 = base + lane;
            const double ang = k3 < K ? vote_angle(r1, r2, c1, c2, k1, k3, l12, l21, cs, n_theta) : NAN;
            const long long ab = __double_as_longlong(ang);
            const int alo = (int)ab, ahi = (int)(ab >> 32);
            unsigned long long m = __ballot(!isnan(ang));
            while (m) {
                const int q = __builtin_ctzll(m);
                m &= m - 1;
                const unsigned lo = (unsigned)__builtin_amdgcn_readlane(alo, q);
                const long long hi = (long long)__builtin_amdgcn_readlane(ahi, q);
                const double a = __longlong_as_double((hi << 32) | lo);
                double t = 2 * a * x;
                t = t - a * a;
                t = t - x * x;
                h = h + exp(div18(t));
            }
        }
        v = w == 0 ? h : v + h;
    }
    // the first of the largest points
    int d = lane;
    if (lane >= NT) v = -1.0;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        const double ov = __shfl_xor(v, o, 64);
        const int od = __shfl_xor(d, o, 64);
        if (ov > v || (ov == v && od < d)) {
            v = ov;
            d = od;
        }
    }
    return v > 0.0 ? d : -1;
}

// Sum over the 64 lanes in a fixed order, the same in every lane: DPP adds
// within each row of 16 lanes, then the four row sums in row order.  Every
// lane of the wave must be active.
template <int CTRL>
__device__ inline double dpp_d(double x) {
    const unsigned long long u = __double_as_longlong(x);
    const int lo = __builtin_amdgcn_update_dpp(0, (int)(u & 0xffffffffu), CTRL, 0xf, 0xf, false);
    const int hi = __builtin_amdgcn_update_dpp(0, (int)(u >> 32), CTRL, 0xf, 0xf, false);
    return __longlong_as_double((long long)(((unsigned long long)(unsigned)hi << 32) | (unsigned)lo));
}
__device__ inline double readlane_d(double x, int l) {
    const unsigned long long u = __double_as_longlong(x);
    const unsigned lo = (unsigned)__builtin_amdgcn_readlane((int)(u & 0xffffffffu), l);
    const unsigned hi = (unsigned)__builtin_amdgcn_readlane((int)(u >> 32), l);
    return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}
__device__ inline double wave_sum(double x) {
    x += dpp_d<0xb1>(x);
    x += dpp_d<0x4e>(x);
    x += dpp_d<0x124>(x);
    x += dpp_d<0x128>(x);
    return ((readlane_d(x, 0) + readlane_d(x, 16)) + readlane_d(x, 32)) + readlane_d(x, 48);
}

// ------------------------------------------------------------- the vote
// Gaussians of the 60 histogram points as an outer product.  Point d = 8 i + j
// (i, j < 8; points 60..63 are ignored) sits at X_i + y_j, X_i = (8 i + 3.5) D
// the middle of its group of eight, y_j = (j - 3.5) D, D = 180/59, and
//   exp(-(a - X_i - y_j)^2/18) = exp(-(a - X_i)^2/18) exp(a y_j/9)
//                                * exp(-y_j^2/18 - X_i y_j/9),
// so the sum over the triangles k is a contraction of A(i, k) and B(k, j),
// followed by a factor per point: one v_mfma_f64_4x4x4 (four 4 x 4 blocks)
// adds four triangles to all 64 points.  A triangle needs three exponents
// instead of 60: u = exp(a D/18), whose odd powers are its row of B, and
// A(i0) of its own group i0, from which A(i0 +- 1) follow by u^(+-16); the
// groups beyond those are below 6e-17 of the triangle's own peak value and
// are left zero.
//
// The two sums differ by rounding only: the exponents here and in
// peak_by_terms are within 2000 in magnitude, so every term above 1e-17 of
// its triangle's largest is within 1e-12 relative, and the largest point is
// certain when no other comes within PEAK_GAP (relative) of it.  Otherwise
// (exact ties, as with a single triangle halfway between two points) the
// histogram is evaluated term by term.
constexpr double PEAK_GAP = 1e-9;
constexpr int NG = 8;          // groups, and points per group
constexpr int WPB = 8;         // waves (pairs) per workgroup
constexpr double DTICK = 180.0 / (NT - 1);

// 1/x to a few units in the last place (x normal, far from the range's ends):
// the hardware estimate and two Newton steps.
__device__ inline double recip(double x) {
    double y = __builtin_amdgcn_rcp(x);
    y = fma(fma(-x, y, 1.0), y, y);
    return fma(fma(-x, y, 1.0), y, y);
}

constexpr int AMBIGUOUS = -2;  // peak[e]: left to terms_kernel

// The clstack rows and columns of a pair and its own lines.
struct PairLines {
    const unsigned short *r1, *r2, *c1, *c2;
    int k1, k2, l12, l21;
};
__device__ inline PairLines lines_of(long long e, int K, const unsigned short* M, const unsigned short* MT) {
    PairLines p;
    pair_of(e, K, p.k1, p.k2);
    p.k1 = __builtin_amdgcn_readfirstlane(p.k1);
    p.k2 = __builtin_amdgcn_readfirstlane(p.k2);
    p.r1 = M + (size_t)p.k1 * K;   // clstack(k1, :)
    p.r2 = M + (size_t)p.k2 * K;   // clstack(k2, :)
    p.c1 = MT + (size_t)p.k1 * K;  // clstack(:, k1)
    p.c2 = MT + (size_t)p.k2 * K;  // clstack(:, k2)
    p.l12 = p.r1[p.k2];
    p.l21 = p.r2[p.k1];
    return p;
}

// Bound: FP64 issue (380 vector instructions per 64 triangles: the angles and
// two exponentials, one lane each; the MFMAs are a sixth of the time).  6.3 ms
// at K = 1000, n_theta = 360 (5e5 pairs x 1000 triangles); an exponential per
// point and triangle took 20.8 ms.  8 KB of LDS per wave hold the operands of 64
// triangles, written one triangle per lane and read in the MFMA's layout
// (16-byte pieces swizzled so that both touch every bank once).
__global__ __launch_bounds__(64 * WPB, 4) void peak_kernel(int K, int n_theta, const unsigned short* M,
                                                           const unsigned short* MT, const double2* cs_g, int* peak,
                                                           int cs_lds) {
    __shared__ __align__(16) double s_a[WPB][64 * NG];
    __shared__ __align__(16) double s_b[WPB][64 * NG];
    __shared__ double s_up[NG], s_dn[NG];  // A(i +- 1)/A(i) at a = 0
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const double GS = NG * DTICK;  // group spacing
    if (tid < NG) {
        const double X = (NG * tid + 3.5) * DTICK;
        s_up[tid] = exp(-X * GS / 9 - GS * GS / 18);
        s_dn[tid] = exp(X * GS / 9 - GS * GS / 18);
    }
    double* const sa = s_a[wave];
    double* const sb = s_b[wave];
    for (int i = lane; i < 64 * NG; i += 64) sa[i] = 0.0;
    const double2* cs = stage_trig(cs_g, n_theta, cs_lds);
    __syncthreads();
    // element (triangle t, c) of an operand: 16-byte piece c/2 of row t stored
    // at piece (c/2) ^ (t/4 % 4)
    auto at = [](int t, int c) { return t * NG + 2 * (((c >> 1) ^ (t >> 2)) & 3) + (c & 1); };
    // this lane's point: block (bi, bj) of the 8 x 8 points, row lane/16 and
    // column lane%4 of the block in the result; as an operand, row (column)
    // lane%4 and triangle lane/16
    const int bi = (lane >> 3) & 1, bj = (lane >> 2) & 1;
    const int pi = 4 * bi + (lane >> 4), pj = 4 * bj + (lane & 3);
    const int d = NG * pi + pj;
    const double yj = (pj - 3.5) * DTICK;
    const double scale = exp(-yj * yj / 18 - (NG * pi + 3.5) * DTICK * yj / 9);
    const int ca = 4 * bi + (lane & 3), cb = 4 * bj + (lane & 3);
    const long long P = (long long)K * (K - 1) / 2;
    const int wid = __builtin_amdgcn_readfirstlane(wave);
    for (long long e = (long long)blockIdx.x * WPB + wid; e < P; e += (long long)gridDim.x * WPB) {
        const PairLines p = lines_of(e, K, M, MT);
        int pk = -1;  // no common line, or no triangle voted
        if (p.l12 != 0) {
            double h = 0.0;
            bool any = false;
            for (int base = 0; base < K; base += 64) {
                const int k3 = base + lane;
                const double cp =
                    k3 < K ? vote_cos(p.r1, p.r2, p.c1, p.c2, p.k1, k3, p.l12, p.l21, cs, n_theta) : NAN;
                const bool on = !isnan(cp);
                if (!__ballot(on)) continue;
                any = true;
                const double a = on ? acos(cp) * (180 / M_PI) : 0.0;
                const int i0 = min(NG - 1, (int)((a * (1.0 / DTICK) + 0.5) * (1.0 / NG)));
                const double dx = a - (NG * i0 + 3.5) * DTICK;
                const double u = exp(a * (DTICK / 18)), w = recip(u);
                const double u2 = u * u, w2 = w * w;
                const double u3 = u * u2, w3 = w * w2, u5 = u3 * u2, w5 = w3 * w2;
                const double row[NG] = {w5 * w2, w5, w3, w, u, u3, u5, u5 * u2};
                const double u16 = (u5 * u3) * (u5 * u3), w16 = (w5 * w3) * (w5 * w3);
                const double g = on ? exp(-dx * dx * (1.0 / 18)) : 0.0;
#pragma unroll
                for (int c = 0; c < NG; c += 2) *(double2*)(sb + at(lane, c)) = make_double2(row[c], row[c + 1]);
                sa[at(lane, i0)] = g;
                if (i0 > 0) sa[at(lane, i0 - 1)] = g * w16 * s_dn[i0];
                if (i0 < NG - 1) sa[at(lane, i0 + 1)] = g * u16 * s_up[i0];
                __builtin_amdgcn_wave_barrier();
#pragma unroll 4
                for (int q = 0; q < 16; q++) {
                    const int t = 4 * q + (lane >> 4);
                    h = __builtin_amdgcn_mfma_f64_4x4x4f64(sa[at(t, ca)], sb[at(t, cb)], h, 0, 0, 0);
                }
                __builtin_amdgcn_wave_barrier();
                sa[at(lane, i0)] = 0.0;
                if (i0 > 0) sa[at(lane, i0 - 1)] = 0.0;
                if (i0 < NG - 1) sa[at(lane, i0 + 1)] = 0.0;
            }
            if (any) {
                const double v = d < NT ? h * scale : 0.0;
                double best = v;
#pragma unroll
                for (int o = 32; o > 0; o >>= 1) best = fmax(best, __shfl_xor(best, o, 64));
                const unsigned long long m = __ballot(!(v < best * (1.0 - PEAK_GAP)));
                pk = __popcll(m) == 1 ? __builtin_amdgcn_readlane(d, __builtin_ctzll(m)) : AMBIGUOUS;
            }
        }
        if (lane == 0) peak[e] = pk;
    }
}

// The pairs that peak_kernel left open (few): each wave scans 64 pairs at a
// time and evaluates the open ones one after another.
__global__ __launch_bounds__(256) void terms_kernel(int K, int n_theta, const unsigned short* M,
                                                    const unsigned short* MT, const double2* cs, int* peak) {
    const int lane = threadIdx.x & 63;
    const int wid = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const long long P = (long long)K * (K - 1) / 2;
    for (long long e0 = ((long long)blockIdx.x * 4 + wid) * 64; e0 < P; e0 += (long long)gridDim.x * 256) {
        unsigned long long todo = __ballot(e0 + lane < P && peak[e0 + lane] == AMBIGUOUS);
        while (todo) {
            const long long e = e0 + __builtin_ctzll(todo);
            todo &= todo - 1;
            const PairLines p = lines_of(e, K, M, MT);
            const int pk = peak_by_terms(K, n_theta, p.r1, p.r2, p.c1, p.c2, p.k1, p.l12, p.l21, cs, lane);
            if (lane == 0) peak[e] = pk;
        }
    }
}

// Triangles within 6 degrees of each pair's peak: their relative rotations,
// averaged into the pair's 2x2 block of S and its transpose.  The rotation's
// second Euler angle has cosine
//   (c - a b)/sqrt(1 - a^2)/sqrt(1 - b^2), negated when the line differences
// of a and b lie on different sides (rotratio_eulerangle_vec.m), a, b, c the
// cosines of the triangle's three line differences: that is the triangle's own
// cosine with the sign of sin t1 sin t2 undone and redone, its negative.  The
// other two angles are the pair's, so one sum over the triangles is enough.
// 2.2 ms at K = 1000; with a workgroup per pair and the rotation's square
// roots, arc cosine and cosine per triangle it took 8.6 ms.
__global__ __launch_bounds__(64 * WPB) void rot_kernel(int K, int n_theta, const unsigned short* M,
                                                       const unsigned short* MT, const double2* cs_g,
                                                       const double2* ln, const Window* win, const int* peak,
                                                       double* S, int cs_lds) {
    const int lane = threadIdx.x & 63;
    const int wid = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const double2* cs = stage_trig(cs_g, n_theta, cs_lds);
    const long long P = (long long)K * (K - 1) / 2;
    const size_t n2 = 2 * (size_t)K;
    for (long long e = (long long)blockIdx.x * WPB + wid; e < P; e += (long long)gridDim.x * WPB) {
        const PairLines p = lines_of(e, K, M, MT);
        const int pk = __builtin_amdgcn_readfirstlane(peak[e]);  // -1: no common line or no vote
        double r00 = 0, r01 = 0, r10 = 0, r11 = 0;
        if (pk >= 0) {
            const double xp = tick(pk);
            const Window w = win[pk];
            int cnt = 0, nrot = 0;
            double sum = 0.0;
            for (int k3 = lane; k3 < K; k3 += 64) {
                const double cp = vote_cos(p.r1, p.r2, p.c1, p.c2, p.k1, k3, p.l12, p.l21, cs, n_theta);
                if (isnan(cp) || cp >= w.o_hi || cp <= w.o_lo) continue;
                if (!(cp < w.i_hi && cp > w.i_lo) && !(fabs(acos(cp) * 180 / M_PI - xp) < 360.0 / NT)) continue;
                cnt++;
                // the rotation's own degeneracy test, with its cosines' order
                const double a = trig(cs, n_theta, (int)p.c2[k3] - (int)p.c1[k3]).x;
                const double b = trig(cs, n_theta, (int)p.r2[k3] - p.l21).x;
                const double c = trig(cs, n_theta, (int)p.r1[k3] - p.l12).x;
                const double cond = 1 + 2 * a * b * c - (a * a + b * b + c * c);
                if (!(cond > 1.0e-5)) continue;
                nrot++;
                sum -= cp;
            }
            sum = wave_sum(sum);
            const double n = wave_sum((double)cnt), nr = wave_sum((double)nrot);
            if (n > 0) {
                const double2 l1 = ln[min(p.l21, n_theta)], l3 = ln[min(p.l12, n_theta)];
                const double ca = l1.x, sa = -l1.y, cc = l3.x, sc = l3.y;
                r00 = (nr * (cc * ca) - sum * (sc * sa)) / n;
                r01 = (-nr * (cc * sa) - sum * (sc * ca)) / n;
                r10 = (nr * (sc * ca) + sum * (cc * sa)) / n;
                r11 = (-nr * (sa * sc) + sum * (cc * ca)) / n;
            }
        }
        if (lane < 4) {
            const int a = lane >> 1, b = lane & 1;
            const double v = lane == 0 ? r00 : lane == 1 ? r01 : lane == 2 ? r10 : r11;
            S[(2 * (size_t)p.k2 + b) * n2 + 2 * (size_t)p.k1 + a] = v;  // S(2k1+a, 2k2+b) = R22(a,b)
            S[(2 * (size_t)p.k1 + a) * n2 + 2 * (size_t)p.k2 + b] = v;  // S(2k2+b, 2k1+a)
        }
    }
}

}  // namespace vote

using namespace clmh;

extern "C" int clm_syncmatrix_vote(clm_ctx* c, int32_t K, int32_t n_theta, const int32_t* d_cl1,
                                   const int32_t* d_cl2, double* d_S, clm_vote_stats* st) {
    using namespace vote;
    if (!c) return CLM_E_ARG;
    if (st) *st = clm_vote_stats{};
    if (K < 1 || K > 65536) return fail(c, CLM_E_ARG, "K = %d outside [1, 65536]", K);
    if (n_theta <= 0 || n_theta > 65535) return fail(c, CLM_E_ARG, "invalid n_theta %d", n_theta);
    if (!d_S || (K > 1 && (!d_cl1 || !d_cl2))) return fail(c, CLM_E_ARG, "null pointer");
    HIPCHK(c, hipSetDevice(c->device));
    int rc;
    const size_t kk = (size_t)K * K;
    const long long P = (long long)K * (K - 1) / 2;
    if ((rc = ensure(c, c->vt_m, kk * 2)) || (rc = ensure(c, c->vt_mt, kk * 2)) ||
        (rc = ensure(c, c->vt_pk, (size_t)std::max<long long>(P, 1) * 4)) ||
        (rc = ensure(c, c->vt_cs, (size_t)(3 * n_theta + 2) * sizeof(double2) + NT * sizeof(Window))))
        return rc;
    unsigned short* M = (unsigned short*)c->vt_m.p;
    unsigned short* MT = (unsigned short*)c->vt_mt.p;
    int* pk = (int*)c->vt_pk.p;
    double2* cs = (double2*)c->vt_cs.p;
    double2* ln = cs + 2 * (size_t)n_theta + 1;
    Window* win = (Window*)(ln + n_theta + 1);
    HIPCHK(c, hipEventRecord(c->ev[0], c->stream));
    setup_kernel<<<K + std::max(2 * n_theta + 1, NT) / 256 + 1, 256, 0, c->stream>>>(K, n_theta, d_cl1, d_cl2, M, MT,
                                                                                     cs, ln, win, d_S);
    HIPCHK(c, hipGetLastError());
    HIPCHK(c, hipEventRecord(c->ev[1], c->stream));
    if (P > 0) {
        const long long nb = std::min<long long>((P + WPB - 1) / WPB, (long long)c->n_cu * 8);
        const long long nt = std::min<long long>((P + 255) / 256, (long long)c->n_cu * 8);
        // the (cos, sin) table in LDS up to 16 KB (n_theta <= 511)
        const size_t cs_bytes = (size_t)(2 * n_theta + 1) * sizeof(double2);
        const int cs_lds = cs_bytes <= 16384;
        const size_t lds = cs_lds ? cs_bytes : 0;
        peak_kernel<<<(unsigned)nb, 64 * WPB, lds, c->stream>>>(K, n_theta, M, MT, cs, pk, cs_lds);
        terms_kernel<<<(unsigned)nt, 256, 0, c->stream>>>(K, n_theta, M, MT, cs, pk);
        rot_kernel<<<(unsigned)nb, 64 * WPB, lds, c->stream>>>(K, n_theta, M, MT, cs, ln, win, pk, d_S, cs_lds);
        HIPCHK(c, hipGetLastError());
    }
    HIPCHK(c, hipEventRecord(c->ev[2], c->stream));
    HIPCHK(c, hipStreamSynchronize(c->stream));
    if (st) {
        float a = 0.f, b = 0.f;
        HIPCHK(c, hipEventElapsedTime(&a, c->ev[0], c->ev[1]));
        HIPCHK(c, hipEventElapsedTime(&b, c->ev[1], c->ev[2]));
        st->ms_build = a;
        st->ms_vote = b;
        st->pairs = P;
    }
    return CLM_OK;
}
