// pft.hip -- polar Fourier transform of a projection stack on the device:
// the step before the common-lines search.
//
// Replaces cryo_pft(p, n_r, n_theta) (fourier/nufft/cryo_pft.m:1-75) with its
// exact evaluation, the non-uniform DFT of fourier/nufft/nudft2.m:40-47 (the
// reference's own fallback when no NUFFT library is installed):
//
//   freqs(m) = ((k)*w0*sin(j*dtheta), (k)*w0*cos(j*dtheta)),  m = j*n_r + k,
//       w0 = 2*pi/(2*n_r - 1), dtheta = 2*pi/n_theta, j < n_theta/2  (:49-58)
//   pf(k, j, i) = sum_{u,v} p(u, v, i) * exp(+1i*(fx(m)*g(u) + fy(m)*g(v)))
//       g(t) = ceil(t - n/2)      (nudft2.m:40-47 evaluated at -freqs, :70)
//   pf(:, n_theta/2 + j, :) = conj(pf(:, j, :))                        (:75)
//
// u is the first (row) index of an image, paired with fx = r*sin(theta); v is
// the second, paired with fy = r*cos(theta).
//
// On the device this is a contraction over the pixels on FP64 MFMA
// (v_mfma_f64_16x16x4f64).  The images are real and the points come in
// quadruples of frequencies (+-fx, +-fy) (ray j, its mirror n_theta/2 - j and
// their conjugates), so the pixels are first folded over both axes into four
// planes, even or odd in u and in v, a = |g(u)|, b = |g(v)|:
//   Scc = sum cos(fx a) cos(fy b) pee(a, b)    Sss = sum sin sin poo
//   Ssc = sum sin(fx a) cos(fy b) poe(a, b)    Scs = sum cos sin peo
//   pf(j) = Scc - Sss + i (Ssc + Scs)          pf(n_theta/2 - j) = Scc + Sss + i (Ssc - Scs)
// Four real products over a quarter of the pixels serve two rays: a quarter
// of the multiplications of the sums as written.  The weights are never
// stored: a lane forms its operand as one product of two table entries.
// Two rays that share a quadrant point have rounded frequencies that differ in
// the last bits.  Ray j's are taken for the sums; for the mirror ray the
// differences times the sums' derivatives are added (shift_kernel), a
// contraction of the same shape whose values are 1e-14 of pf's, so that
// operands of 11 bits leave less than 1e-16.  Error over max |pf| of white noise
// in extended precision, n = 129 and n_r = 65: 2.8e-15 at worst, 7.5e-16 rms; with
// the mean of the two frequencies for both rays 1.2e-14 and 2.4e-15; the sums as
// written with phases rounded to a double, or weights advanced by rotations,
// 1.5e-14 and 6.1e-15.
//
// CLM_PFT_NUFFT: the same sums by a type-2 non-uniform FFT, the method the
// reference's nufft2 uses when a NUFFT library is installed
// (fourier/nufft/nufft_transform.m:108-150, finufft with epsilon 1e-15 by
// default, nufft_initialize.m:29).  Own implementation of the published
// exponential-of-semicircle method (Barnett, Magland and af Klinteberg, SIAM
// J. Sci. Comput. 41(5), 2019): kernel phi(z) = exp(beta (sqrt(1 - z^2) - 1))
// of width NW = 16 grid points, beta = 2.30 NW, on an oversampled grid of
// side N >= 2n (2,3,5-smooth).  Per image:
//   a(x mod N, y mod N) = p(u, v) / (Phi(x) Phi(y)),  x = g(u), y = g(v)
//   b = the unnormalized backward 2-D FFT of a (sum a e^{+2 pi i l x / N})
//   pf(m) = sum_{t, r < NW} phi(2 (sx - lx - t)/NW) phi(2 (sy - ly - r)/NW) b(lx + t, ly + r)
// Images are real, so b(-x, -y) = conj b(x, y) and the points' fx are in [0, pi):
// an image keeps the columns x = 0..N/2 of its grid alone, and a window's few
// columns beyond them are read from their mirrors.  Along x two rows of an image
// go through one complex transform and are taken apart as they are turned.  Half
// the grids and transforms of a complex grid per image, and an image shares
// nothing with its neighbours in the stack: two images in one complex grid cost
// the same, and put the rounding of one's spectrum on the other's (a point
// source, n = 359: 2.0e-14 of its own max |pf|, beside a constant in one grid
// 6.0e-14).
// Here sx = fx(m) N / (2 pi), lx = ceil(sx - NW/2) (sy, ly alike, indices mod
// N) and Phi(x) = int phi(2s/NW) cos(2 pi s x / N) ds over |s| <= NW/2, the
// kernel's Fourier transform (Gauss-Legendre quadrature).  The
// result differs from the exact sums by about 1e-14 of max |pf|.
#include <hip/hip_runtime.h>
#include <hipfft/hipfft.h>

#include <cmath>
#include <vector>

#include "clm_ctx.h"

namespace pft {

typedef double d4 __attribute__((ext_vector_type(4)));
typedef double d2 __attribute__((ext_vector_type(2)));
typedef float f4 __attribute__((ext_vector_type(4)));
typedef _Float16 h2 __attribute__((ext_vector_type(2)));
typedef _Float16 h8 __attribute__((ext_vector_type(8)));

constexpr int KCHUNK = 8192;  // images per staged chunk
constexpr int FA = 32;        // folded columns per staging workgroup

struct Geo {
    int n, n_r, n_theta;
    int M, Mp;       // quadrant points n_r * (n_theta/4 + 1), rows of the tables (padded for the row tiles)
    int c;           // pixel index of the origin: g(c) = 0
    int nh, nab;     // folded side floor(n/2) + 1, blocks of 4 of it
    int nb8;         // blocks of 8 of the folded side
    int Kc, nct;     // images in this chunk, column tiles of 16
};

// tab[0][a*Mp + m] = cos(fx(m) a), tab[1] sin; then cos(fy(m) b) and
// sin(fy(m) b), 4 nab rows each (zero for m >= M).  grid: (Mp/256, 8 nab).
// ray: sin(j dtheta), then cos(j dtheta), j < n_theta/2, as cryo_pft.m:52-58 has
// them.  The phase keeps the product's rounding error.
// dx[a*Mp + m] = (cos(fx a), d a), (sin, d a) for the shift from fx to the
// mirror ray's frequency fx + d: (X, X') of shift_kernel, X' = 2^DSCALE d dX/dfx;
// along y eight b to a point, Y then Y': dy[((kind*nb8 + b/8)*Mp + m)*16 + b%8].
// Null where they are not used.
constexpr int DSCALE = 44;
__global__ void tables_kernel(Geo g, const double* __restrict__ ray, double* tab, h2* dx, _Float16* dy) {
    const int m = blockIdx.x * blockDim.x + threadIdx.x;
    if (m >= g.Mp) return;
    const int na = 4 * g.nab, L = g.n_theta / 2;
    const bool is_x = (int)blockIdx.y < na;
    const int idx = is_x ? blockIdx.y : blockIdx.y - na;
    double s = 0.0, c = 0.0, d = 0.0;
    if (m < g.M) {
        const int k = m % g.n_r, j = m / g.n_r;
        const int jm = L - j;  // the mirrored ray
        const double r = k * (2.0 * M_PI / (2.0 * g.n_r - 1.0));  // cryo_pft.m:49
        const double* t = is_x ? ray : ray + L;
        const double f = r * t[j];
        if (j > 0 && j < jm) d = (is_x ? r * t[jm] : -r * t[jm]) - f;
        const double ph = f * idx, lo = fma(f, (double)idx, -ph);
        double s0, c0;
        sincos(ph, &s0, &c0);
        s = fma(c0, lo, s0);
        c = fma(-s0, lo, c0);
    }
    double* t = tab + (size_t)(is_x ? 0 : 2) * na * g.Mp + (size_t)idx * g.Mp + m;
    t[0] = c;
    t[(size_t)na * g.Mp] = s;
    if (!dx) return;
    d = ldexp(d, DSCALE) * idx;
    const h2 vc = {(_Float16)c, (_Float16)(-d * s)}, vs = {(_Float16)s, (_Float16)(d * c)};
    if (is_x) {
        dx[(size_t)idx * g.Mp + m] = vc;
        dx[(size_t)(na + idx) * g.Mp + m] = vs;
        return;
    }
    const size_t kind = (size_t)g.nb8 * g.Mp * 16;
    _Float16* y = dy + ((size_t)(idx / 8) * g.Mp + m) * 16 + idx % 8;
    y[0] = vc.x;
    y[8] = vc.y;
    y[kind] = vs.x;
    y[kind + 8] = vs.y;
    if (idx + 4 >= na && idx + 4 < 8 * g.nb8)  // past the last four rows
        y[4] = y[12] = y[kind + 4] = y[kind + 12] = (_Float16)0.f;
}

// Folded images, one 512-byte block per (column tile of 16 images, plane,
// 4 values of a, b), the operand of one MFMA:
//   xt[(((ct*4 + plane)*nab + a/4)*nh + b)*64 + (a%4)*16 + image%16],
// planes ee, oo, oe (odd in u), eo; zero past nh and past the last image.
// One workgroup folds FA columns a of the two rows +-b of 16 images: the rows
// are read along u (contiguous) into LDS and written along the images.
// part[(ct*nh + b)*gridDim.x + blockIdx.x][16]: the high word of the largest |p|
// the workgroup has seen of each image.
template <typename T>
__global__ __launch_bounds__(256) void fold_kernel(Geo g, const T* __restrict__ img, long long k0,
                                                   double* __restrict__ xt, unsigned* __restrict__ part) {
    __shared__ double s_p[4][16][FA + 1];  // p(+a,+b), p(-a,+b), p(+a,-b), p(-a,-b), zero where not a pixel
    const int a0 = blockIdx.x * FA, b = blockIdx.y, ct = blockIdx.z;
    const int tid = threadIdx.x;
    unsigned hi[2] = {0, 0};  // of images tid/FA and tid/FA + 8
    static_assert(FA == 32, "half waves");
#pragma unroll
    for (int s = 0; s < 4 * 16 * FA / 256; s++) {
        const int x = tid + 256 * s;
        const int da = x % FA, i = (x / FA) % 16, q = x / (16 * FA);
        const int a = a0 + da;
        // the axes' own pixels count once
        const int u = q & 1 ? g.c - a : g.c + a, v = q & 2 ? g.c - b : g.c + b;
        const bool ok = u >= 0 && u < g.n && v >= 0 && v < g.n && 16 * ct + i < g.Kc && !((q & 1) && a == 0) &&
                        !((q & 2) && b == 0);
        const double p = ok ? (double)img[((size_t)(k0 + 16 * ct + i) * g.n + v) * g.n + u] : 0.0;
        s_p[q][i][da] = p;
        hi[s & 1] = max(hi[s & 1], (unsigned)(__double_as_longlong(p) >> 32) & 0x7fffffffu);
    }
#pragma unroll
    for (int h = 0; h < 2; h++) {
        for (int o = FA / 2; o; o >>= 1) hi[h] = max(hi[h], (unsigned)__shfl_xor((int)hi[h], o, FA));
        if (tid % FA == 0) part[(((size_t)ct * g.nh + b) * gridDim.x + blockIdx.x) * 16 + tid / FA + 8 * h] = hi[h];
    }
    __syncthreads();
    for (int x = tid; x < 16 * FA; x += 256) {
        const int i = x % 16, da = x / 16;
        const int a = a0 + da;
        if (a >= 4 * g.nab) break;
        const double pp = s_p[0][i][da], np = s_p[1][i][da], pn = s_p[2][i][da], nn = s_p[3][i][da];
        const double ep = pp + np, op = pp - np, en = pn + nn, on = pn - nn;
        const bool oa = a != 0, ob = b != 0;  // odd planes vanish on their axis
        double* o = xt + (((size_t)ct * 4 * g.nab + (a >> 2)) * g.nh + b) * 64 + (a & 3) * 16 + i;
        const size_t pl = (size_t)g.nab * g.nh * 64;
        o[0] = ep + en;
        o[pl] = oa && ob ? op - on : 0.0;
        o[2 * pl] = oa ? op + on : 0.0;
        o[3 * pl] = ob ? ep - en : 0.0;
    }
}

// top[i]: the high word of image i's largest |p| (NOT_FINITE and above: it holds
// an infinity or a NaN), over the cnt workgroups that folded it (one maximum an
// image and workgroup by atomics took as long as the folding: an image tile's 16
// words are one line).  One workgroup per column tile.
constexpr unsigned NOT_FINITE = 0x7ff00000u;
__global__ __launch_bounds__(256) void top_kernel(Geo g, const unsigned* __restrict__ part, int cnt,
                                                  unsigned* __restrict__ top) {
    __shared__ unsigned s_m[256];
    const unsigned* p = part + (size_t)blockIdx.x * cnt * 16;
    unsigned m = 0;
#pragma unroll 4
    for (int q = threadIdx.x; q < 16 * cnt; q += 256) m = max(m, p[q]);
    s_m[threadIdx.x] = m;
    __syncthreads();
    if (threadIdx.x < 16) {
        for (int q = 1; q < 16; q++) m = max(m, s_m[threadIdx.x + 16 * q]);
        top[16 * blockIdx.x + threadIdx.x] = m;
    }
}
__device__ inline int top_exponent(unsigned top) { return (int)(top >> 20) - 1023; }

template <typename OutT>
__device__ inline void put(OutT* pf, size_t at, double re, double im);
template <>
__device__ inline void put<double2>(double2* pf, size_t at, double re, double im) {
    pf[at] = make_double2(re, im);
}
template <>
__device__ inline void put<float2>(float2* pf, size_t at, double re, double im) {
    pf[at] = make_float2((float)re, (float)im);
}

// The folded images times 2^-e, e the exponent of the image's largest |p|, in
// FP16 and in the operand order of the 16 x 16 x 32 MFMA:
//   xh[(((ct*4 + plane)*nab + a/4)*nb8 + b/8)*64 + (a%4)*16 + image%16][b%8],
// zero past nh.  One workgroup per (4 values of a, plane, column tile).
__global__ __launch_bounds__(256) void narrow_kernel(Geo g, const double* __restrict__ xt,
                                                     const unsigned* __restrict__ top, h8* __restrict__ xh) {
    const size_t blk = ((size_t)blockIdx.z * 4 + blockIdx.y) * g.nab + blockIdx.x;
    const int lane = threadIdx.x & 63;
    const int e = top_exponent(top[16 * blockIdx.z + (lane & 15)]);
    const double* x = xt + blk * g.nh * 64 + lane;
    for (int bb = threadIdx.x >> 6; bb < g.nb8; bb += 4) {
        h8 v;
#pragma unroll
        for (int q = 0; q < 8; q++) {
            const int b = 8 * bb + q;
            v[q] = (_Float16)(b < g.nh ? (float)ldexp(x[(size_t)b * 64], -e) : 0.f);
        }
        xh[(blk * g.nb8 + bb) * 64 + lane] = v;
    }
}

// What the mirror rays' sums change by from ray j's frequencies to their own,
// times 2^(DSCALE - e): shift[i*Mp + m].  With (X, X') and (Y, Y') of the tables,
// the plane's weights change by X' Y + X Y'.  Tiles, waves and planes as in
// pft_kernel; a lane forms its eight weights of a row tile (one a, eight b) by
// packed FP16 operations from one X pair and eight Y pairs that it keeps over the
// loop of a; the next PD values' operands are on their way meanwhile.
// 243 us for 1000 images of 129 x 129, n_r = 65, n_theta = 360 (the sums take
// 3.24 ms), 1.0 PFLOP/s.  Bound: the weights' vector instructions (the vector units
// are busy 50% of the cycles, the matrix cores 48%, in turn); tiles of 8 x 4 form
// each weight for twice the MFMAs' share and took 212 us, but leave fewer images
// without work for every CU.
template <int RT, int CT, int PD>
__global__ __launch_bounds__(256, 2) void shift_kernel(Geo g, const h8* __restrict__ xh, const h2* __restrict__ dx,
                                                       const _Float16* __restrict__ dy, float2* __restrict__ shift,
                                                       int nmb, int ntiles, int per_xcd) {
    __shared__ float s_s[4][16][16 * CT + 1];
    const int t = (blockIdx.x % 8) * per_xcd + blockIdx.x / 8;
    if (t >= ntiles) return;
    const int mb = t % nmb, kb = t / nmb;
    const int lane = threadIdx.x & 63;
    const int plane = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int r16 = lane & 15, kq = lane >> 4;
    const int m0 = mb * 16 * RT + r16;
    const h2* px = dx + (size_t)((plane == 1 || plane == 2) * 4 * g.nab + kq) * g.Mp + m0;
    const h8* py = (const h8*)(dy + ((size_t)(plane & 1) * g.nb8 * g.Mp + m0) * 16);
    const h8* bp[CT];
#pragma unroll
    for (int c = 0; c < CT; c++) {
        const int ct = min(kb * CT + c, g.nct - 1);  // past the last tile: that tile again, not stored
        bp[c] = xh + ((size_t)ct * 4 + plane) * g.nab * g.nb8 * 64 + lane;
    }
    f4 acc[RT][CT];
#pragma unroll
    for (int r = 0; r < RT; r++)
#pragma unroll
        for (int c = 0; c < CT; c++) acc[r][c] = f4{0.f, 0.f, 0.f, 0.f};
    for (int bb = 0; bb < g.nb8; bb++) {
        h8 y[RT], yd[RT], b[PD][CT];
        h2 x[PD][RT];
        auto load = [&](int ab0, h2 (&x)[PD][RT], h8 (&b)[PD][CT]) {
#pragma unroll
            for (int d = 0; d < PD; d++) {
                const int ab = min(ab0 + d, g.nab - 1);
#pragma unroll
                for (int r = 0; r < RT; r++) x[d][r] = px[(size_t)4 * ab * g.Mp + 16 * r];
#pragma unroll
                for (int c = 0; c < CT; c++) b[d][c] = bp[c][((size_t)ab * g.nb8 + bb) * 64];
            }
        };
#pragma unroll
        for (int r = 0; r < RT; r++) {
            y[r] = py[((size_t)bb * g.Mp + 16 * r) * 2];
            yd[r] = py[((size_t)bb * g.Mp + 16 * r) * 2 + 1];
        }
        load(0, x, b);
        for (int ab = 0; ab < g.nab; ab += PD) {
            h2 xn[PD][RT];
            h8 bn[PD][CT];
            load(ab + PD, xn, bn);
#pragma unroll
            for (int d = 0; d < PD; d++) {
                if (ab + d >= g.nab) break;
#pragma unroll
                for (int r = 0; r < RT; r++) {
                    const _Float16 u = x[d][r].x, v = x[d][r].y;
                    const h8 w = __builtin_elementwise_fma(h8{u, u, u, u, u, u, u, u}, yd[r], h8{v, v, v, v, v, v, v, v} * y[r]);
#pragma unroll
                    for (int c = 0; c < CT; c++)
                        acc[r][c] = __builtin_amdgcn_mfma_f32_16x16x32_f16(w, b[d][c], acc[r][c], 0, 0, 0);
                }
            }
#pragma unroll
            for (int d = 0; d < PD; d++) {
#pragma unroll
                for (int r = 0; r < RT; r++) x[d][r] = xn[d][r];
#pragma unroll
                for (int c = 0; c < CT; c++) b[d][c] = bn[d][c];
            }
        }
    }
    // D tile of the FP32 16x16 MFMAs: lane l, element e holds row 4*(l/16) + e
#pragma unroll
    for (int r = 0; r < RT; r++) {
        __syncthreads();
#pragma unroll
        for (int c = 0; c < CT; c++)
#pragma unroll
            for (int e = 0; e < 4; e++) s_s[plane][4 * kq + e][16 * c + r16] = acc[r][c][e];
        __syncthreads();
#pragma unroll
        for (int q = 0; q < CT; q++) {
            const int row = threadIdx.x & 15, col = (threadIdx.x >> 4) + 16 * q;
            const int m = (mb * RT + r) * 16 + row, i = kb * 16 * CT + col;
            if (m < g.M && i < g.Kc)
                shift[(size_t)i * g.Mp + m] = make_float2(s_s[0][row][col] + s_s[1][row][col], s_s[2][row][col] - s_s[3][row][col]);
        }
    }
}

template <int RT, int CT, int PD>
void shift_launch(hipStream_t st, const Geo& g, const h8* xh, const h2* dx, const _Float16* dy, float2* shift) {
    const int nmb = (g.M + 16 * RT - 1) / (16 * RT), ntiles = nmb * ((g.nct + CT - 1) / CT);
    const int per = (ntiles + 7) / 8;
    shift_kernel<RT, CT, PD><<<8 * per, 256, 0, st>>>(g, xh, dx, dy, shift, nmb, ntiles, per);
}

// One workgroup: 16 RT quadrant points x 16 CT images; wave w contracts plane
// w.  Each step is 4 folded pixels (4 values of a, one b): lane l holds pixel
// a = l/16 of point l%16 of a row tile (A, the product of a table entry along
// a, kept over the loop of b, and one along b) and of image l%16 of a column
// tile (B, one contiguous 512-byte block); the next step's loads are issued
// before this step's MFMAs.  RT x CT accumulator tiles of 16 x 16 FP64.  At
// the end the four planes meet in LDS and every quadrant point gives its two
// rays and their conjugate rays, written along the ray.
// The 1-D grid gives each XCD (dispatch goes round-robin over 8) a contiguous
// range of tiles, points fastest, so that its workgroups stream the same
// images through its L2.
// Bound: FP64 MFMA (busy 86% of the cycles).  3.24 ms for 1000 images of 129 x 129,
// n_r = 65, n_theta = 360: 65 TFLOP/s of the folded work (a large FP64 matrix product
// reaches 72 here).  The unfolded contraction, 3.9 times the work, took 13.7 ms
// at 57 TFLOP/s.  Smaller tiles than 4 x 4 only where they leave fewer MFMA
// cycles on the busiest CU (few images or points).
template <typename OutT, int RT, int CT>
__global__ __launch_bounds__(256, 2) void pft_kernel(Geo g, const double* __restrict__ xt,
                                                     const double* __restrict__ tab,
                                                     const float2* __restrict__ shift,
                                                     const unsigned* __restrict__ top, OutT* __restrict__ pf,
                                                     long long k0, int nmb, int ntiles, int per_xcd) {
    __shared__ double s_s[4][16][16 * CT + 1];
    const int t = (blockIdx.x % 8) * per_xcd + blockIdx.x / 8;
    if (t >= ntiles) return;
    const int mb = t % nmb, kb = t / nmb;
    const int lane = threadIdx.x & 63;
    const int plane = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int r16 = lane & 15, kq = lane >> 4;
    const int na = 4 * g.nab;
    const double* tx = tab + (size_t)(plane == 1 || plane == 2) * na * g.Mp + (size_t)kq * g.Mp + mb * 16 * RT + r16;
    const double* ty = tab + (size_t)(2 + (plane & 1)) * na * g.Mp + mb * 16 * RT + r16;
    const double* bp[CT];
#pragma unroll
    for (int c = 0; c < CT; c++) {
        const int ct = min(kb * CT + c, g.nct - 1);  // past the last tile: that tile again, not stored
        bp[c] = xt + ((size_t)ct * 4 + plane) * g.nab * g.nh * 64 + lane;
    }
    d4 acc[RT][CT];
#pragma unroll
    for (int r = 0; r < RT; r++)
#pragma unroll
        for (int c = 0; c < CT; c++) acc[r][c] = d4{0.0, 0.0, 0.0, 0.0};
    double y[RT], x[RT], bx[CT];
#pragma unroll
    for (int c = 0; c < CT; c++) bx[c] = bp[c][0];
#pragma unroll
    for (int r = 0; r < RT; r++) y[r] = ty[16 * r];
    const int steps = g.nab * g.nh;
    int at = 0;
    for (int ab = 0; ab < g.nab; ab++) {
#pragma unroll
        for (int r = 0; r < RT; r++) x[r] = tx[(size_t)4 * ab * g.Mp + 16 * r];
        for (int b = 0; b < g.nh; b++) {
            at++;
            const size_t nx = at < steps ? (size_t)at * 64 : 0;
            const int nb = b + 1 < g.nh ? b + 1 : 0;
            double yn[RT], bn[CT];
#pragma unroll
            for (int c = 0; c < CT; c++) bn[c] = bp[c][nx];
#pragma unroll
            for (int r = 0; r < RT; r++) yn[r] = ty[(size_t)nb * g.Mp + 16 * r];
#pragma unroll
            for (int r = 0; r < RT; r++) {
                const double w = x[r] * y[r];
#pragma unroll
                for (int c = 0; c < CT; c++)
                    acc[r][c] = __builtin_amdgcn_mfma_f64_16x16x4f64(w, bx[c], acc[r][c], 0, 0, 0);
            }
#pragma unroll
            for (int c = 0; c < CT; c++) bx[c] = bn[c];
#pragma unroll
            for (int r = 0; r < RT; r++) y[r] = yn[r];
        }
    }
    // D tile layout of the FP64 16x16x4 MFMA: lane l, element e holds row
    // 4*e + l/16, column l % 16 (one row per element, unlike the FP32 tiles).
    const int L = g.n_theta / 2;
#pragma unroll
    for (int r = 0; r < RT; r++) {
        __syncthreads();
#pragma unroll
        for (int c = 0; c < CT; c++)
#pragma unroll
            for (int e = 0; e < 4; e++) s_s[plane][4 * e + kq][16 * c + r16] = acc[r][c][e];
        __syncthreads();
#pragma unroll
        for (int q = 0; q < CT; q++) {
            const int row = threadIdx.x & 15, col = (threadIdx.x >> 4) + 16 * q;
            const int m = (mb * RT + r) * 16 + row, i = kb * 16 * CT + col;
            if (m >= g.M || i >= g.Kc) continue;
            const int k = m % g.n_r, j = m / g.n_r;
            const double cc = s_s[0][row][col], ss = s_s[1][row][col], sc = s_s[2][row][col], cs = s_s[3][row][col];
            const size_t ray = (size_t)(k0 + i) * g.n_theta;
            put<OutT>(pf, (ray + j) * g.n_r + k, cc - ss, sc + cs);
            put<OutT>(pf, (ray + j + L) * g.n_r + k, cc - ss, -(sc + cs));
            if (j > 0 && 2 * j < L) {
                double re = cc + ss, im = sc - cs;
                if (shift) {
                    const float2 d = shift[(size_t)i * g.Mp + m];
                    const int e = top_exponent(top[i]) - DSCALE;
                    re += ldexp((double)d.x, e);
                    im += ldexp((double)d.y, e);
                }
                put<OutT>(pf, (ray + L - j) * g.n_r + k, re, im);
                put<OutT>(pf, (ray + 2 * L - j) * g.n_r + k, re, -im);
            }
        }
    }
}

// The folded sums of an image that holds an infinity or a NaN mix it into
// planes that cancel or vanish; the sums as written carry it to every point with
// its weight's sign.  One workgroup per image, which returns at once if the image
// is finite; else the sums over its non-finite pixels (which decide every
// value) in place of the folded ones.
template <typename T, typename OutT>
__global__ __launch_bounds__(256) void non_finite_kernel(Geo g, const T* __restrict__ img, long long k0,
                                                         const unsigned* __restrict__ top, OutT* __restrict__ pf) {
    constexpr int NL = 1024;  // pixels looked through at a time
    __shared__ int s_list[NL];
    __shared__ int s_n;
    const size_t i = k0 + blockIdx.x;
    if (top[blockIdx.x] < NOT_FINITE) return;
    const int px = g.n * g.n, L = g.n_theta / 2, M = g.n_r * L;
    const double omega0 = 2.0 * M_PI / (2.0 * g.n_r - 1.0), dtheta = 2.0 * M_PI / g.n_theta;
    const T* p = img + i * px;
    bool first = true;
    for (int q0 = 0; q0 < px; q0 += NL) {
        if (threadIdx.x == 0) s_n = 0;
        __syncthreads();
        for (int q = q0 + threadIdx.x; q < min(q0 + NL, px); q += 256)
            if (!isfinite((double)p[q])) s_list[atomicAdd(&s_n, 1)] = q;
        __syncthreads();
        const int cnt = s_n;
        for (int m = threadIdx.x; m < M && cnt; m += 256) {
            const int k = m % g.n_r, j = m / g.n_r;
            const double fx = (k * omega0) * sin(j * dtheta), fy = (k * omega0) * cos(j * dtheta);
            double re = 0.0, im = 0.0;
            for (int c = 0; c < cnt; c++) {
                const int q = s_list[c], v = q / g.n, u = q - v * g.n;
                double sn, cs;
                sincos(fx * (u - g.c) + fy * (v - g.c), &sn, &cs);
                re += cs * (double)p[q];
                im += sn * (double)p[q];
            }
            const size_t a = (i * g.n_theta + j) * g.n_r + k, b = a + (size_t)L * g.n_r;
            if (!first) {
                re += pf[a].x;
                im += pf[a].y;
            }
            put<OutT>(pf, a, re, im);
            put<OutT>(pf, b, re, -im);
        }
        if (cnt) first = false;
        __syncthreads();
    }
}

template <int RT, int CT>
void pft_launch(hipStream_t st, const Geo& g, bool c128, const double* xt, const double* tab, const float2* shift,
                const unsigned* top, void* pf, long long k0) {
    const int nmb = (g.M + 16 * RT - 1) / (16 * RT), ntiles = nmb * ((g.nct + CT - 1) / CT);
    const int per = (ntiles + 7) / 8;
    if (c128)
        pft_kernel<double2, RT, CT><<<8 * per, 256, 0, st>>>(g, xt, tab, shift, top, (double2*)pf, k0, nmb, ntiles, per);
    else
        pft_kernel<float2, RT, CT><<<8 * per, 256, 0, st>>>(g, xt, tab, shift, top, (float2*)pf, k0, nmb, ntiles, per);
}

template <typename T>
void non_finite_launch(hipStream_t st, const Geo& g, bool c128, const T* img, long long k0, const unsigned* top,
                       void* pf) {
    if (c128) non_finite_kernel<T, double2><<<g.Kc, 256, 0, st>>>(g, img, k0, top, (double2*)pf);
    else non_finite_kernel<T, float2><<<g.Kc, 256, 0, st>>>(g, img, k0, top, (float2*)pf);
}

// ------------------------------------------------------------ type-2 NUFFT
constexpr int NW = 16;                  // kernel width, grid points per axis
constexpr double NBETA = 2.30 * NW;     // kernel shape for oversampling 2
constexpr int NCHUNK = 2048;            // images per batch of FFTs (at most)
constexpr int NIPW = 4;                 // images per direct interpolation workgroup
constexpr int NBOXG = 8;                // images per boxed interpolation workgroup
constexpr int BOXCAP = 1792;            // grid values of a box: 28 KB of LDS, five workgroups a CU

struct NGeo {
    int n, n_r, n_theta, M;  // image side, rays, polar points M = n_r * n_theta/2
    int N, H;                // oversampled grid side, columns kept of it (N/2 + 1)
    int np;                  // pairs of pixel rows, (n + 1)/2
    int x0;                  // g(0) = ceil(-n/2): pixel u sits at x = x0 + u
    int Kc;                  // images in this chunk
};

__device__ inline double es_kernel(double z) {
    return fabs(z) <= 1.0 ? exp(NBETA * (sqrt(1.0 - z * z) - 1.0)) : 0.0;
}

// Per polar point m: the first grid index of its window on each axis and
// the NW kernel weights along it, y (along which b is contiguous) first.  Frequencies as in
// tables_kernel (cryo_pft.m:49-58).
__global__ void nweights_kernel(NGeo g, int2* base, double* wt) {
    const int m = blockIdx.x * blockDim.x + threadIdx.x;
    if (m >= g.M) return;
    const int k = m % g.n_r, j = m / g.n_r;
    const double omega0 = 2.0 * M_PI / (2.0 * g.n_r - 1.0);
    const double dtheta = 2.0 * M_PI / g.n_theta;
    const double fx = (k * omega0) * sin(j * dtheta), fy = (k * omega0) * cos(j * dtheta);
    const double sx = fx * (g.N / (2.0 * M_PI)), sy = fy * (g.N / (2.0 * M_PI));
    const int lx = (int)ceil(sx - 0.5 * NW), ly = (int)ceil(sy - 0.5 * NW);
    base[m] = make_int2(ly, lx);
    double* w = wt + (size_t)m * 2 * NW;
    for (int t = 0; t < NW; t++) {
        w[t] = es_kernel(2.0 * (sy - (ly + t)) / NW);
        w[NW + t] = es_kernel(2.0 * (sx - (lx + t)) / NW);
    }
}

// dec[u] = Phi(x0 + u), the kernel's Fourier transform at the pixel offsets:
// NW/2 sum_q wq[q] cos(pi zq[q] NW x / N) over the NQ quadrature nodes, a wave
// per offset (a lane per node, lanes summed by halves).
constexpr int NQ = 200;
__global__ __launch_bounds__(64) void dec_kernel(NGeo g, const double* __restrict__ zq,
                                                 const double* __restrict__ wq, double* __restrict__ dec) {
    const double x = g.x0 + (int)blockIdx.x;
    double acc = 0.0;
    for (int q = threadIdx.x; q < NQ; q += 64) acc += wq[q] * cos(M_PI * zq[q] * NW * x / g.N);
    for (int s = 32; s; s >>= 1) acc += __shfl_xor(acc, s);
    if (threadIdx.x == 0) dec[blockIdx.x] = 0.5 * NW * acc;
}

// Rows of the chunk's grids that hold pixels, two to a complex row, a[i][v/2][x mod
// N]: p(u, v, k0 + i) / (dec[u] dec[v]) where a pixel sits, zero elsewhere, in the
// real part for even v and the imaginary part for odd.
template <typename T>
__global__ void deconv_kernel(NGeo g, const T* __restrict__ img, long long k0, const double* __restrict__ dec,
                              double2* __restrict__ a) {
    const long long q = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    const long long pN = (long long)g.np * g.N;
    if (q >= pN * g.Kc) return;
    const int i = (int)(q / pN);
    const int r = (int)(q % pN);
    const int v = 2 * (r / g.N), lx = r - (v / 2) * g.N;
    const int xmax = g.x0 + g.n - 1;  // pixel offsets x0..xmax; N >= 2n keeps x and x - N apart
    const int x = lx <= xmax ? lx : lx - g.N;
    double2 val = make_double2(0.0, 0.0);
    if (x >= g.x0) {
        const int u = x - g.x0;
        const size_t at = ((size_t)(k0 + i) * g.n + v) * g.n + u;
        val.x = (double)img[at] / (dec[u] * dec[v]);
        if (v + 1 < g.n) val.y = (double)img[at + g.n] / (dec[u] * dec[v + 1]);
    }
    a[q] = val;
}

// The rows' transforms over x, taken apart (z(x) = row_v(x) + i row_{v+1}(x), both
// Hermitian) and turned to b[i][x][y mod N] (x <= N/2, y contiguous) with zeros in
// the rows that held no pixel, for the transforms over y.  Those rows (half of them
// and more) are neither transformed over x nor read, and b is left turned: the
// interpolation reads it with its axes exchanged.  Tiles of 32 x 32 through LDS.
// For 100 images, N = 720: 62 us (transforms over x) + 115 (this, 663 MB: HBM bound)
// + 147 (over y).  Real-to-complex transforms along x took 70, but a second kernel
// compiled at the first use of each size (2.3 s against 1.2, n = 150).
__global__ __launch_bounds__(256) void turn_kernel(NGeo g, const double2* __restrict__ a, double2* __restrict__ b) {
    __shared__ double2 s_t[32][33];
    const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;
    const int x0 = blockIdx.x * 32, y0 = blockIdx.y * 32;
    const int xmax = g.x0 + g.n - 1;
    const int x = x0 + tx, xm = x ? g.N - x : 0;
    a += (size_t)blockIdx.z * g.np * g.N;
    b += (size_t)blockIdx.z * g.H * g.N;
#pragma unroll
    for (int r = 0; r < 4; r++) {
        const int ly = y0 + ty + 8 * r;
        const int v = (ly <= xmax ? ly : ly - g.N) - g.x0;
        double2 o = make_double2(0.0, 0.0);
        if (ly < g.N && v >= 0 && x < g.H) {
            const double2 z = a[(size_t)(v >> 1) * g.N + x], m = a[(size_t)(v >> 1) * g.N + xm];
            o = v & 1 ? make_double2(0.5 * (z.y + m.y), 0.5 * (m.x - z.x)) : make_double2(0.5 * (z.x + m.x), 0.5 * (z.y - m.y));
        }
        s_t[ty + 8 * r][tx] = o;
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < 4; r++) {
        const int xr = x0 + ty + 8 * r;
        if (xr < g.H && y0 + tx < g.N) b[(size_t)xr * g.N + y0 + tx] = s_t[tx][ty + 8 * r];
    }
}

// Where grid value (x, y mod N) of an image is kept, and whether its conjugate
// is: x is in [-NW/2, N/2 + NW/2], and columns outside 0..N/2 are mirrors.
struct Cell {
    int at;
    bool conj;
};
__device__ inline Cell cell_of(const NGeo& g, int x, int y) {
    y %= g.N;
    if (y < 0) y += g.N;
    const bool mir = x < 0 || x >= g.H;
    if (mir) {
        x = x < 0 ? -x : g.N - x;
        y = y ? g.N - y : 0;
    }
    return Cell{x * g.N + y, mir};
}

// Sum over the 16 lanes of each row (quad_perm [1,0,3,2], [2,3,0,1],
// row_ror 4, row_ror 8): every lane of the row gets it.  All lanes active.
template <int CTRL>
__device__ inline double dpp64(double x) {
    const unsigned long long u = __double_as_longlong(x);
    const int lo = __builtin_amdgcn_update_dpp(0, (int)(u & 0xffffffffu), CTRL, 0xf, 0xf, false);
    const int hi = __builtin_amdgcn_update_dpp(0, (int)(u >> 32), CTRL, 0xf, 0xf, false);
    return __longlong_as_double((long long)(((unsigned long long)(unsigned)hi << 32) | (unsigned)lo));
}
__device__ inline double row16_sum(double x) {
    x += dpp64<0xb1>(x);
    x += dpp64<0x4e>(x);
    x += dpp64<0x124>(x);
    x += dpp64<0x128>(x);
    return x;
}

__device__ inline void put_pf(double2* o, double re, double im) { *o = make_double2(re, im); }
__device__ inline void put_pf(float2* o, double re, double im) { *o = make_float2((float)re, (float)im); }

// pf of the chunk's images at the polar points.  Workgroup: 16 points (4
// per wave, 16 lanes each; lane t = y offset of the window) x NIPW images; each
// lane walks the NW columns of the point's window in order, then the point's 16
// lanes are summed.  pf(k, j) and its conjugate pf(k, j + n_theta/2)
// (cryo_pft.m:75).
template <typename OutT>
__global__ __launch_bounds__(256) void interp_kernel(NGeo g, const double2* __restrict__ b,
                                                     const int2* __restrict__ base, const double* __restrict__ wt,
                                                     OutT* __restrict__ pf, long long k0) {
    __shared__ double s_wx[16][NW];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int t = lane & 15, ps = wave * 4 + (lane >> 4);
    const int m = blockIdx.x * 16 + ps;
    const bool act = m < g.M;
    int2 bs = make_int2(0, 0);
    double wy = 0.0;
    if (act) {
        bs = base[m];
        wy = wt[(size_t)m * 2 * NW + t];
        s_wx[ps][t] = wt[(size_t)m * 2 * NW + NW + t];
    }
    __syncthreads();
    const int L = g.n_theta / 2;
    const int k = act ? m % g.n_r : 0, j = act ? m / g.n_r : 0;
    const size_t HN = (size_t)g.H * g.N;
    for (int ii = 0; ii < NIPW; ii++) {
        const int i = blockIdx.y * NIPW + ii;
        if (i >= g.Kc) break;  // the same for the whole workgroup
        const double2* bi = b + i * HN;
        double re = 0.0, im = 0.0;
        if (act) {
#pragma unroll 4
            for (int r = 0; r < NW; r++) {
                const double w = s_wx[ps][r] * wy;
                const Cell c = cell_of(g, bs.y + r, bs.x + t);
                const double2 v = bi[c.at];
                re = fma(w, v.x, re);
                im = fma(c.conj ? -w : w, v.y, im);
            }
        }
        re = row16_sum(re);
        im = row16_sum(im);
        if (act && t < 2)
            put_pf(pf + ((size_t)(k0 + i) * g.n_theta + j + t * L) * g.n_r + k, re, t ? -im : im);
    }
}

// The same sums, bit for bit, with the windows read from LDS: a workgroup's 16
// points are neighbours on one ray, so their windows lie in one box of the
// grid, which is read once instead of 16 times.  The next image's box is on its
// way into registers while this one is summed; a lane keeps its 16 weights for
// all NBOXG images.  The direct form reads 256 grid values a point and image
// through the vector L1 and is bound there.  383 us for 100 images, n = 359, 180 x
// 180 points: the vector units are busy 69% of it and LDS 65% (a fifth of that on
// bank conflicts).
template <typename OutT>
__global__ __launch_bounds__(256) void interp_box_kernel(NGeo g, const d2* __restrict__ b,
                                                         const int2* __restrict__ base,
                                                         const double* __restrict__ wt, OutT* __restrict__ pf,
                                                         long long k0, int nkb) {
    __shared__ d2 s_box[BOXCAP];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int t = lane & 15, ps = wave * 4 + (lane >> 4);
    const int j = blockIdx.x / nkb, kb = (blockIdx.x - j * nkb) * 16;
    const int k = kb + ps, kl = min(kb + 15, g.n_r - 1);
    const bool act = k < g.n_r;
    // the windows' first indices are monotone along a ray, so its ends bound the box
    const int2 b0 = base[j * g.n_r + kb], b1 = base[j * g.n_r + kl];
    const int y0 = min(b0.x, b1.x), x0 = min(b0.y, b1.y);
    const int W = abs(b1.x - b0.x) + NW, H = abs(b1.y - b0.y) + NW;
    const int cells = min(W * H, BOXCAP);
    const int m = j * g.n_r + min(k, kl);  // lanes past the ray's end repeat its last point
    const int2 bs = base[m];
    const double wy = wt[(size_t)m * 2 * NW + t];
    double w[NW];
#pragma unroll
    for (int r = 0; r < NW; r++) w[r] = wt[(size_t)m * 2 * NW + NW + r] * wy;
    const int at = (bs.y - x0) * W + bs.x - y0 + t;
    constexpr int NC = (BOXCAP + 255) / 256;  // cells per thread
    unsigned off[NC];                         // bytes into a grid (below 2^32: N <= 4096)
    unsigned conj = 0;                        // bit q: cell q is a mirror
#pragma unroll
    for (int q = 0; q < NC; q++) {
        const int c = min((int)threadIdx.x + q * 256, cells - 1);
        const int r = c / W;
        const Cell o = cell_of(g, x0 + r, y0 + c - r * W);
        off[q] = o.at * (unsigned)sizeof(d2);
        conj |= (unsigned)o.conj << q;
    }
    const size_t HN = (size_t)g.H * g.N;
    const int i0 = blockIdx.y * NBOXG, i1 = min(i0 + NBOXG, g.Kc);
    const char* bc = (const char*)(b + i0 * HN);
    const int L = g.n_theta / 2;
    d2 nx[NC];
#pragma unroll
    for (int q = 0; q < NC; q++)
        if (q * 256 < cells) nx[q] = *(const d2*)(bc + off[q]);
    for (int i = i0; i < i1; i++) {
        __syncthreads();  // the last box is no longer read
#pragma unroll
        for (int q = 0; q < NC; q++)
            if ((int)threadIdx.x + q * 256 < cells) {
                if (conj >> q & 1) nx[q].y = -nx[q].y;
                s_box[threadIdx.x + q * 256] = nx[q];
            }
        __syncthreads();
        if (i + 1 < i1) {
            bc += HN * sizeof(d2);
#pragma unroll
            for (int q = 0; q < NC; q++)
                if (q * 256 < cells) nx[q] = *(const d2*)(bc + off[q]);
        }
        double re = 0.0, im = 0.0;
#pragma unroll
        for (int r = 0; r < NW; r++) {
            const d2 v = s_box[at + r * W];
            re = fma(w[r], v.x, re);
            im = fma(w[r], v.y, im);
        }
        re = row16_sum(re);
        im = row16_sum(im);
        if (act && t < 2)
            put_pf(pf + ((size_t)(k0 + i) * g.n_theta + j + t * L) * g.n_r + k, re, t ? -im : im);
    }
}

}  // namespace pft

using namespace clmh;

namespace {

int pft_check(clm_ctx* c, const clm_pft_params* p) {
    if (!p) return fail(c, CLM_E_ARG, "null params");
    if (p->n_theta <= 0 || p->n_theta % 2) return fail(c, CLM_E_ARG, "`n_theta` must be even.");
    if (p->n < 1 || p->n > 4096) return fail(c, CLM_E_UNSUP, "image side n = %d out of range [1, 4096]", p->n);
    if (p->n_r < 1 || p->K < 0) return fail(c, CLM_E_ARG, "invalid n_r = %d or K = %d", p->n_r, p->K);
    if ((long long)p->n_r * (p->n_theta / 2) > (1LL << 26))
        return fail(c, CLM_E_UNSUP, "n_r * n_theta/2 = %lld polar points exceeds 2^26",
                    (long long)p->n_r * (p->n_theta / 2));
    if (p->img_dtype != CLM_R64 && p->img_dtype != CLM_R32)
        return fail(c, CLM_E_ARG, "unknown image dtype %d", p->img_dtype);
    if (p->pf_dtype != CLM_C128 && p->pf_dtype != CLM_C64) return fail(c, CLM_E_ARG, "unknown pf dtype %d", p->pf_dtype);
    if (p->method != CLM_PFT_EXACT && p->method != CLM_PFT_NUFFT)
        return fail(c, CLM_E_ARG, "unknown pft method %d", p->method);
    if (p->method == CLM_PFT_NUFFT && p->n > 2048)
        return fail(c, CLM_E_UNSUP, "image side n = %d: the NUFFT method takes n <= 2048", p->n);
    return CLM_OK;
}

int pft_run(clm_ctx* c, const clm_pft_params* p, const void* d_img, void* d_pf, clm_pft_stats* st) {
    using namespace pft;
    Geo g{};
    g.n = p->n;
    g.n_r = p->n_r;
    g.n_theta = p->n_theta;
    g.M = p->n_r * (p->n_theta / 4 + 1);
    g.Mp = (g.M + 63) / 64 * 64;  // whole blocks of the tallest tile
    g.c = p->n / 2;
    g.nh = p->n / 2 + 1;
    g.nab = (g.nh + 3) / 4;
    const int K = p->K;
    const int kc = K < KCHUNK ? K : KCHUNK;
    int rc;
    g.nb8 = (g.nh + 7) / 8;
    // the mirror rays' shifts: 3e-14, nothing to a result in single precision
    const bool c128 = p->pf_dtype == CLM_C128, shifted = c128 && p->n_theta > 4;
    const int nct = (kc + 15) / 16, nfold = (4 * g.nab + FA - 1) / FA;
    const size_t ntab = (size_t)16 * g.nab * g.Mp, nxt = (size_t)nct * 4 * g.nab * g.nh * 64;
    const size_t npart = (size_t)nct * g.nh * nfold * 16;  // then 16 nct for top
    const size_t ndx = shifted ? (size_t)8 * g.nab * g.Mp : 0, ndy = shifted ? (size_t)32 * g.nb8 * g.Mp : 0;
    const size_t nxh = shifted ? (size_t)nct * 4 * g.nab * g.nb8 * 64 : 0, nsh = shifted ? (size_t)kc * g.Mp : 0;
    if ((rc = ensure(c, c->pft_ax, ntab * sizeof(double) + ndx * sizeof(h2) + ndy * sizeof(_Float16))) ||
        (rc = ensure(c, c->pft_xt, nxt * sizeof(double) + nxh * sizeof(h8) + nsh * sizeof(float2) +
                                       (npart + 16 * nct) * sizeof(unsigned))))
        return rc;
    const int L = g.n_theta / 2;
    if (c->pft_ray_T != g.n_theta) {
        // the rays' sines and cosines, as clm_pft_freqs returns them
        std::vector<double> h(2 * (size_t)L);
        const double dtheta = 2.0 * M_PI / g.n_theta;  // cryo_pft.m:50
        for (int j = 0; j < L; j++) {
            h[j] = sin(j * dtheta);
            h[L + j] = cos(j * dtheta);
        }
        c->pft_ray_T = 0;
        if ((rc = ensure(c, c->pft_ray, h.size() * sizeof(double)))) return rc;
        HIPCHK(c, hipMemcpyAsync(c->pft_ray.p, h.data(), h.size() * sizeof(double), hipMemcpyHostToDevice, c->stream));
        HIPCHK(c, hipStreamSynchronize(c->stream));  // h is released on return
        c->pft_ray_T = g.n_theta;
    }
    hipEvent_t* ev = c->ev;
    double* tab = (double*)c->pft_ax.p;
    h2* dx = shifted ? (h2*)(tab + ntab) : nullptr;
    _Float16* dy = (_Float16*)(dx + ndx);
    double* xt = (double*)c->pft_xt.p;
    h8* xh = (h8*)(xt + nxt);
    float2* shift = shifted ? (float2*)(xh + nxh) : nullptr;
    unsigned* part = (unsigned*)((float2*)(xh + nxh) + nsh);
    unsigned* top = part + npart;
    HIPCHK(c, hipEventRecord(ev[0], c->stream));
    tables_kernel<<<dim3((g.Mp + 255) / 256, 8 * g.nab), 256, 0, c->stream>>>(
        g, (const double*)c->pft_ray.p, tab, dx, dy);
    HIPCHK(c, hipGetLastError());
    HIPCHK(c, hipEventRecord(ev[1], c->stream));
    float ms_stage = 0.f, ms_pft = 0.f;
    int chunks = 0;
    for (long long k0 = 0; k0 < K; k0 += KCHUNK) {
        g.Kc = (int)((K - k0) < KCHUNK ? (K - k0) : KCHUNK);
        g.nct = (g.Kc + 15) / 16;
        const dim3 fgrid(nfold, g.nh, g.nct);
        HIPCHK(c, hipEventRecord(ev[2], c->stream));
        if (p->img_dtype == CLM_R64)
            fold_kernel<double><<<fgrid, 256, 0, c->stream>>>(g, (const double*)d_img, k0, xt, part);
        else
            fold_kernel<float><<<fgrid, 256, 0, c->stream>>>(g, (const float*)d_img, k0, xt, part);
        HIPCHK(c, hipGetLastError());
        top_kernel<<<g.nct, 256, 0, c->stream>>>(g, part, g.nh * nfold, top);
        HIPCHK(c, hipEventRecord(ev[3], c->stream));
        if (shifted) {
            narrow_kernel<<<dim3(g.nab, 4, g.nct), 256, 0, c->stream>>>(g, xt, top, xh);
            // small tiles while three a CU hold all of them (one image: 25 us
            // against 51; 100: 72 against 57)
            const long long small = (long long)((g.M + 31) / 32) * g.nct;
            if (small <= 3LL * c->n_cu) shift_launch<2, 1, 4>(c->stream, g, xh, dx, dy, shift);
            else shift_launch<4, 4, 2>(c->stream, g, xh, dx, dy, shift);
            HIPCHK(c, hipGetLastError());
        }
        // the tile whose busiest CU has the fewest cycles: 64 per MFMA, and
        // about 24 per operand load of a step
        const int rts[] = {4, 2, 1, 1}, cts[] = {4, 4, 4, 1};
        int best = 0;
        double cost = 0;
        for (int q = 0; q < 4; q++) {
            const long long tiles = (long long)((g.M + 16 * rts[q] - 1) / (16 * rts[q])) * ((g.nct + cts[q] - 1) / cts[q]);
            const double cq = (double)((tiles + c->n_cu - 1) / c->n_cu) * (64 * rts[q] * cts[q] + 24 * (rts[q] + cts[q]));
            if (q == 0 || cq < cost) {
                cost = cq;
                best = q;
            }
        }
        if (best == 0) pft_launch<4, 4>(c->stream, g, c128, xt, tab, shift, top, d_pf, k0);
        else if (best == 1) pft_launch<2, 4>(c->stream, g, c128, xt, tab, shift, top, d_pf, k0);
        else if (best == 2) pft_launch<1, 4>(c->stream, g, c128, xt, tab, shift, top, d_pf, k0);
        else pft_launch<1, 1>(c->stream, g, c128, xt, tab, shift, top, d_pf, k0);
        HIPCHK(c, hipGetLastError());
        if (p->img_dtype == CLM_R64) non_finite_launch(c->stream, g, c128, (const double*)d_img, k0, top, d_pf);
        else non_finite_launch(c->stream, g, c128, (const float*)d_img, k0, top, d_pf);
        HIPCHK(c, hipGetLastError());
        HIPCHK(c, hipEventRecord(ev[4], c->stream));
        HIPCHK(c, hipEventSynchronize(ev[4]));
        float a = 0.f, b = 0.f;
        HIPCHK(c, hipEventElapsedTime(&a, ev[2], ev[3]));
        HIPCHK(c, hipEventElapsedTime(&b, ev[3], ev[4]));
        ms_stage += a;
        ms_pft += b;
        chunks++;
    }
    HIPCHK(c, hipStreamSynchronize(c->stream));
    if (st) {
        float t = 0.f;
        HIPCHK(c, hipEventElapsedTime(&t, ev[0], ev[1]));
        st->ms_tables = t;
        st->ms_stage = ms_stage;
        st->ms_pft = ms_pft;
        st->chunks = chunks;
    }
    return CLM_OK;
}

// ------------------------------------------------------------ type-2 NUFFT
// Gauss-Legendre rule of q nodes on [-1, 1]: roots of P_q by Newton's method
// (P_q from the three-term recurrence), weights 2 / ((1 - z^2) P_q'(z)^2).
void gauss_legendre(int q, std::vector<double>& x, std::vector<double>& w) {
    x.assign(q, 0.0);
    w.assign(q, 0.0);
    for (int i = 0; i < (q + 1) / 2; i++) {
        double z = std::cos(M_PI * (i + 0.75) / (q + 0.5)), dp = 1.0;
        for (int it = 0; it < 100; it++) {
            double p1 = 1.0, p0 = 0.0;
            for (int jj = 1; jj <= q; jj++) {
                const double pm = p0;
                p0 = p1;
                p1 = ((2.0 * jj - 1.0) * z * p0 - (jj - 1.0) * pm) / jj;
            }
            dp = q * (z * p1 - p0) / (z * z - 1.0);
            const double dz = p1 / dp;
            z -= dz;
            if (std::fabs(dz) < 1e-16) break;
        }
        x[i] = -z;
        x[q - 1 - i] = z;
        w[i] = w[q - 1 - i] = 2.0 / ((1.0 - z * z) * dp * dp);
    }
}

// Nodes z of the kernel's quadrature, then their weights times phi(z): NQ
// each, formed once.
const std::vector<double>& kernel_nodes() {
    static const std::vector<double> nodes = [] {
        std::vector<double> z, w;
        gauss_legendre(pft::NQ, z, w);
        for (int q = 0; q < pft::NQ; q++) z.push_back(w[q] * std::exp(pft::NBETA * (std::sqrt(1.0 - z[q] * z[q]) - 1.0)));
        return z;
    }();
    return nodes;
}

// Smallest 2^a 3^b 5^c >= n.
int smooth_at_least(int n) {
    for (int m = n;; m++) {
        int r = m;
        for (int f : {2, 3, 5})
            while (r % f == 0) r /= f;
        if (r == 1) return m;
    }
}

// Plan of `batch` contiguous transforms of N points; the context keeps the
// FFT_PLANS last used (two a shape), most recent first.
hipfftHandle fft_plan(clm_ctx* c, int N, int batch, int* rc) {
    constexpr int S = clm_ctx::FFT_PLANS;
    int s = 0;
    while (s < S && !(c->fft_plan[s] && c->fft_side[s] == N && c->fft_batch[s] == batch)) s++;
    hipfftHandle h = nullptr;
    if (s < S) {
        h = (hipfftHandle)c->fft_plan[s];
    } else {
        hipfftResult r = hipfftPlan1d(&h, N, HIPFFT_Z2Z, batch);
        if (r == HIPFFT_SUCCESS) r = hipfftSetStream(h, c->stream);
        if (r != HIPFFT_SUCCESS) {
            if (h) (void)hipfftDestroy(h);
            *rc = fail(c, CLM_E_HIP, "hipFFT plan of %d x %d failed (hipfftResult %d)", N, batch, (int)r);
            return nullptr;
        }
        s = S - 1;
        if (c->fft_plan[s]) (void)hipfftDestroy((hipfftHandle)c->fft_plan[s]);
    }
    for (; s > 0; s--) {
        c->fft_plan[s] = c->fft_plan[s - 1];
        c->fft_side[s] = c->fft_side[s - 1];
        c->fft_batch[s] = c->fft_batch[s - 1];
    }
    c->fft_plan[0] = (void*)h;
    c->fft_side[0] = N;
    c->fft_batch[0] = batch;
    return h;
}

int nufft_run(clm_ctx* c, const clm_pft_params* p, const void* d_img, void* d_pf, clm_pft_stats* st) {
    using namespace pft;
    NGeo g{};
    g.n = p->n;
    g.n_r = p->n_r;
    g.n_theta = p->n_theta;
    g.M = p->n_r * (p->n_theta / 2);
    g.N = smooth_at_least(std::max(2 * p->n, 2 * NW));
    g.H = g.N / 2 + 1;
    g.np = (p->n + 1) / 2;
    g.x0 = (int)std::ceil(-0.5 * p->n);
    const int K = p->K;
    const size_t NN = (size_t)g.N * g.N;
    // images per batch: at most NCHUNK, and grids of at most 4 GiB
    const int kc = (int)std::max<long long>(1, std::min<long long>({(long long)K, (long long)NCHUNK,
                                                                     (4LL << 30) / (long long)(NN * sizeof(double2))}));
    // boxed interpolation where the box of 16 points of a ray fits: its sides
    // are at most 15 steps of N / (2 n_r - 1) times the ray's |sin| and |cos|,
    // plus 18, and their product is largest on the diagonal.  That is where n_r
    // is about n/2 or more; sparser points share too little of their windows.
    const double side = 15.0 * g.N / (2.0 * g.n_r - 1.0) * M_SQRT1_2 + NW + 2;
    const bool boxed = side * side <= BOXCAP;
    int rc;
    // the grids' half columns, the pairs of rows
    if ((rc = ensure(c, c->pft_grid, (size_t)kc * g.H * g.N * sizeof(double2))) ||
        (rc = ensure(c, c->pft_xt, (size_t)kc * g.np * g.N * sizeof(double2))) ||
        (rc = ensure(c, c->pft_base, (size_t)g.M * sizeof(int2))) ||
        (rc = ensure(c, c->pft_wt, (size_t)g.M * 2 * NW * sizeof(double))) ||
        (rc = ensure(c, c->pft_dec, (size_t)(g.n + 2 * NQ) * sizeof(double))))
        return rc;
    hipEvent_t* ev = c->ev;
    HIPCHK(c, hipEventRecord(ev[0], c->stream));
    // deconvolution factors Phi(x0 + u), u < n, from the quadrature nodes
    const std::vector<double>& nodes = kernel_nodes();
    double* dec = (double*)c->pft_dec.p;
    double* dnodes = dec + g.n;
    HIPCHK(c, hipMemcpyAsync(dnodes, nodes.data(), nodes.size() * sizeof(double), hipMemcpyHostToDevice, c->stream));
    dec_kernel<<<g.n, 64, 0, c->stream>>>(g, dnodes, dnodes + NQ, dec);
    HIPCHK(c, hipGetLastError());
    nweights_kernel<<<(g.M + 255) / 256, 256, 0, c->stream>>>(g, (int2*)c->pft_base.p, (double*)c->pft_wt.p);
    HIPCHK(c, hipGetLastError());
    HIPCHK(c, hipEventRecord(ev[1], c->stream));
    float ms_stage = 0.f, ms_fft = 0.f, ms_pft = 0.f;
    int chunks = 0;
    double2* grid = (double2*)c->pft_grid.p;
    double2* rows = (double2*)c->pft_xt.p;
    for (long long k0 = 0; k0 < K; k0 += kc) {
        g.Kc = (int)((K - k0) < kc ? (K - k0) : kc);
        hipfftHandle plan_x = fft_plan(c, g.N, g.np * g.Kc, &rc);
        hipfftHandle plan_y = plan_x ? fft_plan(c, g.N, g.H * g.Kc, &rc) : nullptr;
        if (!plan_y) return rc;
        HIPCHK(c, hipEventRecord(ev[2], c->stream));
        const long long nq = (long long)g.np * g.N * g.Kc;
        const unsigned dgrd = (unsigned)((nq + 255) / 256);
        if (p->img_dtype == CLM_R64)
            deconv_kernel<double><<<dgrd, 256, 0, c->stream>>>(g, (const double*)d_img, k0, dec, rows);
        else
            deconv_kernel<float><<<dgrd, 256, 0, c->stream>>>(g, (const float*)d_img, k0, dec, rows);
        HIPCHK(c, hipGetLastError());
        HIPCHK(c, hipEventRecord(ev[3], c->stream));
        hipfftDoubleComplex *fx = (hipfftDoubleComplex*)rows, *fy = (hipfftDoubleComplex*)grid;
        hipfftResult fr = hipfftExecZ2Z(plan_x, fx, fx, HIPFFT_BACKWARD);
        if (fr == HIPFFT_SUCCESS) {
            const dim3 tgrd((g.H + 31) / 32, (g.N + 31) / 32, g.Kc);
            turn_kernel<<<tgrd, 256, 0, c->stream>>>(g, rows, grid);
            HIPCHK(c, hipGetLastError());
            fr = hipfftExecZ2Z(plan_y, fy, fy, HIPFFT_BACKWARD);
        }
        if (fr != HIPFFT_SUCCESS) return fail(c, CLM_E_HIP, "hipFFT transform failed (hipfftResult %d)", (int)fr);
        HIPCHK(c, hipEventRecord(ev[4], c->stream));
        const int2* base = (const int2*)c->pft_base.p;
        const double* wt = (const double*)c->pft_wt.p;
        if (boxed) {
            const int nkb = (g.n_r + 15) / 16;
            const dim3 igrid((g.n_theta / 2) * nkb, (g.Kc + NBOXG - 1) / NBOXG);
            if (p->pf_dtype == CLM_C128)
                interp_box_kernel<double2><<<igrid, 256, 0, c->stream>>>(g, (const d2*)grid, base, wt, (double2*)d_pf, k0, nkb);
            else
                interp_box_kernel<float2><<<igrid, 256, 0, c->stream>>>(g, (const d2*)grid, base, wt, (float2*)d_pf, k0, nkb);
        } else {
            const dim3 igrid((g.M + 15) / 16, (g.Kc + NIPW - 1) / NIPW);
            if (p->pf_dtype == CLM_C128)
                interp_kernel<double2><<<igrid, 256, 0, c->stream>>>(g, grid, base, wt, (double2*)d_pf, k0);
            else
                interp_kernel<float2><<<igrid, 256, 0, c->stream>>>(g, grid, base, wt, (float2*)d_pf, k0);
        }
        HIPCHK(c, hipGetLastError());
        HIPCHK(c, hipEventRecord(ev[5], c->stream));
        HIPCHK(c, hipEventSynchronize(ev[5]));
        float a = 0.f, b = 0.f, d = 0.f;
        HIPCHK(c, hipEventElapsedTime(&a, ev[2], ev[3]));
        HIPCHK(c, hipEventElapsedTime(&b, ev[3], ev[4]));
        HIPCHK(c, hipEventElapsedTime(&d, ev[4], ev[5]));
        ms_stage += a;
        ms_fft += b;
        ms_pft += d;
        chunks++;
    }
    HIPCHK(c, hipStreamSynchronize(c->stream));
    if (st) {
        float t = 0.f;
        HIPCHK(c, hipEventElapsedTime(&t, ev[0], ev[1]));
        st->ms_tables = t;
        st->ms_stage = ms_stage;
        st->ms_fft = ms_fft;
        st->ms_pft = ms_pft;
        st->chunks = chunks;
        st->grid_side = g.N;
    }
    return CLM_OK;
}

int pft_dispatch(clm_ctx* c, const clm_pft_params* p, const void* d_img, void* d_pf, clm_pft_stats* st) {
    return p->method == CLM_PFT_NUFFT ? nufft_run(c, p, d_img, d_pf, st) : pft_run(c, p, d_img, d_pf, st);
}

}  // namespace

namespace clmh {
void pft_release(clm_ctx* c) {
    for (int s = 0; s < clm_ctx::FFT_PLANS; s++) {
        if (c->fft_plan[s]) (void)hipfftDestroy((hipfftHandle)c->fft_plan[s]);
        c->fft_plan[s] = nullptr;
        c->fft_side[s] = c->fft_batch[s] = 0;
    }
}
}  // namespace clmh

extern "C" {

int clm_pft_freqs(int32_t n_r, int32_t n_theta, double* freqs) {
    if (n_r < 1 || n_theta <= 0 || n_theta % 2 || !freqs) return CLM_E_ARG;
    const int L = n_theta / 2;
    const size_t M = (size_t)n_r * L;
    const double omega0 = 2.0 * M_PI / (2.0 * n_r - 1.0);
    const double dtheta = 2.0 * M_PI / n_theta;
    for (int j = 0; j < L; j++) {
        const double sn = sin(j * dtheta), cs = cos(j * dtheta);
        for (int k = 0; k < n_r; k++) {
            const size_t m = (size_t)j * n_r + k;
            freqs[m] = (k * omega0) * sn;
            freqs[M + m] = (k * omega0) * cs;
        }
    }
    return CLM_OK;
}

int clm_pft_device(clm_ctx* c, const clm_pft_params* p, const void* d_img, void* d_pf, clm_pft_stats* st) {
    if (!c) return CLM_E_ARG;
    int rc = pft_check(c, p);
    if (rc) return rc;
    if (st) *st = clm_pft_stats{};
    if (p->K == 0) return CLM_OK;
    if (!d_img || !d_pf) return fail(c, CLM_E_ARG, "null image or pf pointer");
    HIPCHK(c, hipSetDevice(c->device));
    return pft_dispatch(c, p, d_img, d_pf, st);
}

int clm_pft(clm_ctx* c, const clm_pft_params* p, const void* img, void* pf, clm_pft_stats* st) {
    if (!c) return CLM_E_ARG;
    int rc = pft_check(c, p);
    if (rc) return rc;
    if (st) *st = clm_pft_stats{};
    if (p->K == 0) return CLM_OK;
    if (!img || !pf) return fail(c, CLM_E_ARG, "null image or pf pointer");
    HIPCHK(c, hipSetDevice(c->device));
    const size_t nimg = (size_t)p->n * p->n * p->K * (p->img_dtype == CLM_R64 ? 8 : 4);
    const size_t npf = (size_t)p->n_r * p->n_theta * p->K * (p->pf_dtype == CLM_C128 ? 16 : 8);
    if ((rc = ensure(c, c->pft_img, nimg)) || (rc = ensure(c, c->pft_out, npf))) return rc;
    HIPCHK(c, hipMemcpyAsync(c->pft_img.p, img, nimg, hipMemcpyHostToDevice, c->stream));
    if ((rc = pft_dispatch(c, p, c->pft_img.p, c->pft_out.p, st))) return rc;
    HIPCHK(c, hipMemcpyAsync(pf, c->pft_out.p, npf, hipMemcpyDeviceToHost, c->stream));
    HIPCHK(c, hipStreamSynchronize(c->stream));
    return CLM_OK;
}

}  // extern "C"
