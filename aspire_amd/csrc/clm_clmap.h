// clm_clmap.h -- the common-lines search with map_filter_radius > 0
// (cryo_clmatrix_cpu.m:383-385): every shift's correlation map is filtered
// by cryo_average_clmap (sinograms/cryo_average_clmap.m:20-48) before the
// first-maximum search, and the filtered value is what the pair keeps.
//
// The filter replaces each entry by a weighted sum over its (2d+1)^2
// neighbourhood in the map extended to 2L rows (rows L..2L-1 repeat the map
// with its column halves swapped, :30), circularly:
//   out(l1, c) = sum_{i,j=0..2d} W(i,j) map_ext((l1-d+i) mod 2L, (c-d+j) mod 2L)
// A neighbourhood sum cannot be bounded from one cell's maximum, so this
// path does not use the 16-bit engine's pruning: it evaluates every map entry
// in FP64.  clmap64_kernel does so on the FP64 matrix cores and keeps the
// candidates within the rounding of the maximum, which are then evaluated
// with the oracle's arithmetic and order (every tap's sum, then the taps in
// order); clmap_kernel evaluates every entry that way, for the pairs with more
// such candidates than a list holds.  Either way the results equal the FP64
// oracle's bit for bit.
//
// clmap_kernel: one workgroup per listed pair (persistent over pairs).  Per
// shift, the map is computed in 48 x 80 tiles of the extended map (output
// tiles of (48 - 2d) x (80 - 2d) with their halo), r in chunks of 32 staged in
// LDS: each thread owns a 4 x 4 block of the tile.  map_ext(r', c) is
// C_{h(r') xor h(c)}(r' mod L, c mod L) with h(x) = x >= L, so the row
// operand is P1 .* ph or conj(P1) .* ph by that parity.
#pragma once
#include "clm_search64.h"

namespace clm {

constexpr int CM_R = 48, CM_C = 80, CM_RC = 32;

struct ClmapArgs {
    const StackDev* stacks;
    const SlotRef* list;  // the pairs to evaluate
    const int* n_dev;     // their number
};

__global__ __launch_bounds__(256) void clmap_kernel(ClmapArgs a) {
    __shared__ double2 sA[CM_R][CM_RC];   // P1 .* ph
    __shared__ double2 sF[CM_R][CM_RC];   // conj(P1) .* ph
    __shared__ double2 sB[CM_C][CM_RC];   // P2
    __shared__ double sM[CM_R][CM_C + 1];  // map tile
    __shared__ double s_v[256];
    __shared__ long long s_k[256];
    const int tid = threadIdx.x;
    const int bi = tid / 20, bj = tid % 20;  // 12 x 20 blocks of 4 x 4 (threads 240..255 idle)
    const int n_list = *a.n_dev;
    for (int item = blockIdx.x; item < n_list; item += gridDim.x) {
        const StackDev& sd = a.stacks[a.list[item].stack];
        const Geom& g = sd.g;
        const int slot = a.list[item].slot;
        int k1, k2;
        slot_to_pair(slot, g.K, k1, k2);
        const int L = g.L, L2 = 2 * L, R = g.R, d = sd.filt, w = 2 * d + 1;
        const int OR = CM_R - 2 * d, OC = CM_C - 2 * d;
        const double2* P1 = sd.P64 + (size_t)k1 * L * R;
        const double2* P2 = sd.P64 + (size_t)k2 * L * R;
        double bv = -INFINITY;
        long long bk = 0x7fffffffffffffffLL;
        for (int j = 0; j < g.S; j++) {
            const double2* ph = sd.ph64 + (size_t)j * R;
            for (int row0 = 0; row0 < L; row0 += OR) {
                for (int col0 = 0; col0 < L2; col0 += OC) {
                    double acc[4][4];
#pragma unroll
                    for (int x = 0; x < 4; x++)
#pragma unroll
                        for (int y = 0; y < 4; y++) acc[x][y] = 0.0;
                    // parity of each owned entry: flipped row operand?
                    bool flip[4][4];
#pragma unroll
                    for (int x = 0; x < 4; x++) {
                        const int rp = ((row0 - d + 4 * bi + x) % L2 + L2) % L2;
#pragma unroll
                        for (int y = 0; y < 4; y++) {
                            const int cc = ((col0 - d + 4 * bj + y) % L2 + L2) % L2;
                            flip[x][y] = (rp >= L) != (cc >= L);
                        }
                    }
                    for (int r0 = 0; r0 < R; r0 += CM_RC) {
                        const int nr = R - r0 < CM_RC ? R - r0 : CM_RC;
                        __syncthreads();
                        for (int q = tid; q < CM_R * CM_RC; q += 256) {
                            const int ti = q / CM_RC, rr = q % CM_RC;
                            if (rr < nr) {
                                const int rp = ((row0 - d + ti) % L2 + L2) % L2;
                                const double2 p = P1[(size_t)(rp % L) * R + r0 + rr];
                                const double2 f = ph[r0 + rr];
                                sA[ti][rr] = make_double2(p.x * f.x - p.y * f.y, p.x * f.y + p.y * f.x);
                                sF[ti][rr] = make_double2(p.x * f.x + p.y * f.y, p.x * f.y - p.y * f.x);
                            }
                        }
                        for (int q = tid; q < CM_C * CM_RC; q += 256) {
                            const int tj = q / CM_RC, rr = q % CM_RC;
                            if (rr < nr) {
                                const int cc = ((col0 - d + tj) % L2 + L2) % L2;
                                sB[tj][rr] = P2[(size_t)(cc % L) * R + r0 + rr];
                            }
                        }
                        __syncthreads();
                        if (tid < 240) {
                            for (int rr = 0; rr < nr; rr++) {
                                double2 xa[4], xf[4], xb[4];
#pragma unroll
                                for (int x = 0; x < 4; x++) {
                                    xa[x] = sA[4 * bi + x][rr];
                                    xf[x] = sF[4 * bi + x][rr];
                                    xb[x] = sB[4 * bj + x][rr];
                                }
#pragma unroll
                                for (int x = 0; x < 4; x++)
#pragma unroll
                                    for (int y = 0; y < 4; y++) {
                                        const double2 o = flip[x][y] ? xf[x] : xa[x];
                                        const double t = o.x * xb[y].x;
                                        const double u = o.y * xb[y].y;
                                        acc[x][y] = acc[x][y] + (t + u);
                                    }
                            }
                        }
                    }
                    __syncthreads();
                    if (tid < 240) {
#pragma unroll
                        for (int x = 0; x < 4; x++)
#pragma unroll
                            for (int y = 0; y < 4; y++) sM[4 * bi + x][4 * bj + y] = 2.0 * acc[x][y];
                    }
                    __syncthreads();
                    // stencil over this tile's outputs
                    for (int o = tid; o < OR * OC; o += 256) {
                        const int oi = o / OC, oj = o % OC;
                        const int l1 = row0 + oi, c = col0 + oj;
                        if (l1 >= L || c >= L2) continue;
                        double v = 0.0;
                        for (int i = 0; i < w; i++)
                            for (int jx = 0; jx < w; jx++) v = v + sd.wts[i * w + jx] * sM[oi + i][oj + jx];
                        if (isnan(v)) continue;
                        const long long key = tie_key(j, c, l1);
                        if (better64(v, key, bv, bk)) {
                            bv = v;
                            bk = key;
                        }
                    }
                }
            }
        }
        // block-wide best (value, then smallest key)
        s_v[tid] = bv;
        s_k[tid] = bk;
        __syncthreads();
        for (int s = 128; s > 0; s >>= 1) {
            if (tid < s && better64(s_v[tid + s], s_k[tid + s], s_v[tid], s_k[tid])) {
                s_v[tid] = s_v[tid + s];
                s_k[tid] = s_k[tid + s];
            }
            __syncthreads();
        }
        if (tid == 0) write_result(sd, slot, s_v[0], s_k[0]);
        __syncthreads();
    }
}

// ------------------------------------------------ on the FP64 matrix cores
constexpr int CF_T = 64;       // extended tile side: CF_T - 2d outputs and a halo
constexpr int CF_LD = CF_T + 2;  // doubles per row of the tile in LDS
constexpr int CF_MAXW = 21;    // taps per side at the largest radius

inline size_t clmap64_lds() {
    return (size_t)2 * CF_T * CF_LD * 8 + (size_t)4 * S64_LIST * 16 + 2 * CF_MAXW * 8 + 128;
}

// The filtered value at tie key `key` with the oracle's arithmetic and order:
// a lane per tap adds the R terms, then the taps are added in order.  Called
// by the whole wave; taps: (2d+1)^2 doubles of LDS of its own.
__device__ inline double eval_filtered(const StackDev& sd, int k1, int k2, long long key, double* taps, int lane) {
    const Geom& g = sd.g;
    const int L = g.L, L2 = 2 * L, R = g.R, d = sd.filt, w = 2 * d + 1;
    const int l1 = key_l1(key), c = key_l2p(key);
    const double2* P1 = sd.P64 + (size_t)k1 * L * R;
    const double2* P2 = sd.P64 + (size_t)k2 * L * R;
    const double2* ph = sd.ph64 + (size_t)key_j(key) * R;
    for (int t = lane; t < w * w; t += 64) {
        const int i = t / w, jx = t - i * w;
        const int rp = ((l1 - d + i) % L2 + L2) % L2, cc = ((c - d + jx) % L2 + L2) % L2;
        const bool flip = (rp >= L) != (cc >= L);
        const double2* p = P1 + (size_t)(rp >= L ? rp - L : rp) * R;
        const double2* b = P2 + (size_t)(cc >= L ? cc - L : cc) * R;
        double acc = 0.0;
#pragma unroll 4
        for (int r = 0; r < R; r++) acc = acc + term64(p[r], ph[r], b[r], flip);
        taps[t] = 2.0 * acc;
    }
    __builtin_amdgcn_wave_barrier();
    double v = 0.0;
    for (int t = 0; t < w * w; t++) v = v + sd.wts[t] * taps[t];
    __builtin_amdgcn_wave_barrier();
    return v;
}

// One workgroup per pair (and range of units), a unit being one shift on one
// tile of CF_T x CF_T lines (l1, l2) with a halo of d, both halves C1 and C2 at
// once: a row or column beyond the map is a line of the other half, so the
// halo needs no other columns.  Wave w computes rows 16 w..16 w + 15 against
// four column tiles, operands straight from the rays in the MFMA's layout; the
// two maps go to LDS, the weights 1.25^-(|i| + |j|) are applied along the
// columns (into registers, and back) and then along the rows.
// The values differ from the oracle's by at most E = sum(W) n1 n2 2^-53 times
// the two evaluations' numbers of roundings; what is within 2 E of the maximum
// is listed per wave and evaluated again (eval_filtered).
// Bound: FP64 issue, the matrix products a third of the time and the stencil
// and its LDS reads the rest.  1.8 ms for 4950 pairs at n_r = 33, n_theta =
// 360, one shift, d = 1; clmap_kernel, which forms every entry on the vector
// units, takes 12.8 ms.
__global__ __launch_bounds__(256, 2) void clmap64_kernel(Search64Args a) {
    extern __shared__ __align__(16) char s_mem[];
    double* s_T = (double*)s_mem;                       // [2][CF_T][CF_LD]
    double* s_v = s_T + 2 * CF_T * CF_LD;               // [4][S64_LIST]
    long long* s_k = (long long*)(s_v + 4 * S64_LIST);  // [4][S64_LIST]
    double* s_w = (double*)(s_k + 4 * S64_LIST);        // [2][CF_MAXW] weights along the rows, the columns
    double* s_rv = s_w + 2 * CF_MAXW;
    long long* s_rk = (long long*)(s_rv + 4);
    int* s_lost = (int*)(s_rk + 4);
    int* s_stop = s_lost + 4;  // a wave has stopped (CandList)
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r16 = lane & 15, kq = lane >> 4;
    CandList cl{s_v + wave * S64_LIST, s_k + wave * S64_LIST};
    const long long n = a.x.n_all < a.x.item0 + a.x.item_cap ? a.x.n_all : a.x.item0 + a.x.item_cap;
    for (long long it = a.x.item0 + blockIdx.x; it < n; it += gridDim.x) {
        int stk, slot;
        exact_item(a.x, it, stk, slot);
        const StackDev& sd = a.x.stacks[__builtin_amdgcn_readfirstlane(stk)];
        const int S = sd.g.S, L = sd.g.L, L2 = 2 * L, R = sd.g.R, d = sd.filt, w = 2 * d + 1;
        int k1, k2;
        slot_to_pair(slot, sd.g.K, k1, k2);
        const double2* P1 = sd.P64 + (size_t)k1 * L * R;
        const double2* P2 = sd.P64 + (size_t)k2 * L * R;
        __syncthreads();
        if (tid == 0) *s_stop = 0;
        if (tid < w) {
            s_w[tid] = 2.0 * sd.wts[tid * w + d];  // 2: a map entry is twice its sum
            s_w[CF_MAXW + tid] = sd.wts[d * w + tid] / sd.wts[d * w + d];
        }
        __syncthreads();
        double sa = 0.0, sb = 0.0;
        for (int i = 0; i < w; i++) {
            sa += s_w[i];
            sb += s_w[CF_MAXW + i];
        }
        const double E = sa * sb * (double)sd.nrm[k1] * (double)sd.nrm[k2] * 0x1p-53 *
                         2.0 * (2.0 * (R + 8) + w * w + 4 * d + 16);
        cl.reset(2.0 * E);
        const int OT = CF_T - 2 * d, NO = (L + OT - 1) / OT;  // outputs per tile side, tiles per side
        const int U = S * NO * NO;
        const int u0 = (int)((long long)blockIdx.y * U / a.x.sj), u1 = (int)((long long)(blockIdx.y + 1) * U / a.x.sj);
        const int KS = (R + 3) / 4;
        int stop = 0;
        for (int u = u0; u < u1 && !stop; u++) {
            const int j = u / (NO * NO), tr = (u / NO) % NO, tc = u % NO;
            const int row0 = tr * OT, col0 = tc * OT;
            const double2* ph = sd.ph64 + (size_t)j * R;
            // extended index x (from -d) -> line and whether it is the other half's
            auto wrap = [&](int x, bool& f) {
                if (x < 0) x += L2;
                while (x >= L2) x -= L2;
                f = x >= L;
                return f ? x - L : x;
            };
            bool f;
            const double2* pa = P1 + (size_t)wrap(row0 - d + 16 * wave + r16, f) * R;
            const double2* pb[4];
            bool fc[4];
#pragma unroll
            for (int c = 0; c < 4; c++) pb[c] = P2 + (size_t)wrap(col0 - d + 16 * c + r16, fc[c]) * R;
            d4 C1[4], C2[4];
#pragma unroll
            for (int c = 0; c < 4; c++) C1[c] = C2[c] = d4{0.0, 0.0, 0.0, 0.0};
            double2 p = make_double2(0.0, 0.0), q = p, b[4];
#pragma unroll
            for (int c = 0; c < 4; c++) b[c] = p;
            if (kq < R) {
                p = pa[kq];
                q = ph[kq];
#pragma unroll
                for (int c = 0; c < 4; c++) b[c] = pb[c][kq];
            }
            for (int ks = 0; ks < KS; ks++) {
                const int r = 4 * (ks + 1) + kq;  // the next step's samples
                double2 pn = make_double2(0.0, 0.0), qn = pn, bn[4];
#pragma unroll
                for (int c = 0; c < 4; c++) bn[c] = pn;
                if (r < R) {
                    pn = pa[r];
                    qn = ph[r];
#pragma unroll
                    for (int c = 0; c < 4; c++) bn[c] = pb[c][r];
                }
                const double xr = p.x * q.x, yi = p.y * q.y, xi = p.x * q.y, yr = p.y * q.x;
                const double are = xr - yi, aim = xi + yr;  // P1 .* ph
                const double fre = xr + yi, fim = xi - yr;  // conj(P1) .* ph
#pragma unroll
                for (int c = 0; c < 4; c++) {
                    C1[c] = __builtin_amdgcn_mfma_f64_16x16x4f64(are, b[c].x, C1[c], 0, 0, 0);
                    C2[c] = __builtin_amdgcn_mfma_f64_16x16x4f64(fre, b[c].x, C2[c], 0, 0, 0);
                    C1[c] = __builtin_amdgcn_mfma_f64_16x16x4f64(aim, b[c].y, C1[c], 0, 0, 0);
                    C2[c] = __builtin_amdgcn_mfma_f64_16x16x4f64(fim, b[c].y, C2[c], 0, 0, 0);
                }
                p = pn;
                q = qn;
#pragma unroll
                for (int c = 0; c < 4; c++) b[c] = bn[c];
            }
            __syncthreads();  // the previous unit's reads of the tile are done
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const int i = 16 * wave + 4 * e + kq;
                bool fr;
                wrap(row0 - d + i, fr);
#pragma unroll
                for (int c = 0; c < 4; c++) {
                    const bool o = fr != fc[c];
                    double* t = s_T + (size_t)i * CF_LD + 16 * c + r16;
                    t[0] = o ? C2[c][e] : C1[c][e];
                    t[CF_T * CF_LD] = o ? C1[c][e] : C2[c][e];
                }
            }
            __syncthreads();
            // the units before this one's: all waves read it between two barriers
            // that a wave of this unit writes it after
            const int stopped = *s_stop;
            // rows (half, i) dealt to the waves, a lane per column; the taps
            // outermost, so that 32 reads are in flight
            double sum[32];
            const double* const t0 = s_T + (size_t)wave * CF_LD + min(lane, OT - 1);
#pragma unroll
            for (int x = 0; x < 32; x++) sum[x] = 0.0;
            for (int y = 0; y < w; y++) {
                const double wt = s_w[CF_MAXW + y];
#pragma unroll
                for (int x = 0; x < 32; x++) sum[x] = fma(wt, t0[4 * x * CF_LD + y], sum[x]);
            }
            __syncthreads();
#pragma unroll
            for (int x = 0; x < 32; x++) s_T[(size_t)(4 * x + wave) * CF_LD + lane] = sum[x];
            __syncthreads();
#pragma unroll
            for (int x = 0; x < 32; x++) sum[x] = 0.0;
            for (int y = 0; y < w; y++) {
                const double wt = s_w[y];
#pragma unroll
                for (int x = 0; x < 32; x++) {
                    const int i = min(4 * (x & 15) + wave, OT - 1);  // rows past the outputs: the last one again
                    sum[x] = fma(wt, s_T[(size_t)((x >> 4) * CF_T + i + y) * CF_LD + lane], sum[x]);
                }
            }
            stop = __builtin_amdgcn_readfirstlane(stopped);
            const bool okc = lane < OT && col0 + lane < L;
            const int rows = min(OT, L - row0);
            double m = -INFINITY;
#pragma unroll
            for (int x = 0; x < 32; x++)
                if (4 * (x & 15) + wave < rows) m = fmax(m, sum[x]);
            if (!okc) m = -INFINITY;
            if (!__ballot(m >= cl.thr && m > -INFINITY)) continue;
            // rare once the maximum has been seen
#pragma unroll
            for (int o = 32; o > 0; o >>= 1) m = fmax(m, __shfl_xor(m, o, 64));
            cl.raise(m);
#pragma unroll
            for (int x = 0; x < 32; x++) {
                const int h = x >> 4, i = 4 * (x & 15) + wave;
                if (i < rows) cl.keep(okc, sum[x], tie_key(j, h * L + col0 + lane, row0 + i), lane);
            }
            if (lane == 0 && cl.stopped()) *s_stop = 1;
        }
        // the workgroup's maximum, then the candidates within the margin of it
        // with the oracle's arithmetic
        double M;
        const bool over = cl.finish(s_rv, s_lost, wave, lane, M);
        double bv = -INFINITY;
        long long bk = 0x7fffffffffffffffLL;
        if (!over)
            for (int i = 0; i < cl.n; i++)
                if (cl.v[i] >= M - cl.mg) {
                    const long long key = cl.k[i];
                    const double v = eval_filtered(sd, k1, k2, key, s_T + wave * CF_MAXW * CF_MAXW, lane);
                    if (!isnan(v) && better64(v, key, bv, bk)) { bv = v; bk = key; }
                }
        search64_store(a, sd, it, stk, slot, over, bv, bk, s_rv, s_rk, wave, lane);
    }
}

}  // namespace clm
