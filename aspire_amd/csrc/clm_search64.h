// clm_search64.h -- the FP64 search (CLM_FP64_REF) on the FP64 matrix cores.
//
// Every candidate of every pair is evaluated in FP64 by MFMA, and the ones
// whose value comes within the rounding error of the maximum are evaluated
// again with the oracle's arithmetic and order (eval64), so the records are
// bit-identical to the oracle's.  With a row a = P1 .* ph_e,
//   X = Re(a) . Re(P2),  Y = Im(a) . Im(P2):
// on a symmetric shift grid C1 at shift e is 2 (X + Y) and C2 at shift
// S - 1 - e is 2 (X - Y); otherwise C2 has rows conj(P1) .* ph_e of its own
// and each row gives X + Y only.
//
// This sum and the oracle's (R terms, each of two products of rounded factors)
// are each within (R + 8) 2^-53 sum |a||b| <= (R + 8) 2^-53 n1 n2 of the exact
// value, n1 and n2 the images' largest half-line norms.  With d = eps64 n1 n2,
// eps64 twice both coefficients and what the phases of shifts e and S - 1 - e
// differ from conjugates, a candidate more than 2 d below this sum's maximum
// is below the oracle's.  Pairs with more candidates inside that margin than a
// list holds (exact ties, as of radially symmetric images) go to
// exact64_kernel.
#pragma once

namespace clm {

typedef double d4 __attribute__((ext_vector_type(4)));

constexpr int S64_ROWS = 64;   // rows l1 staged at a time
constexpr int S64_LIST = 64;   // candidates kept per wave
// Sets of up to 64 candidates that found no room in a wave's list, after which
// the wave stops: its pair is one of ties everywhere and goes to the exhaustive
// kernels (4950 pairs of radially symmetric images: 44.4 ms there alone, 52.3
// after a whole search, 44.3 so; filtered 17.4, 19.6, 18.2).
constexpr int S64_STOP = 64;

struct Search64Args {
    Exact64Args x;            // items, shift ranges (over units, see below), sv/sk
    int* ovf_count;           // pairs left to exact64_kernel
    SlotRef* ovf_list;
};

// A wave's running maximum and the candidates within the margin of it.
struct CandList {
    double* v;       // LDS, S64_LIST each
    long long* k;
    double mg, wm, thr;  // margin, maximum, keep threshold
    int n, lost;  // entries; sets that did not all fit
    __device__ inline void reset(double margin) {
        mg = margin;
        wm = thr = -INFINITY;
        n = lost = 0;
    }
    __device__ inline bool stopped() const { return lost > S64_STOP; }
    // Raise the threshold for a new maximum (wave-uniform).
    __device__ inline void raise(double m) {
        wm = fmax(wm, m);
        thr = wm - mg;
    }
    // Keep each lane's candidate (ok, value x, tie key) at or above the
    // threshold; called by the whole wave.
    __device__ inline void keep(bool ok, double x, long long key, int lane) {
        const bool on = ok && x >= thr;
        const unsigned long long mask = __ballot(on);
        if (!mask) return;
        const int cnt = __popcll(mask);
        if (n + cnt > S64_LIST) {  // drop what fell below the threshold
            const double ov = lane < n ? v[lane] : 0.0;
            const long long okey = lane < n ? k[lane] : 0;
            const bool kp = lane < n && ov >= thr;
            const unsigned long long km = __ballot(kp);
            __builtin_amdgcn_wave_barrier();
            if (kp) {
                const int pos = __popcll(km & lanemask_lt());
                v[pos] = ov;
                k[pos] = okey;
            }
            n = __popcll(km);
            __builtin_amdgcn_wave_barrier();
        }
        if (on) {
            const int pos = n + __popcll(mask & lanemask_lt());
            if (pos < S64_LIST) {
                v[pos] = x;
                k[pos] = key;
            }
        }
        if (n + cnt > S64_LIST) lost++;
        n = min(n + cnt, S64_LIST);
        __builtin_amdgcn_wave_barrier();
    }
    // The workgroup's maximum M; true if a list lost entries that the margin
    // may hold, or a wave has stopped.  Called by the four waves of the workgroup.
    __device__ inline bool finish(double* s_rv, int* s_lost, int wave, int lane, double& M) {
        if (lane == 0) {
            s_rv[wave] = wm;
            s_lost[wave] = stopped() ? 2 : lost != 0;
        }
        __syncthreads();
        M = s_rv[0];
#pragma unroll
        for (int w = 1; w < 4; w++) M = fmax(M, s_rv[w]);
        bool over = false;
#pragma unroll
        for (int w = 0; w < 4; w++) over = over || s_lost[w] == 2 || (s_lost[w] && s_rv[w] >= M - mg);
        __syncthreads();
        return over;
    }
};

// Key written for an item's range whose list overflowed (sj > 1).
constexpr long long S64_LOST = -1;

// An item's best of the four waves' (bv, bk): to its outputs, to its range's
// place (sj > 1) or, where a list overflowed, to the list of open pairs.
__device__ inline void search64_store(const Search64Args& a, const StackDev& sd, long long it, int stk, int slot,
                                      bool over, double bv, long long bk, double* s_rv, long long* s_rk, int wave,
                                      int lane) {
    if (lane == 0) {
        s_rv[wave] = bv;
        s_rk[wave] = bk;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int w = 1; w < 4; w++)
            if (better64(s_rv[w], s_rk[w], bv, bk)) { bv = s_rv[w]; bk = s_rk[w]; }
        if (a.x.sj > 1) {
            const long long o = (it - a.x.item0) * a.x.sj + blockIdx.y;
            a.x.sv[o] = bv;
            a.x.sk[o] = over ? S64_LOST : bk;
        } else if (over) {
            a.ovf_list[atomicAdd(a.ovf_count, 1)] = SlotRef{stk, slot};
        } else {
            write_result(sd, slot, bv, bk);
        }
    }
    __syncthreads();
}

// LDS bytes: the staged rows, [r][row] with a row more than staged (the
// threads that write a column then hit different banks), one phase row per
// wave, the candidate lists and the per-wave results.
inline size_t search64_lds(int KS) {
    return (size_t)4 * KS * (S64_ROWS + 1) * 16 + (size_t)4 * 4 * KS * 16 + (size_t)4 * S64_LIST * 16 + 128;
}

// One workgroup per pair (and range of units): wave w holds columns l2 of
// image k2 (CT tiles of 16, all KS k-steps of 4) in registers, the workgroup
// stages 64 rows l1 of image k1 in LDS, and a unit is one evaluation shift on
// one such row block: per row tile of 16 and k-step, one LDS read, one
// complex product with the phases, and 2 CT MFMAs.
// Bound: FP64 MFMA.  7.4 ms for 4950 pairs at n_r = 45, n_theta = 360, 13
// shifts: 61 TFLOP/s issued (a large FP64 matrix product reaches 72 here), of
// which 15% are the padding of 180 rows and columns to 192 and of 44 samples
// to 48.  exact64_kernel, which forms both maps on the vector units, takes
// 44.5 ms.
template <int KS, int CT, bool SYM>
__global__ __launch_bounds__(256, (KS * CT * 4 + CT * 16 <= 200 ? 2 : 1)) void search64_kernel(Search64Args a) {
    extern __shared__ __align__(16) char s_mem[];
    double2* s_p = (double2*)s_mem;                           // [4 KS][S64_ROWS + 1]
    double2* s_ph = s_p + 4 * KS * (S64_ROWS + 1);            // [4][4 KS]
    double* s_v = (double*)(s_ph + 4 * 4 * KS);               // [4][S64_LIST]
    long long* s_k = (long long*)(s_v + 4 * S64_LIST);        // [4][S64_LIST]
    double* s_rv = (double*)(s_k + 4 * S64_LIST);             // [4] wave maxima, then best values
    long long* s_rk = (long long*)(s_rv + 4);                 // [4] best keys
    int* s_lost = (int*)(s_rk + 4);                           // [4]
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r16 = lane & 15, kq = lane >> 4;
    double2* const ph_w = s_ph + wave * 4 * KS;
    CandList cl{s_v + wave * S64_LIST, s_k + wave * S64_LIST};
    const long long n_tot = a.x.list ? (long long)*a.x.n_dev : a.x.n_all;
    const long long n = n_tot < a.x.item0 + a.x.item_cap ? n_tot : a.x.item0 + a.x.item_cap;
    for (long long it = a.x.item0 + blockIdx.x; it < n; it += gridDim.x) {
        int stk, slot;
        exact_item(a.x, it, stk, slot);
        const StackDev& sd = a.x.stacks[__builtin_amdgcn_readfirstlane(stk)];
        const int S = sd.g.S, L = sd.g.L, R = sd.g.R;
        int k1, k2;
        slot_to_pair(slot, sd.g.K, k1, k2);
        const double2* P1 = sd.P64 + (size_t)k1 * L * R;
        const double2* P2 = sd.P64 + (size_t)k2 * L * R;
        const double mg = 2.0 * (double)sd.eps64 * (double)sd.nrm[k1] * (double)sd.nrm[k2];
        const int NE = SYM ? S : 2 * S;
        const int NT = (L + 15) / 16, NRB = (L + S64_ROWS - 1) / S64_ROWS;
        const int U = NRB * NE;
        const int u0 = (int)((long long)blockIdx.y * U / a.x.sj), u1 = (int)((long long)(blockIdx.y + 1) * U / a.x.sj);
        cl.reset(mg);
        for (int cg = 0; cg < NT; cg += 4 * CT) {
            const int ct0 = cg + wave * CT;
            const bool work = ct0 < NT;
            double bre[CT][KS], bim[CT][KS];
#pragma unroll
            for (int c = 0; c < CT; c++) {
                const int l2 = (ct0 + c) * 16 + r16;
#pragma unroll
                for (int ks = 0; ks < KS; ks++) {
                    const int r = 4 * ks + kq;
                    double2 b = make_double2(0.0, 0.0);
                    if (l2 < L && r < R) b = P2[(size_t)l2 * R + r];
                    bre[c][ks] = b.x;
                    bim[c][ks] = b.y;
                }
            }
            int rb_now = -1;
            for (int u = u0; u < u1; u++) {
                const int rb = u / NE, e = u - rb * NE;
                if (rb != rb_now) {
                    rb_now = rb;
                    __syncthreads();
                    for (int x = tid; x < S64_ROWS * 4 * KS; x += 256) {
                        const int row = x / (4 * KS), r = x - row * (4 * KS);
                        const int l1 = rb * S64_ROWS + row;
                        double2 p = make_double2(0.0, 0.0);
                        if (l1 < L && r < R) p = P1[(size_t)l1 * R + r];
                        s_p[r * (S64_ROWS + 1) + row] = p;
                    }
                    __syncthreads();
                }
                if (!work || cl.stopped()) continue;
                // conj(P1) .* ph = conj(P1 .* conj(ph)): the rows of the second
                // half of an asymmetric grid take conjugate phases here and the
                // imaginary part's sign below
                const bool flip = !SYM && e >= S;
                const double2* ph = sd.ph64 + (size_t)(flip ? e - S : e) * R;
                for (int r = lane; r < 4 * KS; r += 64) {
                    double2 q = make_double2(0.0, 0.0);
                    if (r < R) q = ph[r];
                    if (flip) q.y = -q.y;
                    ph_w[r] = q;
                }
                __builtin_amdgcn_wave_barrier();
                const int nrt = min(S64_ROWS / 16, NT - rb * (S64_ROWS / 16));
                for (int rt = 0; rt < nrt; rt++) {
                    d4 X[CT], Y[CT];
#pragma unroll
                    for (int c = 0; c < CT; c++) X[c] = Y[c] = d4{0.0, 0.0, 0.0, 0.0};
                    const double2* pr = s_p + kq * (S64_ROWS + 1) + rt * 16 + r16;
#pragma unroll
                    for (int ks = 0; ks < KS; ks++) {
                        const double2 p = pr[4 * ks * (S64_ROWS + 1)];
                        const double2 q = ph_w[4 * ks + kq];
                        const double ar = fma(p.x, q.x, -(p.y * q.y));
                        const double ai = fma(p.x, q.y, p.y * q.x);
#pragma unroll
                        for (int c = 0; c < CT; c++) {
                            X[c] = __builtin_amdgcn_mfma_f64_16x16x4f64(ar, bre[c][ks], X[c], 0, 0, 0);
                            Y[c] = __builtin_amdgcn_mfma_f64_16x16x4f64(ai, bim[c][ks], Y[c], 0, 0, 0);
                        }
                    }
                    // element i of a tile: row 4 i + kq, column r16
                    const int l1b = rb * S64_ROWS + rt * 16 + kq;
                    double m = -INFINITY;
#pragma unroll
                    for (int c = 0; c < CT; c++) {
                        const bool okc = (ct0 + c) * 16 + r16 < L;
#pragma unroll
                        for (int i = 0; i < 4; i++) {
                            const bool ok = okc && l1b + 4 * i < L;
                            double v;
                            if (SYM) v = X[c][i] + fabs(Y[c][i]);
                            else     v = flip ? X[c][i] - Y[c][i] : X[c][i] + Y[c][i];
                            m = fmax(m, ok ? v : -INFINITY);
                        }
                    }
                    if (!__ballot(m >= cl.thr && m > -INFINITY)) continue;
                    // rare once the maximum has been seen: raise the threshold
                    // and list every candidate at or above it
#pragma unroll
                    for (int o = 32; o > 0; o >>= 1) m = fmax(m, __shfl_xor(m, o, 64));
                    cl.raise(m);
#pragma unroll
                    for (int c = 0; c < CT; c++)
#pragma unroll
                        for (int i = 0; i < 4; i++) {
                            const int l1 = l1b + 4 * i, l2 = (ct0 + c) * 16 + r16;
#pragma unroll
                            for (int s = 0; s < (SYM ? 2 : 1); s++) {
                                const bool minus = SYM ? s == 1 : flip;
                                const double v = minus ? X[c][i] - Y[c][i] : X[c][i] + Y[c][i];
                                const int j = SYM ? (minus ? S - 1 - e : e) : (flip ? e - S : e);
                                cl.keep(l1 < L && l2 < L, v, tie_key(j, minus ? L + l2 : l2, l1), lane);
                            }
                        }
                }
            }
        }
        // the workgroup's maximum, then the candidates within the margin of it
        // with the oracle's arithmetic
        double M;
        const bool over = cl.finish(s_rv, s_lost, wave, lane, M);
        double bv = -INFINITY;
        long long bk = 0x7fffffffffffffffLL;
        if (!over)
            for (int i = 0; i < cl.n; i++)
                if (cl.v[i] >= M - mg) {
                    const long long key = cl.k[i];
                    const double v = eval64(sd, k1, k2, key, lane);
                    if (!isnan(v) && better64(v, key, bv, bk)) { bv = v; bk = key; }
                }
        search64_store(a, sd, it, stk, slot, over, bv, bk, s_rv, s_rk, wave, lane);
    }
}

// Best over an item's ranges (sj > 1), one thread per item.
__global__ void search64_reduce_kernel(Search64Args a) {
    const long long n_tot = a.x.list ? (long long)*a.x.n_dev : a.x.n_all;
    const long long it = a.x.item0 + (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (it >= n_tot || it >= a.x.item0 + a.x.item_cap) return;
    double bv = -INFINITY;
    long long bk = 0x7fffffffffffffffLL;
    bool over = false;
    for (int y = 0; y < a.x.sj; y++) {
        const long long o = (it - a.x.item0) * a.x.sj + y;
        over = over || a.x.sk[o] == S64_LOST;
        if (better64(a.x.sv[o], a.x.sk[o], bv, bk)) { bv = a.x.sv[o]; bk = a.x.sk[o]; }
    }
    int stk, slot;
    exact_item(a.x, it, stk, slot);
    if (over) a.ovf_list[atomicAdd(a.ovf_count, 1)] = SlotRef{stk, slot};
    else write_result(a.x.stacks[stk], slot, bv, bk);
}

using Search64Fn = void (*)(Search64Args);

template <int KS, bool SYM>
inline Search64Fn pick_search64_ct(int ct) {
    if constexpr (KS < 32)
        if (ct == 3) return search64_kernel<KS, 3, SYM>;
    return ct == 1 ? search64_kernel<KS, 1, SYM> : search64_kernel<KS, 2, SYM>;
}

// The kernel for R radial samples and L lines, and its k-steps: k-steps as
// compile-time register arrays, padded to a multiple of 4 samples; columns
// over four waves, at most 3 tiles each (L <= 192 in one sweep; 2 with 32
// k-steps, whose registers hold no more).
inline Search64Fn pick_search64(int R, int L, bool sym, int& KS) {
    KS = R <= 16 ? 4 : R <= 32 ? 8 : R <= 48 ? 12 : R <= 64 ? 16 : R <= 96 ? 24 : 32;
    const int NT = (L + 15) / 16, most = KS < 32 ? 12 : 8;
    const int sweeps = (NT + most - 1) / most, ct = (NT + 4 * sweeps - 1) / (4 * sweeps);
#define CLM_S64(ks) case ks: return sym ? pick_search64_ct<ks, true>(ct) : pick_search64_ct<ks, false>(ct)
    switch (KS) {
        CLM_S64(4);
        CLM_S64(8);
        CLM_S64(12);
        CLM_S64(16);
        CLM_S64(24);
        default: return sym ? pick_search64_ct<32, true>(ct) : pick_search64_ct<32, false>(ct);
    }
#undef CLM_S64
}

}  // namespace clm
