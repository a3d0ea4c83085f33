// clm_kernels.hip -- gfx950 kernels of the common-lines engine (the pair
// kernel and A-stack templates are in clm_pair.h).
//
// The hot path of ASPIRE's cryo_clmatrix_cpu (sinograms/cryo_clmatrix_cpu.m:
// 296-399) for every pair (k1,k2), every shift s_j and every pair of lines:
//   C1 = 2 Re((P1 .* ph_j)^H P2),  C2 = 2 Re((conj(P1) .* ph_j)^H P2)
// followed by a first-max argmax.  Here it is computed as
//   X_e = Re(P1.*ph_e)^T Re(P2),   Y_e = Im(P1.*ph_e)^T Im(P2)
//   C1(s_e) = 2 (X_e + Y_e),       C2(-s_e) = 2 (X_e - Y_e)
// (exact identity: conj(P1).*ph_{-s} = conj(P1.*ph_s)), so one MFMA pass over
// the evaluation shifts e yields both maps; on a symmetric shift grid the
// best of the two at every position is t = X + |Y|.
//
// Kernels:
//   prep_kernel      line assembly, filter, band zeroing, normalization
//                    (:96, :277-293, cryo_raynormalize.m:17-24) -> FP64 and
//                    FP32 half lines + MFMA operand planes.
//   pair_kernel      persistent all-pairs MFMA contraction with a fused
//                    max epilogue (pass 1: best cells; pass 2: every
//                    candidate above a certified threshold).
//   rescore_kernel   FP32 re-score of the surviving candidates, FP64
//                    re-score of near ties, reference tie order.
//   exact64_kernel   FP64 exhaustive search of one pair, the reference's own
//                    arithmetic: the fallback of the other paths and of the
//                    FP64 search (clm_search64.h).
#include "clm_pair.h"

namespace clm {

// -------------------------------------------------------------- preprocess
// Lines (k, l): one workgroup per image and PREP_NL consecutive lines.  The
// two blocks of pf columns that these lines are assembled from (l.. and
// L + l..) are contiguous, so they come in as whole cache lines; everything
// but the two sums over a line is done one element per thread.  The sums run
// in one thread per line, over terms left in LDS, in the oracle's order, so
// P64 is bit-identical to the CPU restatement.
// HBM bound: 103 us at K = 1000, n_r = 45 (0.49 GB read and written, 4.8
// TB/s; a plain device copy reaches 5.1 here) and 264 us at K = 1500,
// n_r = 65, complex128.  One thread per line, with every load and store a
// stride of a whole line apart, took 784 and 1830 us.
constexpr int PREP_T = 256;

// Lines per workgroup.  Sixteen read whole cache lines, eight leave room in LDS for
// twice the workgroups, whose two serial sums per line hide each other.  K = 1000,
// complex128, us with 16 and 8 lines: n_r = 33 97 and 122, 45 118 and 141, 65 193 and
// 183, 66 216 and 200, 79 228 and 214, 90 299 and 229, 97 319 and 258.  The line
// lies where 16 need 34 KB of LDS; between 46 and 66 points it is within 8% either way.
__host__ __device__ inline int prep_lines(int n_r) { return n_r <= 66 ? 16 : 8; }
// per line: 2 n_r - 1 terms (the row padded to an odd number of doubles, for
// the banks of the threads that walk the rows) and R complex values
__host__ __device__ inline size_t prep_lds_bytes(int n_r) {
    return (size_t)prep_lines(n_r) * ((size_t)(2 * n_r + 1) * 8 + (size_t)n_r * 16) + 2 * 16 * sizeof(double);
}

template <typename InT>
__global__ __launch_bounds__(PREP_T) void prep_kernel(const InT* __restrict__ pf, Geom g,
                            const double* __restrict__ H,  // 2n_r-1, zeroed band
                            double2* __restrict__ P64,     // [K][L][R] or null
                            float2* __restrict__ P32,      // [K][L][Rp]
                            void* __restrict__ Bop,        // [K][2][Lp][Rp]
                            int op_kind,                   // 0 f32, 1 bf16, 2 f16
                            unsigned* __restrict__ nrm_bits,  // [K] float bits
                            unsigned long long* __restrict__ n_small,
                            const double* __restrict__ lsh) { // [K][L] per-line shift (px) or null
    extern __shared__ __align__(16) char s_prep[];
    const int n_r = g.n_r, R = g.R, L = g.L, T = g.T, Rp = g.Rp, Lp = g.Lp;
    const int NL = prep_lines(n_r);
    const int ldt = 2 * n_r + 1;
    double2* s_z = (double2*)s_prep;                  // [NL][n_r] filtered half rays
    double* s_t = (double*)(s_z + (size_t)NL * n_r);  // [NL][ldt] terms of the sums
    double* s_nr = s_t + (size_t)NL * ldt;            // [NL] line norms
    const int tid = threadIdx.x;
    // lines run over the padded range l < Lp so padding rows of the operand
    // planes are written (zeros) by the same launch
    const int nblk = (Lp + NL - 1) / NL;
    const int k = blockIdx.x / nblk, l0 = (blockIdx.x % nblk) * NL;
    const int nl = min(NL, L - l0);    // lines with rays (may be <= 0)
    const int nlp = min(NL, Lp - l0);  // lines of the operand planes
    auto put = [&](size_t idx, float v) {
        if (op_kind == 0) ((float*)Bop)[idx] = v;
        else if (op_kind == 1) ((__bf16*)Bop)[idx] = (__bf16)v;
        else ((_Float16*)Bop)[idx] = (_Float16)v;
    };
    const int nv = max(nl, 0) * n_r;
    // element i of a line (i = 0..2 n_r - 2) is column L + l at n_r - 1 - i
    // below the middle, column l at i - (n_r - 1) from there on
    for (int half = 0; half < 2; half++) {
        const InT* base = pf + 2 * ((size_t)k * T + (half ? 0 : L) + l0) * n_r;
        for (int x = tid; x < nv; x += PREP_T) {
            const int j = x / n_r, rr = x - j * n_r;
            if (!half && rr == 0) continue;
            const int i = half ? n_r - 1 + rr : n_r - 1 - rr;
            const double re = (double)base[2 * x] * H[i], im = (double)base[2 * x + 1] * H[i];
            s_t[j * ldt + i] = re * re + im * im;
            if (!half) s_z[j * n_r + i] = make_double2(re, im);
        }
    }
    __syncthreads();
    if (tid < nl) {
        const double* t = s_t + tid * ldt;
        double ss = 0.0;
        for (int i = 0; i < 2 * n_r - 1; i++) ss += t[i];
        const double nr = sqrt(ss);
        if (nr < 1.0e-13) atomicAdd(n_small, 1ull);
        s_nr[tid] = nr;
    }
    __syncthreads();
    for (int x = tid; x < nlp * Rp; x += PREP_T) {
        const int j = x / Rp, r = x - j * Rp, l = l0 + j;
        float fr = 0.f, fi = 0.f;
        if (j < nl && r < R) {
            const double nr = s_nr[j];
            const double2 z = s_z[j * n_r + r];
            double re = z.x / nr, im = z.y / nr;
            if (lsh) {
                // line moved by a px: times exp(-2*pi*i*rk*a/(2R+1)), rk = r - R,
                // the phase the shift search applies for shift a
                const double a = lsh[(size_t)k * L + l];
                const double th = ((-2.0 * M_PI * (double)(r - R)) * a) / (double)(2 * R + 1);
                const double c = cos(th), sn = sin(th);
                const double xr = re * c - im * sn, xi = re * sn + im * c;
                re = xr;
                im = xi;
            }
            if (P64) P64[((size_t)k * L + l) * R + r] = make_double2(re, im);
            fr = (float)re;
            fi = (float)im;
            s_t[j * ldt + r] = re * re + im * im;
        }
        if (j < nl) P32[((size_t)k * L + l) * Rp + r] = make_float2(fr, fi);
        put((((size_t)k * 2 + 0) * Lp + l) * Rp + r, fr);
        put((((size_t)k * 2 + 1) * Lp + l) * Rp + r, fi);
    }
    __syncthreads();
    // max half-line norm of the image, rounded up (bound input of the
    // certified threshold).  Non-finite norms are left out: their lines
    // give NaN correlations, which every max below ignores.
    if (tid < 16) {
        float hf = 0.f;
        if (tid < nl) {
            const double* t = s_t + tid * ldt;
            double hn = 0.0;
            for (int r = 0; r < R; r++) hn += t[r];
            hf = (float)(sqrt(hn) * (1.0 + 1.0e-6));
            if (!isfinite(hf)) hf = 0.f;
        }
#pragma unroll
        for (int o = 8; o > 0; o >>= 1) hf = fmaxf(hf, __shfl_xor(hf, o, 16));
        if (tid == 0 && nl > 0) atomicMax(nrm_bits + k, __float_as_uint(hf));
    }
}

// ------------------------------------------------------------ re-scoring
struct RescoreArgs {
    const StackDev* stacks;   // the whole table (SlotRef.stack indexes it)
    int stack0, nstacks;      // mode 0: stacks [stack0, stack0 + nstacks)
    int mode;                 // 0: every pair of those stacks (pass-1 records),
                              // 1: list with pass-2 candidates, 2: list with pass-1 records
    long long n_items;        // mode 0: total pairs of all stacks
    const int* n_items_dev;   // modes 1, 2: number of list entries (device)
    int item_cap;             // modes 1, 2: entries beyond this are not processed
    const SlotRef* ulist;     // modes 1, 2: u -> (stack, slot)
    int stack_shift;          // modes 1, 2: added to the listed stack index
    const EmitRec* erecs;     // mode 1: candidates of entry u
    int* unc_count;           // mode 0: uncertain pairs appended here
    SlotRef* unc_list;
    int* fb_count;            // both: pairs for the FP64 exhaustive search
    SlotRef* fb_list;
    unsigned long long* stat;  // counts, one area per workgroup & stat_mask: ST_* of it
    int stat_mask;
    int Rmax;                 // longest ray of the stacks served (LDS rows)
};

// Counts of a job: areas of ST_STRIDE words (a cache line), which the host
// adds up.  An atomic on one address takes 11 ns wherever it comes from, so
// workgroups that end together are spread over areas.
constexpr int ST_STRIDE = 16;
constexpr int ST_64 = 1, ST_CELL = 6, ST_EMIT = 7;  // FP64 candidates, cells, second-pass candidates

// Order key of the reference's tie rule (shift index first, then the column
// of [C1 C2], then the row): smaller key wins among equal values.  Packed in
// fields (S <= 4096, L <= 768), so that a key comes apart without divisions.
__device__ inline long long tie_key(int j, int l2p, int l1) {
    return ((long long)j << 32) | (unsigned)(l2p << 16 | l1);
}
__device__ inline int key_l1(long long key) { return (int)key & 0xffff; }
__device__ inline int key_l2p(long long key) { return (int)((unsigned)key >> 16); }
__device__ inline int key_j(long long key) { return (int)(key >> 32); }

__device__ inline bool better(float v, long long k, float bv, long long bk) {
    return v > bv || (v == bv && k < bk);
}
__device__ inline bool better64(double v, long long k, double bv, long long bk) {
    return v > bv || (v == bv && k < bk);
}

// Term r of C(l1, l2p) at shift j in FP64, the oracle's arithmetic: the row
// a = P1(r).*ph_j(r) (conj(P1) for the C2 half, flip), then a.re*b.re +
// a.im*b.im.
__device__ inline double term64(double2 p, double2 q, double2 b, bool flip) {
    double xr, xi;
    if (!flip) { xr = p.x * q.x - p.y * q.y; xi = p.x * q.y + p.y * q.x; }
    else       { xr = p.x * q.x + p.y * q.y; xi = p.x * q.y - p.y * q.x; }
    const double t = xr * b.x, u = xi * b.y;
    return t + u;
}

__device__ inline double readlane64(double x, int l) {
    const unsigned long long u = __double_as_longlong(x);
    const unsigned lo = (unsigned)__builtin_amdgcn_readlane((int)(u & 0xffffffffu), l);
    const unsigned hi = (unsigned)__builtin_amdgcn_readlane((int)(u >> 32), l);
    return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}

// Stack of flat pair index `item` (stacks sorted by pair_base).
__device__ inline int find_stack(const StackDev* st, int n, long long item) {
    int lo = 0, hi = n - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (st[mid].pair_base <= item) lo = mid; else hi = mid - 1;
    }
    return lo;
}

// x / d and x mod d by the reciprocal inv = 1/d, corrected: exact for
// 0 <= x < 2^24 (rows and cells of a map are below 7 million), a third of the
// instructions of an integer division.
__device__ inline int div_by(int x, int d, float inv, int& rem) {
    int q = (int)((float)x * inv);
    int r = x - q * d;
    if (r < 0) { q--; r += d; }
    if (r >= d) { q++; r -= d; }
    rem = r;
    return q;
}

// Geometry of a stack and its reciprocals, in registers.
struct CandGeom {
    int L, Lp, NCT, NROWS;
    float iL, iNCT;
};
__device__ inline CandGeom cand_geom(const Geom& g) {
    return CandGeom{g.L, g.Lp, g.NCT, g.NROWS, 1.0f / g.L, 1.0f / g.NCT};
}

// Decode candidate q of a pair: pass-1 cells expand to 16 rows each,
// pass-2 lists hold (row, col) directly.  row = -1 marks padding.
__device__ inline void cand_rc(const CandGeom& g, int mode, const PairRec& rec, const EmitRec* er,
                               int q, int& row, int& col) {
    if (mode == 0) {
        const uint32_t c = rec.cell[q >> 4];
        const int cl = c & 63, cid = c >> 6;
        int ct;
        const int at = div_by(cid, g.NCT, g.iNCT, ct);
        const int ri = q & 15;
        row = at * 32 + 8 * (ri >> 2) + 4 * (cl >> 5) + (ri & 3);
        col = ct * 32 + (cl & 31);
    } else {
        const uint32_t c = er->cand[q];
        row = (int)(c / (unsigned)g.Lp);
        col = (int)(c - (unsigned)row * (unsigned)g.Lp);
    }
    if (row >= g.NROWS || col >= g.L) row = -1;
}

// C at tie key `key` of pair (k1, k2) in FP64, bit-identical to the oracle:
// lane r forms term r (r = lane, lane + 64, ...) and the terms are added in
// order r = 0..R-1, acc = acc + term, as the oracle adds them.  Called by the
// whole wave with a wave-uniform key; the result is the same in every lane.
__device__ inline double eval64(const StackDev& sd, int k1, int k2, long long key, int lane) {
    const Geom& g = sd.g;
    const int l1 = key_l1(key);
    const int l2p = key_l2p(key);
    const int j = key_j(key);
    const double2* P1 = sd.P64 + ((size_t)k1 * g.L + l1) * g.R;
    const bool flip = l2p >= g.L;
    const double2* P2 = sd.P64 + ((size_t)k2 * g.L + (flip ? l2p - g.L : l2p)) * g.R;
    const double2* ph = sd.ph64 + (size_t)j * g.R;
    double acc = 0.0;
    for (int c0 = 0; c0 < g.R; c0 += 64) {
        const int r = c0 + lane;
        const double tr = r < g.R ? term64(P1[r], ph[r], P2[r], flip) : 0.0;
        const int n = min(64, g.R - c0);
        for (int q = 0; q < n; q++) acc = acc + readlane64(tr, q);
    }
    return 2.0 * acc;
}

__device__ inline void write_result(const StackDev& sd, int slot, double v, long long key) {
    const Geom& g = sd.g;
    if (v > 0.0) {
        const int l1 = key_l1(key);
        const int l2p = key_l2p(key);
        const int j = key_j(key);
        if (sd.cl1) sd.cl1[slot] = l1 + 1;
        if (sd.cl2) sd.cl2[slot] = l2p + 1;
        if (sd.jidx) sd.jidx[slot] = j;
        if (sd.corr) sd.corr[slot] = v;
        if (sd.shift1d) sd.shift1d[slot] = sd.shiftv[j];
    } else {
        if (sd.cl1) sd.cl1[slot] = 0;
        if (sd.cl2) sd.cl2[slot] = 0;
        if (sd.jidx) sd.jidx[slot] = -1;
        if (sd.corr) sd.corr[slot] = 0.0;
        if (sd.shift1d) sd.shift1d[slot] = 0.0;
    }
}

constexpr int RS_MAXV = 2 * MAXE;  // FP32 values kept per pair (2 per row)
constexpr int RS_NB = 4;           // FP64 candidates evaluated together

// Dynamic LDS of rescore_kernel: per wave the FP32 values of a pair (cells of
// the first pass, or a second-pass list), then the FP64 terms and keys of
// RS_NB candidates (R terms each, rows of an odd number of doubles).
__host__ __device__ inline int rescore_nval(int mode) { return mode == 1 ? RS_MAXV : 2 * 16 * MAXC; }
__host__ __device__ inline size_t rescore_lds_bytes(int mode, int R) {
    return 4 * ((size_t)rescore_nval(mode) * 4 + (size_t)RS_NB * (R | 1) * 8 + RS_NB * 8);
}

// One wave per pair.  FP32 re-score with 4 lanes per candidate row (32 rows
// per step, the row's lanes reading adjacent 16-byte pieces), values kept in
// LDS; then FP64 re-score of every candidate within tau of the FP32 best,
// RS_NB at a time: a lane per term, all their loads in flight together, and
// the terms of each added by one lane in the oracle's order.
// Bound by the L1 accesses of the row loads where there are many pairs (3.1 ms
// for 499,500 pairs with 6.8 cells each at n_r = 45; 3.4 with one candidate
// per step in FP64, divisions to take a tie key apart and one counter for
// all), by latency where there are few: with TEAM the four waves of a workgroup
// share a pair's rows and candidates (780 pairs, 34 us; a wave each 53).
template <bool TEAM>
__global__ __launch_bounds__(256, 4) void rescore_kernel(RescoreArgs a) {
    extern __shared__ __align__(16) char s_rs[];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int W = blockDim.x >> 6;
    const int nvmax = rescore_nval(a.mode);
    const int ldt = a.Rmax | 1;
    double* const sterm = (double*)s_rs + (size_t)wave * RS_NB * ldt;
    long long* const skey = (long long*)((double*)s_rs + (size_t)4 * RS_NB * ldt) + wave * RS_NB;
    float* const sval = (float*)((long long*)((double*)s_rs + (size_t)4 * RS_NB * ldt) + 4 * RS_NB) + (size_t)(TEAM ? 0 : wave) * nvmax;
    // a team's bests, one per wave
    __shared__ double s_tv[4];
    __shared__ long long s_tk[4];
    const bool lead = !TEAM || wave == 0;
    const int q = lane & 3, rl = lane >> 2;  // k-quarter, row within a set of 16
    const bool listed = a.mode != 0, emit = a.mode == 1;
    const long long n_items = listed ? (long long)min(*a.n_items_dev, a.item_cap) : a.n_items;
    // counts, summed over the workgroup's items and added once at the end
    __shared__ unsigned long long s_cnt[3][4];
    unsigned long long c_cell = 0, c_emit = 0, c_64 = 0;
    for (long long item = TEAM ? (long long)blockIdx.x : (long long)blockIdx.x * W + wave; item < n_items;
         item += TEAM ? (long long)gridDim.x : (long long)gridDim.x * W) {
        int stk, slot;
        if (!listed) {
            stk = a.stack0 + (a.nstacks > 1 ? find_stack(a.stacks + a.stack0, a.nstacks, item) : 0);
            slot = (int)(item - a.stacks[stk].pair_base);
        } else {
            stk = a.ulist[item].stack + a.stack_shift;
            slot = a.ulist[item].slot;
        }
        // the stack's geometry and pointers in registers: results are stored
        // through sd, so references into it would be re-read on every row
        const StackDev& sd = a.stacks[__builtin_amdgcn_readfirstlane(stk)];
        const Geom g = sd.g;
        const CandGeom cg = cand_geom(g);
        const float2* const P32 = sd.P32;
        const float2* const ph32 = sd.ph32;
        const int kq = g.Rp / 4;  // multiple of 4
        const PairRec& rec = sd.recs[slot];
        const int k1 = rec.k1, k2 = rec.k2;
        const EmitRec* er = emit ? a.erecs + item : nullptr;
        const int cmode = emit ? 1 : 0;
        int nrows;
        if (!emit) {
            if (rec.flags & F_EMPTY) {
                if (lead && lane == 0) write_result(sd, slot, 0.0, 0);
                continue;
            }
            if (rec.flags & (F_UNCERTAIN | F_OVERFLOW)) {
                if (lead && lane == 0) { const int u = atomicAdd(a.unc_count, 1); a.unc_list[u] = SlotRef{stk, slot}; }
                continue;
            }
            nrows = 16 * rec.ncells;
            if (lead) c_cell += (unsigned long long)rec.ncells;
        } else {
            if (er->overflow) {
                if (lead && lane == 0) { const int u = atomicAdd(a.fb_count, 1); a.fb_list[u] = SlotRef{stk, slot}; }
                continue;
            }
            nrows = er->n;
            if (lead) c_emit += (unsigned long long)nrows;
        }
        // ---- FP32 re-score
        float bv = -INFINITY;
        long long bk = 0x7fffffffffffffffLL;
        for (int base = TEAM ? 32 * wave : 0; base < nrows; base += TEAM ? 32 * W : 32) {
            int row[2], col[2], e[2], l1[2];
            const float4 *p[2], *bb[2], *ph[2];
            float X[2] = {0.f, 0.f}, Y[2] = {0.f, 0.f};
#pragma unroll
            for (int u = 0; u < 2; u++) {
                const int r = base + 16 * u + rl;
                row[u] = -1;
                col[u] = 0;
                if (r < nrows) cand_rc(cg, cmode, rec, er, r, row[u], col[u]);
                const int rc = row[u] < 0 ? 0 : row[u];  // rows without a candidate read row 0, unused
                if (row[u] < 0) col[u] = 0;
                e[u] = div_by(rc, cg.L, cg.iL, l1[u]);
                // the 4 lanes of a row read 4 adjacent 16-byte pieces per
                // load (lane q: pieces q, q + 4, ...), so one load touches
                // 16 half cache lines instead of 64 lines
                p[u] = (const float4*)(P32 + ((size_t)k1 * g.L + l1[u]) * g.Rp) + q;
                bb[u] = (const float4*)(P32 + ((size_t)k2 * g.L + col[u]) * g.Rp) + q;
                ph[u] = (const float4*)(ph32 + (size_t)e[u] * g.Rp) + q;
            }
            const int nu = base + 16 < nrows ? 2 : 1;
#pragma unroll 2
            for (int i = 0; i < kq / 2; i++) {
#pragma unroll
                for (int u = 0; u < 2; u++) {
                    if (u >= nu) break;
                    const float4 pv = p[u][4 * i], qv = ph[u][4 * i], b4 = bb[u][4 * i];
                    const float ar0 = fmaf(pv.x, qv.x, -pv.y * qv.y);
                    const float ai0 = fmaf(pv.x, qv.y, pv.y * qv.x);
                    const float ar1 = fmaf(pv.z, qv.z, -pv.w * qv.w);
                    const float ai1 = fmaf(pv.z, qv.w, pv.w * qv.z);
                    X[u] = fmaf(ar0, b4.x, X[u]);
                    Y[u] = fmaf(ai0, b4.y, Y[u]);
                    X[u] = fmaf(ar1, b4.z, X[u]);
                    Y[u] = fmaf(ai1, b4.w, Y[u]);
                }
            }
#pragma unroll
            for (int u = 0; u < 2; u++) {
                if (u >= nu) break;
                X[u] += __shfl_xor(X[u], 1, 64);
                Y[u] += __shfl_xor(Y[u], 1, 64);
                X[u] += __shfl_xor(X[u], 2, 64);
                Y[u] += __shfl_xor(Y[u], 2, 64);
                float v1 = -INFINITY, v2 = -INFINITY;
                long long q1 = 0x7fffffffffffffffLL, q2 = 0x7fffffffffffffffLL;
                if (row[u] >= 0) {
                    if (g.sym) {
                        v1 = 2.f * (X[u] + Y[u]); q1 = tie_key(e[u], col[u], l1[u]);
                        v2 = 2.f * (X[u] - Y[u]); q2 = tie_key(g.S - 1 - e[u], g.L + col[u], l1[u]);
                    } else if (e[u] < g.S) {
                        v1 = 2.f * (X[u] + Y[u]); q1 = tie_key(e[u], col[u], l1[u]);
                    } else {
                        // rows e >= S carry the phase of -s_{e-S}: C2(s_{e-S}) = 2(X - Y)
                        v2 = 2.f * (X[u] - Y[u]); q2 = tie_key(e[u] - g.S, g.L + col[u], l1[u]);
                    }
                }
                const int r = base + 16 * u + rl;
                if (q == 0 && r < nrows && 2 * r + 1 < nvmax) {
                    sval[2 * r] = v1;
                    sval[2 * r + 1] = v2;
                }
                if (better(v1, q1, bv, bk)) { bv = v1; bk = q1; }
                if (better(v2, q2, bv, bk)) { bv = v2; bk = q2; }
            }
        }
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) {
            const float ov = __shfl_xor(bv, o, 64);
            const long long ok = __shfl_xor(bk, o, 64);
            if (better(ov, ok, bv, bk)) { bv = ov; bk = ok; }
        }
        if constexpr (TEAM) {  // the team's best (a float's value is exact as a double)
            if (lane == 0) {
                s_tv[wave] = (double)bv;
                s_tk[wave] = bk;
            }
            __syncthreads();
            for (int w = 0; w < W; w++)
                if (better((float)s_tv[w], s_tk[w], bv, bk)) { bv = (float)s_tv[w]; bk = s_tk[w]; }
            __syncthreads();
        }
        double fv = (double)bv;
        long long fk = bk;
        if (sd.fp64 && bv > -INFINITY) {
            __builtin_amdgcn_wave_barrier();
            // ---- FP64 re-score of every candidate within tau of the FP32
            // best (the best by value, then tie key, does not depend on the
            // visiting order)
            const float lim = bv - sd.tau;
            double b64 = -INFINITY;
            long long k64 = 0x7fffffffffffffffLL;
            const int nv = min(2 * nrows, nvmax);
            const double2* const P1 = sd.P64 + (size_t)k1 * g.L * g.R;
            const double2* const P2 = sd.P64 + (size_t)k2 * g.L * g.R;
            const double2* const ph64 = sd.ph64;
            for (int base = 0; base < nv; base += 64) {
                const int ic = base + lane;
                const bool on = ic < nv && sval[ic] >= lim;
                const unsigned long long mask = __ballot(on);
                const int n = __popcll(mask);
                if (lead) c_64 += (unsigned long long)n;
                const int pos = __popcll(mask & lanemask_lt());
                for (int c0 = TEAM ? RS_NB * wave : 0; c0 < n; c0 += TEAM ? RS_NB * W : RS_NB) {
                    if (on && pos >= c0 && pos < c0 + RS_NB) {
                        int row, col;
                        cand_rc(cg, cmode, rec, er, ic >> 1, row, col);
                        int l1;
                        const int e = div_by(row, cg.L, cg.iL, l1);
                        long long key;
                        if (g.sym) key = (ic & 1) ? tie_key(g.S - 1 - e, g.L + col, l1) : tie_key(e, col, l1);
                        else key = e < g.S ? tie_key(e, col, l1) : tie_key(e - g.S, g.L + col, l1);
                        skey[pos - c0] = key;
                    }
                    __builtin_amdgcn_wave_barrier();
                    const int nb = min(RS_NB, n - c0);
#pragma unroll
                    for (int c = 0; c < RS_NB; c++) {
                        if (c >= nb) break;
                        const long long key = skey[c];
                        const int l1 = key_l1(key);
                        const int l2p = key_l2p(key);
                        const int j = key_j(key);
                        const bool flip = l2p >= g.L;
                        const double2* a1 = P1 + (size_t)l1 * g.R;
                        const double2* a2 = P2 + (size_t)(flip ? l2p - g.L : l2p) * g.R;
                        const double2* aq = ph64 + (size_t)j * g.R;
                        for (int r = lane; r < g.R; r += 64) sterm[c * ldt + r] = term64(a1[r], aq[r], a2[r], flip);
                    }
                    __builtin_amdgcn_wave_barrier();
                    if (lane < nb) {
                        double acc = 0.0;
                        const double* t = sterm + lane * ldt;
                        for (int r = 0; r < g.R; r++) acc = acc + t[r];
                        const double v = 2.0 * acc;
                        const long long key = skey[lane];
                        if (!isnan(v) && better64(v, key, b64, k64)) { b64 = v; k64 = key; }
                    }
                    __builtin_amdgcn_wave_barrier();
                }
            }
            // lanes 0..RS_NB-1 hold the bests of their candidates
#pragma unroll
            for (int o = RS_NB / 2; o > 0; o >>= 1) {
                const double ov = __shfl_xor(b64, o, 64);
                const long long ok = __shfl_xor(k64, o, 64);
                if (better64(ov, ok, b64, k64)) { b64 = ov; k64 = ok; }
            }
            if constexpr (TEAM) {
                if (lane == 0) {
                    s_tv[wave] = b64;
                    s_tk[wave] = k64;
                }
                __syncthreads();
                for (int w = 0; w < W; w++)
                    if (better64(s_tv[w], s_tk[w], b64, k64)) { b64 = s_tv[w]; k64 = s_tk[w]; }
                __syncthreads();
            }
            fv = b64;
            fk = k64;
        }
        if (lead && lane == 0) write_result(sd, slot, fv, fk);
        __builtin_amdgcn_wave_barrier();
    }
    if (lane == 0) {
        s_cnt[0][wave] = c_64;
        s_cnt[1][wave] = c_cell;
        s_cnt[2][wave] = c_emit;
    }
    __syncthreads();
    if (threadIdx.x < 3) {
        unsigned long long n = 0;
        for (int w = 0; w < W; w++) n += s_cnt[threadIdx.x][w];
        const int at = threadIdx.x == 0 ? ST_64 : threadIdx.x == 1 ? ST_CELL : ST_EMIT;
        if (n) atomicAdd(a.stat + (size_t)(blockIdx.x & a.stat_mask) * ST_STRIDE + at, n);
    }
}

// Pass-2 (or refinement) tiles from an uncertain list, on the device: one
// pair per tile (entry u -> tile u and explicit pair u); the tiles name stack
// r.stack + stack_shift (the FP32 twin of r.stack for the refinement).
// Entries past `cap` have no pass-2 buffers and go straight to the FP64
// exhaustive list.
__global__ void build_pass2_kernel(const StackDev* stacks, const int* n_unc, const SlotRef* ulist, int cap,
                                   int4* tiles, int4* plist, int* ntiles, int* fb_count, SlotRef* fb_list,
                                   int stack_shift) {
    const int n = *n_unc;
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i == 0) *ntiles = min(n, cap);
    for (int u = i; u < n; u += gridDim.x * blockDim.x) {
        const SlotRef r = ulist[u];
        if (u < cap) {
            const PairRec& rec = stacks[r.stack].recs[r.slot];
            tiles[u] = make_int4(rec.k1, u, 1 | ((r.stack + stack_shift) << 4), -1);
            plist[u] = make_int4(rec.k2, r.slot, u, 0);
        } else {
            const int f = atomicAdd(fb_count, 1);
            fb_list[f] = r;
        }
    }
}

// ------------------------------------------------------ FP64 exhaustive
// Every candidate of a pair in FP64 with the oracle's arithmetic: for shift
// j and map m the rows a(r) = P1(r).*ph_j(r) (conj(P1) for C2) are formed
// exactly as the oracle forms them, and each entry accumulates
// acc = acc + (a.re*b.re + a.im*b.im) over r = 0..R-1 in order, so every value
// is bit-identical to the oracle's.  Computed as 64 x 64 output tiles (rows
// l1, columns l2 of one map) with 16 outputs per thread and the operands of
// 32 consecutive r staged in LDS.  The best (value, tie key) wins; the key
// is the reference's first-max order.
struct Exact64Args {
    const StackDev* stacks;   // the whole table (SlotRef.stack indexes it)
    int stack0, nstacks;      // without a list: stacks [stack0, stack0 + nstacks)
    const SlotRef* list;      // pairs to compute, or null: every pair of those stacks
    const int* n_dev;         // list length (device)
    long long n_all;          // pairs when list is null
    long long item0;          // this launch handles items [item0, item0 + item_cap)
    long long item_cap;
    int sj;                   // shift ranges per item (gridDim.y); 1: a workgroup does the whole item
    double* sv;               // sj > 1: best value and key per (item - item0, range)
    long long* sk;
};

__device__ inline void slot_to_pair(long long s, int K, int& k1, int& k2) {
    // e(k1,k2) = k1*K - k1*(k1+1)/2 + (k2-k1-1)
    double Kd = (double)K;
    double d = (2.0 * Kd - 1.0) * (2.0 * Kd - 1.0) - 8.0 * (double)s;
    int a = (int)floor(((2.0 * Kd - 1.0) - sqrt(d > 0 ? d : 0)) / 2.0);
    if (a < 0) a = 0;
    auto first = [&](long long x) { return x * K - x * (x + 1) / 2; };
    while (a > 0 && first(a) > s) a--;
    while (first(a + 1) <= s) a++;
    k1 = a;
    k2 = (int)(s - first(a)) + a + 1;
}

__device__ inline void exact_item(const Exact64Args& a, long long it, int& stk, int& slot) {
    if (a.list) { stk = a.list[it].stack; slot = a.list[it].slot; }
    else {
        stk = a.stack0 + (a.nstacks > 1 ? find_stack(a.stacks + a.stack0, a.nstacks, it) : 0);
        slot = (int)(it - a.stacks[stk].pair_base);
    }
}

__global__ __launch_bounds__(256) void exact64_kernel(Exact64Args a) {
    __shared__ double2 sA[32][64];  // a(r) of 64 rows l1, 32 consecutive r
    __shared__ double2 sB[32][64];  // P2(r) of 64 columns l2
    const long long n_tot = a.list ? (long long)*a.n_dev : a.n_all;
    const long long n = n_tot < a.item0 + a.item_cap ? n_tot : a.item0 + a.item_cap;
    const int tid = threadIdx.x, tx = tid & 15, ty = tid >> 4;
    for (long long it = a.item0 + blockIdx.x; it < n; it += gridDim.x) {
        int stk, slot;
        exact_item(a, it, stk, slot);
        const StackDev& sd = a.stacks[stk];
        const int S = sd.g.S, L = sd.g.L, R = sd.g.R;
        int k1, k2;
        slot_to_pair(slot, sd.g.K, k1, k2);
        const int j0 = (int)((long long)blockIdx.y * S / a.sj), j1 = (int)((long long)(blockIdx.y + 1) * S / a.sj);
        const int NT = (L + 63) / 64;
        const double2* P1 = sd.P64 + (size_t)k1 * L * R;
        const double2* P2 = sd.P64 + (size_t)k2 * L * R;
        double bv = -INFINITY;
        long long bk = 0x7fffffffffffffffLL;
        for (int j = j0; j < j1; j++) {
            const double2* ph = sd.ph64 + (size_t)j * R;
            for (int m = 0; m < 2; m++)
                for (int rt = 0; rt < NT; rt++)
                    for (int ct = 0; ct < NT; ct++) {
                        double acc[4][4];
#pragma unroll
                        for (int i = 0; i < 4; i++)
#pragma unroll
                            for (int k = 0; k < 4; k++) acc[i][k] = 0.0;
                        for (int r0 = 0; r0 < R; r0 += 32) {
                            const int rn = R - r0 < 32 ? R - r0 : 32;
                            __syncthreads();
                            for (int idx = tid; idx < 32 * 64; idx += 256) {
                                const int rr = idx >> 6, col = idx & 63;
                                double2 av = make_double2(0.0, 0.0), bb = make_double2(0.0, 0.0);
                                const int l1 = rt * 64 + col, l2 = ct * 64 + col;
                                if (rr < rn && l1 < L) {
                                    const double2 pv = P1[(size_t)l1 * R + r0 + rr], qv = ph[r0 + rr];
                                    const double pr = pv.x, pi = pv.y, qr = qv.x, qi = qv.y;
                                    if (m == 0) av = make_double2(pr * qr - pi * qi, pr * qi + pi * qr);
                                    else        av = make_double2(pr * qr + pi * qi, pr * qi - pi * qr);
                                }
                                if (rr < rn && l2 < L) bb = P2[(size_t)l2 * R + r0 + rr];
                                sA[rr][col] = av;
                                sB[rr][col] = bb;
                            }
                            __syncthreads();
                            for (int rr = 0; rr < rn; rr++) {
                                double2 A[4], B[4];
#pragma unroll
                                for (int i = 0; i < 4; i++) {
                                    A[i] = sA[rr][ty + 16 * i];
                                    B[i] = sB[rr][tx + 16 * i];
                                }
#pragma unroll
                                for (int i = 0; i < 4; i++)
#pragma unroll
                                    for (int k = 0; k < 4; k++) {
                                        const double t = A[i].x * B[k].x, u = A[i].y * B[k].y;
                                        acc[i][k] = acc[i][k] + (t + u);
                                    }
                            }
                        }
#pragma unroll
                        for (int i = 0; i < 4; i++)
#pragma unroll
                            for (int k = 0; k < 4; k++) {
                                const int l1 = rt * 64 + ty + 16 * i, l2 = ct * 64 + tx + 16 * k;
                                if (l1 < L && l2 < L) {
                                    const double v = 2.0 * acc[i][k];
                                    const long long key = tie_key(j, l2 + m * L, l1);
                                    if (!isnan(v) && better64(v, key, bv, bk)) { bv = v; bk = key; }
                                }
                            }
                    }
        }
        // workgroup best (LDS of the tiles reused)
        __syncthreads();
        double* s_v = (double*)&sA[0][0];
        long long* s_k = (long long*)&sB[0][0];
        s_v[tid] = bv;
        s_k[tid] = bk;
        __syncthreads();
        for (int o = 128; o > 0; o >>= 1) {
            if (tid < o && better64(s_v[tid + o], s_k[tid + o], s_v[tid], s_k[tid])) {
                s_v[tid] = s_v[tid + o];
                s_k[tid] = s_k[tid + o];
            }
            __syncthreads();
        }
        if (tid == 0) {
            if (a.sj == 1) write_result(sd, slot, s_v[0], s_k[0]);
            else {
                const long long e = (it - a.item0) * a.sj + blockIdx.y;
                a.sv[e] = s_v[0];
                a.sk[e] = s_k[0];
            }
        }
        __syncthreads();
    }
}

// Best over an item's shift ranges (sj > 1), one thread per item.
__global__ void exact64_reduce_kernel(Exact64Args a) {
    const long long n_tot = a.list ? (long long)*a.n_dev : a.n_all;
    const long long it = a.item0 + (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (it >= n_tot || it >= a.item0 + a.item_cap) return;
    double bv = -INFINITY;
    long long bk = 0x7fffffffffffffffLL;
    for (int y = 0; y < a.sj; y++) {
        const long long e = (it - a.item0) * a.sj + y;
        if (better64(a.sv[e], a.sk[e], bv, bk)) { bv = a.sv[e]; bk = a.sk[e]; }
    }
    int stk, slot;
    exact_item(a, it, stk, slot);
    write_result(a.stacks[stk], slot, bv, bk);
}

// FP32 operand planes [K][2][Lp][Rp] of a stack from its FP32 half lines
// (the values prep_kernel writes for FP32 operands; zero padding).
__global__ void bop32_kernel(Geom g, const float2* __restrict__ P32, float* __restrict__ Bop) {
    const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    const long long n = (long long)g.K * 2 * g.Lp * g.Rp;
    if (i >= n) return;
    const int r = (int)(i % g.Rp);
    const int l = (int)((i / g.Rp) % g.Lp);
    const int plane = (int)((i / ((long long)g.Rp * g.Lp)) % 2);
    const long long k = i / ((long long)g.Rp * g.Lp * 2);
    float v = 0.f;
    if (l < g.L) {
        const float2 z = P32[((size_t)k * g.L + l) * g.Rp + r];
        v = plane ? z.y : z.x;
    }
    Bop[i] = v;
}

__global__ void fill_i32(int* p, int n, int v) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = v;
}

// ------------------------------------------------------ windowed search
// Per-line 1-D shift of image k implied by a proposed 2-D shift (x, y):
// a(l) = sin(l*pi/L)*x + cos(l*pi/L)*y, the coefficients of the shift
// equations (cryo_clmatrix_cpu.m:722-738), rounded to a multiple of `step`
// so that window shifts land on the reference grid.
__global__ void lineshift_kernel(const float* __restrict__ prop, int K, int L, double step,
                                 double* __restrict__ lsh) {
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= (long)K * L) return;
    const int k = (int)(i / L), l = (int)(i % L);
    const double th = (double)l * M_PI / (double)L;
    const double a = sin(th) * (double)prop[2 * k] + cos(th) * (double)prop[2 * k + 1];
    lsh[i] = rint(a / step) * step;
}

// Window result -> reference grid.  Line l1 of image k1 was moved by a1 and
// line l2 of k2 by a2, so window shift s at a C1 column is grid shift
// s + a1 - a2 and at a C2 column s - a1 - a2.  Pairs whose window peak is
// below `gate`, or whose grid shift is off the grid, are flagged for the
// exhaustive search; the others are written in the reference's form.
__global__ void window_merge_kernel(int K, int L, const double* __restrict__ lsh,
                                    const int32_t* __restrict__ wcl1, const int32_t* __restrict__ wcl2,
                                    const double* __restrict__ wcorr, const double* __restrict__ wshift,
                                    double gate, double max_shift, double step, int S_full,
                                    const double* __restrict__ shiftv_full,
                                    int32_t* cl1, int32_t* cl2, int32_t* jidx, double* corr, double* shift1d,
                                    uint8_t* __restrict__ flag, unsigned long long* __restrict__ counts) {
    const long long P = (long long)K * (K - 1) / 2;
    const long long e = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    const bool valid = e < P;
    bool ok = false, gated = false;
    if (valid) {
        int k1, k2;
        slot_to_pair(e, K, k1, k2);
        const int c1 = wcl1[e], c2 = wcl2[e];
        const double v = wcorr[e];
        int j = -1;
        gated = c1 > 0 && v >= gate;
        if (gated) {
            const double a1 = lsh[(size_t)k1 * L + (c1 - 1)];
            const int l2 = (c2 - 1) % L;
            const double a2 = lsh[(size_t)k2 * L + l2];
            const double sfull = c2 <= L ? wshift[e] + a1 - a2 : wshift[e] - a1 - a2;
            j = (int)rint((sfull + max_shift) / step);
            ok = j >= 0 && j < S_full;
        }
        if (ok) {
            if (cl1) cl1[e] = c1;
            if (cl2) cl2[e] = c2;
            if (jidx) jidx[e] = j;
            if (corr) corr[e] = v;
            if (shift1d) shift1d[e] = shiftv_full[j];
            flag[e] = 0;
        } else {
            flag[e] = 1;
        }
    }
    // counts 0: accepted, 1: below the gate, 2: off the grid; one atomic per
    // wave and kind (an atomic per pair on one address serialises)
    const unsigned long long m0 = __ballot(valid && ok);
    const unsigned long long m1 = __ballot(valid && !gated);
    const unsigned long long m2 = __ballot(valid && gated && !ok);
    if ((threadIdx.x & 63) == 0) {
        if (m0) atomicAdd(counts + 0, (unsigned long long)__popcll(m0));
        if (m1) atomicAdd(counts + 1, (unsigned long long)__popcll(m1));
        if (m2) atomicAdd(counts + 2, (unsigned long long)__popcll(m2));
    }
}

// Common lines of known rotations and the best 1-D shift along each: the
// per-pair loop of cryo_estimate_shifts.m:142-223 (pair order k1 < k2; the
// reference draws its pairs in random order, which the solution does not
// depend on).
__device__ inline bool first_max(double v, int s, double bv, int bs) {
    return !isnan(v) && (isnan(bv) || v > bv || (v == bv && s < bs));
}

// Read-only FP64 data read through the constant address space: loads from a
// wave-uniform address become scalar loads.
typedef const double __attribute__((address_space(4)))* ConstD;

// The shift index of one pair's rays p (image k1) and b (image k2) as the
// reference finds it: lane s evaluates the shifts s, s + 64, ... with the FP64
// terms of eval64 added in order over the ray, then the wave finds the first
// maximum of C1 and of C2 (NaN ignored, as MATLAB's max).  Called by the whole
// wave with uniform rays.
__device__ inline int shift_by_terms(const Geom& g, const double2* ph64, const double2* ray1, const double2* ray2,
                                     int lane) {
    const ConstD ri = (ConstD)ray1, rj = (ConstD)ray2;
    double b1 = NAN, b2 = NAN;
    int s1 = 0, s2 = 0;
    for (int s0 = 0; s0 < g.S; s0 += 64) {
        const int s = s0 + lane;
        const int sc = s < g.S ? s : g.S - 1;
        double a1 = 0.0, a2 = 0.0;
        for (int r = 0; r < g.R; r++) {
            const double2 pv = make_double2(ri[2 * r], ri[2 * r + 1]);
            const double2 bv = make_double2(rj[2 * r], rj[2 * r + 1]);
            const double2 qv = ph64[(size_t)sc * g.R + r];
            a1 = a1 + term64(pv, qv, bv, false);
            a2 = a2 + term64(pv, qv, bv, true);
        }
        const double c1 = 2.0 * a1, c2 = 2.0 * a2;
        if (s < g.S && first_max(c1, s, b1, s1)) { b1 = c1; s1 = s; }
        if (s < g.S && first_max(c2, s, b2, s2)) { b2 = c2; s2 = s; }
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        const double v1 = __shfl_xor(b1, o, 64), v2 = __shfl_xor(b2, o, 64);
        const int t1 = __shfl_xor(s1, o, 64), t2 = __shfl_xor(s2, o, 64);
        if (first_max(v1, t1, b1, s1)) { b1 = v1; s1 = t1; }
        if (first_max(v2, t2, b2, s2)) { b2 = v2; s2 = t2; }
    }
    // an all-NaN max is NaN at index 1 (s = 0) in MATLAB, as here
    return b1 > b2 ? s1 : s2;
}

// Largest and second largest value, and the largest's index.
struct Top2 {
    double v, w;
    int s;
    __device__ inline void add(double x, int sx) {
        if (x > v) { w = v; v = x; s = sx; }
        else if (x > w) w = x;
    }
    __device__ inline void join(double ov, double ow, int os) {
        if (ov > v) { w = fmax(v, ow); v = ov; s = os; }
        else w = fmax(w, ov);
    }
};

// One wave takes 64 consecutive pairs at a time.  Each lane finds its own
// pair's common line (and writes the outputs of a pair that the selection
// leaves out); the selected pairs are then correlated 16 at a time on the FP64
// matrix cores: with z = conj(p) b and w = p b (p, b the pair's rays),
//   C1(s) = 2 sum_r cos z.re + sin z.im,   C2(s) = 2 sum_r cos w.re + sin w.im,
// cos + i sin = ph_s(r), a product of the pairs' rows (r, re and im) with the
// table of phases.  Only the index of the maximum is kept, so it is certain
// where the winning value is farther from the next one, and from the other
// map's best, than both evaluations' rounding (eps64 of the image norms);
// otherwise the pair is evaluated term by term.
// Bound: the gather of the rays (2 KB per pair at n_r = 65) and FP64 MFMA
// about equally.  0.71 ms for 1.12 M pairs, 41 shifts, n_r = 65 (3.3 TB/s of
// rays); with a wave per pair, a lane per shift and every term in the oracle's
// order it took 4.05 ms.
// With PH_LDS the shift phases are staged in LDS once per workgroup as [r][s],
// so that the lanes (one per shift) read consecutive entries at each ray
// index; otherwise they are read from the [s][r] table in global memory.
template <bool PH_LDS>
__global__ __launch_bounds__(512, 4) void rotlines_kernel(const StackDev* __restrict__ sdp,
                                                          const double* __restrict__ rot,
                                                          const uint8_t* __restrict__ sel, int n_theta,
                                                          int32_t* __restrict__ cl1, int32_t* __restrict__ cl2,
                                                          double* __restrict__ shift1d) {
    typedef double d4 __attribute__((ext_vector_type(4)));
    extern __shared__ double2 s_ph[];  // [R][S] when PH_LDS
    const StackDev& sd = *sdp;
    const Geom g = sd.g;
    const double2* const ph64 = sd.ph64;
    const double2* const P64 = sd.P64;
    const long long K = g.K, P = K * (K - 1) / 2;
    const int lane = threadIdx.x & 63, r16 = lane & 15, kq = lane >> 4;
    if (PH_LDS) {
        for (int i = threadIdx.x; i < g.S * g.R; i += blockDim.x) {
            const int s = i / g.R, r = i - s * g.R;
            s_ph[r * g.S + s] = ph64[i];
        }
        __syncthreads();
    }
    const long long nw = (long long)gridDim.x * (blockDim.x >> 6);
    // the wave's index, made visibly uniform (scalar) for the compiler
    const int wid = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    for (long long base = ((long long)blockIdx.x * (blockDim.x >> 6) + wid) * 64; base < P; base += nw * 64) {
        const long long el = base + lane;
        const bool act = el < P && (!sel || sel[el]);
        if (el < P && !act) {
            cl1[el] = -1;
            cl2[el] = -1;
            shift1d[el] = 0.0;
        }
        const unsigned long long todo = __ballot(act);
        if (!todo) continue;
        // ---- the lane's pair: rays (image and line) of both images
        int ray1 = 0, ray2 = 0;  // k L + line
        double tol = 0.0;
        if (act) {
            int q1, q2;
            slot_to_pair(el, (int)K, q1, q2);
            // commonline_R(R_k1.', R_k2.', n_theta): Ut = R_k2.' * R_k1, entry
            // (a, b) = sum over m of R_k2(m, a) R_k1(m, b), m in order
            const double* Ri = rot + 9 * (size_t)q1;
            const double* Rj = rot + 9 * (size_t)q2;
            auto ut = [&](int a, int b) {
                return (Rj[3 * a] * Ri[3 * b] + Rj[1 + 3 * a] * Ri[1 + 3 * b]) + Rj[2 + 3 * a] * Ri[2 + 3 * b];
            };
            const double PI = M_PI;  // 4*atan(1.0) in commonline_R.m:27
            const double aij = atan2(ut(2, 0), -ut(2, 1)) + PI;
            const double aji = atan2(-ut(0, 2), ut(1, 2)) + PI;
            // round half away from zero, then mod n_theta; angles are in [0, 2 pi]
            // (a rotation with NaN entries gives line 0)
            double xij = round(aij / (2 * PI) * n_theta), xji = round(aji / (2 * PI) * n_theta);
            if (!(xij >= 0.0 && xij <= n_theta)) xij = 0.0;
            if (!(xji >= 0.0 && xji <= n_theta)) xji = 0.0;
            int cij = (int)xij % n_theta;
            int cji = (int)xji % n_theta;
            const int L2 = n_theta / 2;
            if (cij >= L2) {  // cryo_estimate_shifts.m:155-163
                cij -= L2;
                cji -= L2;
            }
            if (cji < 0) cji += n_theta;
            cl1[el] = cij + 1;
            cl2[el] = cji + 1;
            ray1 = q1 * g.L + cij;
            ray2 = q2 * g.L + (cji < L2 ? cji : cji - L2);
            tol = 2.0 * sd.eps64 * (double)sd.nrm[q1] * (double)sd.nrm[q2];
        }
        // ---- 16 selected pairs at a time: row r16 is the (first + r16)-th
        const int n = __popcll(todo), at = __popcll(todo & lanemask_lt());
        // lane i of `src` holds the lane of the i-th selected pair
        int src = 0;
        {
            unsigned long long m = todo;
            for (int i = 0; i < n; i++) {
                const int l = __builtin_ctzll(m);
                m &= m - 1;
                if (lane == i) src = l;
            }
        }
        int win = -1;  // this lane's pair's shift index
        for (int first = 0; first < n; first += 16) {
            const int from = __shfl(src, min(first + r16, n - 1), 64);
            const double2* p = P64 + (size_t)__shfl(ray1, from, 64) * g.R;
            const double2* b = P64 + (size_t)__shfl(ray2, from, 64) * g.R;
            Top2 c1[4], c2[4];  // rows 4 i + kq of the two maps
#pragma unroll
            for (int i = 0; i < 4; i++) c1[i] = c2[i] = Top2{-INFINITY, -INFINITY, 0};
            for (int s0 = 0; s0 < g.S; s0 += 48) {
                d4 X[3], Y[3];
#pragma unroll
                for (int c = 0; c < 3; c++) X[c] = Y[c] = d4{0.0, 0.0, 0.0, 0.0};
                int sc[3];
#pragma unroll
                for (int c = 0; c < 3; c++) sc[c] = min(s0 + 16 * c + r16, g.S - 1);
#pragma unroll 2
                for (int r0 = 0; r0 < g.R; r0 += 4) {
                    const int r = r0 + kq;
                    double2 pv = make_double2(0.0, 0.0), bv = pv;
                    if (r < g.R) {
                        pv = p[r];
                        bv = b[r];
                    }
                    const int rc = min(r, g.R - 1);
                    const double xx = pv.x * bv.x, yy = pv.y * bv.y, xy = pv.x * bv.y, yx = pv.y * bv.x;
                    const double zr = xx + yy, zi = xy - yx, wr = xx - yy, wi = xy + yx;
#pragma unroll
                    for (int c = 0; c < 3; c++) {
                        if (s0 + 16 * c >= g.S) break;
                        const double2 q = PH_LDS ? s_ph[rc * g.S + sc[c]] : ph64[(size_t)sc[c] * g.R + rc];
                        X[c] = __builtin_amdgcn_mfma_f64_16x16x4f64(zr, q.x, X[c], 0, 0, 0);
                        Y[c] = __builtin_amdgcn_mfma_f64_16x16x4f64(wr, q.x, Y[c], 0, 0, 0);
                        X[c] = __builtin_amdgcn_mfma_f64_16x16x4f64(zi, q.y, X[c], 0, 0, 0);
                        Y[c] = __builtin_amdgcn_mfma_f64_16x16x4f64(wi, q.y, Y[c], 0, 0, 0);
                    }
                }
#pragma unroll
                for (int c = 0; c < 3; c++) {
                    const int s = s0 + 16 * c + r16;
                    if (s < g.S)
#pragma unroll
                        for (int i = 0; i < 4; i++) {
                            c1[i].add(X[c][i], s);
                            c2[i].add(Y[c][i], s);
                        }
                }
            }
            // over the 16 lanes of a row, then the row's pair takes its result
#pragma unroll
            for (int i = 0; i < 4; i++) {
#pragma unroll
                for (int o = 8; o > 0; o >>= 1) {
                    c1[i].join(__shfl_xor(c1[i].v, o, 64), __shfl_xor(c1[i].w, o, 64), __shfl_xor(c1[i].s, o, 64));
                    c2[i].join(__shfl_xor(c2[i].v, o, 64), __shfl_xor(c2[i].w, o, 64), __shfl_xor(c2[i].s, o, 64));
                }
                // row 4 i + q sits in lanes 16 q..: its pair reads it there
                const int row = at - first;
                const int from_lane = 16 * (row & 3);
                const double v1 = __shfl(c1[i].v, from_lane & 63, 64), w1 = __shfl(c1[i].w, from_lane & 63, 64);
                const double v2 = __shfl(c2[i].v, from_lane & 63, 64), w2 = __shfl(c2[i].w, from_lane & 63, 64);
                const int t1 = __shfl(c1[i].s, from_lane & 63, 64), t2 = __shfl(c2[i].s, from_lane & 63, 64);
                if (act && row >= 0 && row < 16 && (row >> 2) == i) {
                    if (v1 - v2 > tol && v1 - w1 > tol) win = t1;
                    else if (v2 - v1 > tol && v2 - w2 > tol) win = t2;
                }
            }
        }
        // the pairs whose maximum is not certain
        unsigned long long open = __ballot(act && win < 0);
        while (open) {
            const int l = __builtin_ctzll(open);
            open &= open - 1;
            const int y1 = __builtin_amdgcn_readlane(ray1, l), y2 = __builtin_amdgcn_readlane(ray2, l);
            const int s = shift_by_terms(g, ph64, P64 + (size_t)y1 * g.R, P64 + (size_t)y2 * g.R, lane);
            if (lane == l) win = s;
        }
        if (act) shift1d[el] = sd.shiftv[win];
    }
}

// Partner-subset search: the pairs left out keep the outputs of a pair with
// no common line (cryo_clmatrix_gpu_1.m:346-350 searches only the drawn
// partners; clstack and corrstack stay zero elsewhere).  The selected pairs'
// outputs are written by the search itself.
__global__ void subset_init_kernel(long long P, const uint8_t* __restrict__ sel, int32_t* __restrict__ cl1,
                                   int32_t* __restrict__ cl2, int32_t* __restrict__ jidx, double* __restrict__ corr,
                                   double* __restrict__ shift1d) {
    const long long stride = (long long)gridDim.x * blockDim.x;
    for (long long e = (long long)blockIdx.x * blockDim.x + threadIdx.x; e < P; e += stride) {
        if (sel[e]) continue;
        cl1[e] = 0;
        cl2[e] = 0;
        jidx[e] = -1;
        corr[e] = 0.0;
        shift1d[e] = 0.0;
    }
}

// Flagged pairs -> explicit pass-1 tiles, in pair order.  Three steps: per
// row counts, one scan, per row ordered compaction.
__global__ void row_count_kernel(int K, const uint8_t* __restrict__ flag, int ppw, int* __restrict__ cnt,
                                 int* __restrict__ tcnt) {
    __shared__ int s_c;
    const int k1 = blockIdx.x;
    if (k1 >= K - 1) return;
    if (threadIdx.x == 0) s_c = 0;
    __syncthreads();
    const long long f = (long long)k1 * K - (long long)k1 * (k1 + 1) / 2;
    const int n = K - 1 - k1;
    int c = 0;
    for (int i = threadIdx.x; i < n; i += blockDim.x) c += flag[f + i] ? 1 : 0;
    atomicAdd(&s_c, c);
    __syncthreads();
    if (threadIdx.x == 0) {
        cnt[k1] = s_c;
        tcnt[k1] = (s_c + ppw - 1) / ppw;
    }
}

// Exclusive scans of cnt and tcnt over n rows (one workgroup of 1024).
// Totals go to tot[0] (pairs) and tot[1] (tiles).
__global__ __launch_bounds__(1024) void row_scan_kernel(int n, const int* __restrict__ cnt,
                                                        const int* __restrict__ tcnt, int* __restrict__ off,
                                                        int* __restrict__ toff, int* __restrict__ tot) {
    __shared__ int sa[1024], sb[1024];
    const int t = threadIdx.x, T = blockDim.x;
    const int per = (n + T - 1) / T;
    const int lo = min(n, t * per), hi = min(n, lo + per);
    int a = 0, b = 0;
    for (int i = lo; i < hi; i++) { a += cnt[i]; b += tcnt[i]; }
    sa[t] = a;
    sb[t] = b;
    __syncthreads();
    for (int o = 1; o < T; o <<= 1) {
        const int va = t >= o ? sa[t - o] : 0, vb = t >= o ? sb[t - o] : 0;
        __syncthreads();
        sa[t] += va;
        sb[t] += vb;
        __syncthreads();
    }
    int ea = sa[t] - a, eb = sb[t] - b;
    for (int i = lo; i < hi; i++) {
        off[i] = ea;
        toff[i] = eb;
        ea += cnt[i];
        eb += tcnt[i];
    }
    if (t == T - 1) {
        tot[0] = sa[t];
        tot[1] = sb[t];
    }
}

__global__ __launch_bounds__(256) void row_emit_kernel(int K, int stack, const uint8_t* __restrict__ flag, int ppw,
                                                       const int* __restrict__ off, const int* __restrict__ toff,
                                                       SlotRef* __restrict__ list, int4* __restrict__ plist,
                                                       int4* __restrict__ tiles) {
    __shared__ int s_w[4];
    const int k1 = blockIdx.x;
    if (k1 >= K - 1) return;
    const long long f = (long long)k1 * K - (long long)k1 * (k1 + 1) / 2;
    const int n = K - 1 - k1;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    int base = off[k1];
    const int tb = toff[k1], ob = off[k1];
    for (int i0 = 0; i0 < n; i0 += blockDim.x) {
        const int i = i0 + threadIdx.x;
        const bool on = i < n && flag[f + i];
        const unsigned long long m = __ballot(on);
        if (lane == 0) s_w[wave] = __popcll(m);
        __syncthreads();
        int pre = 0;
        for (int w = 0; w < wave; w++) pre += s_w[w];
        const int tot = s_w[0] + s_w[1] + s_w[2] + s_w[3];
        if (on) {
            const int pos = base + pre + __popcll(m & ((1ull << lane) - 1ull));
            const int slot = (int)(f + i);
            list[pos] = SlotRef{stack, slot};
            plist[pos] = make_int4(k1 + 1 + i, slot, pos, 0);
        }
        base += tot;
        __syncthreads();
    }
    // tiles of this row: PPW consecutive listed pairs each
    const int cnt = base - ob;
    for (int q = threadIdx.x * ppw; q < cnt; q += blockDim.x * ppw)
        tiles[tb + q / ppw] = make_int4(k1, ob + q, min(ppw, cnt - q) | (stack << 4), -1);
}

}  // namespace clm
