// Device-resident Jacobi-PCG of libgip_hip (GIP_LinearSolver.h:45-117).
//
// FP64 iteration k, the reference recurrences and roundings
// (GIP_LinearSolver.h:85-116):
//   direction  beta = rho_k / rho_{k-1}; p = 1.0 s + beta p   (:107-113);
//              here too the x updates due (:95), since p is read anyway:
//              the previous iteration's, or on long operators every second
//              time the two before
//   product    Ap = A p, partials of p.Ap                     (:87-91)
//   update     alpha = rho_k / p.Ap; r += (-alpha) Ap; s = Dinv r;
//              partials of r.s and r.r                        (:93-105)
// Operators of at most 2^19 rows (2048 chunks of 256 rows) take two
// kernels per iteration: the direction is formed inside the product, and
// every workgroup of a kernel re-reduces the previous kernel's partials in
// its prologue (fence-free: plain stores, ordered by the kernel boundary;
// every workgroup computes bit-identical scalars), so a kernel costs about
// one memory round trip before it stores.  Up to kRowsMin rows, three or
// four kernels: grid-stride sweeps whose prologues re-reduce the partials,
// the product's folded first where they are more than 2048 or come from the
// dictionary.  Longer operators sweep one row per
// thread in dispatch order (the pace of a plain stream of each kernel's
// access mix) and take their scalars from one-workgroup kernels (fold +
// finalize) instead, since that many workgroups cannot each re-reduce the
// partials; see the long-path section below.  Scalars that must survive a
// kernel (rho and alpha of the last two iterations, beta, the state word)
// are written by one workgroup: rho and alpha into the slots of their
// iteration's parity, which no workgroup of the same kernel reads.  Every
// kernel reads the solver's state word and returns when the solve has
// finished, so the host queues many iterations and polls the state only now
// and then.
//
// MIXED: the same iteration in FP32 (operator values, vectors and SpMV;
// dot products accumulate in FP64; on long operators three or four kernels whose
// grid-stride sweeps re-reduce the partials in their prologues: the
// row-per-thread form measured 18% slower per FP32 iteration at 256^3)
// on the correction equation, inside an
// FP64 defect-correction loop: when the FP32 residual has dropped by
// inner_tol (or reaches the target) the FP32 correction is added to the
// FP64 x, the FP64 true residual b - A x replaces the FP32 residual (the
// search direction is kept: reliable-update residual replacement, restarted
// with beta = 0 when the recursive residual had drifted more than 10x from
// the true one), and convergence is decided on that FP64 residual only.
// Each correction also takes the FP64 Galerkin step along the constant
// vector 1 of the solved rows, x += c 1 with c = (1.r)/(1.A1): for the
// pinned Neumann pressure Laplacian that vector is the near-null mode
// (eigenvalue ~ pin/N), which FP32 arithmetic cannot resolve; left to the
// FP32 iteration it re-enters through round-off and the corrections
// diverge.  For an SPD operator the step never increases the A-norm error.
// The FP32 iteration is deflated by the same vector (A p replaced by
// A p - A1 (1.Ap)/(1.A1)), so its residual stays orthogonal to 1 and the
// constant mode is left to the FP64 step.
#include <algorithm>
#include <cmath>
#include <cstring>
#include <mutex>
#include <new>
#include <vector>

#include "gip_blas1.h"
#include "gip_internal.h"
#include "gip_rows.h"
#include "gip_spmv.h"

namespace gip {

// Device scalar slots of a solver.
enum {
    S_RHO0 = 0,     // rho of even iterations
    S_RHO1 = 1,     // rho of odd iterations
    S_RR = 3,       // r.r (FP64: last update; MIXED: last status or true residual)
    S_BB = 4,       // b.b
    S_TOL2 = 6,     // (tol ||b||)^2, negative when no tolerance
    S_TRUE_RR = 7,  // FP64 true residual of the last correction (MIXED)
    S_ZAZ = 8,      // 1.A1 over the solved rows (MIXED coarse step)
    S_ALPHA0 = 10,  // alpha of even iterations, as the update kernel formed it
    S_ALPHA1 = 11,  // alpha of odd iterations
    S_BETA = 12,    // beta of the next direction update (FP64, long operators)
    S_COUNT = 16
};
// State word: ST_RUN, ST_BREAK, or ST_CONV; the direction kernel of
// iteration k writes ST_CONV | k << 2, so readers look at the low two bits.
enum { ST_RUN = 0, ST_CONV = 1, ST_BREAK = 2, ST_MASK = 3 };
// Partial-sum arrays, kMaxRedBlocks doubles each.
// P_DN2: p.Ap partials of odd iterations on operators small enough for the
// fused direction-product kernel (which reads the previous iteration's
// partials while writing its own).
// P_SA, P_SA2: partials of 1.Ap of the mixed inner iteration (the constant
// vector's deflation), by iteration parity on small operators.
enum { P_DN = 0, P_RS = 1, P_RR = 2, P_BB = 3, P_RS2 = 4, P_RR2 = 5, P_SUMR = 6, P_DN2 = 7, P_SA = 8, P_SA2 = 9,
       P_COUNT = 10 };

// The nonzero entries of A 1 in FP32, when there are at most kAzList of
// them (count > kAzList: too many, the kernels read A 1 row by row).  A
// pinned Neumann Laplacian has zero row sums but at its pinned row, so its
// A 1 has one nonzero and the long update kernel need not stream A 1.
constexpr int kAzList = 8;
struct AzList {
    int count;
    int idx[kAzList];
    float val[kAzList];
};

struct PcgDev {
    int n, G;      // solved rows, workgroups of the sweeping kernels (<= kMaxRedBlocks)
    int nchunk;    // 256-row chunks: workgroups of the product kernels
    int wpc;       // product partials per chunk the fold reads (one per wavefront, or one)
    int Gdn;       // p.Ap partials the next kernels read (<= kMaxRedBlocks)
    double *chunk; // partials of the product: with the fold, kWaves per
                   // 256-row chunk (one per wavefront); without it, one per
                   // chunk, and these are the P_DN partials themselves
    double *chunk_s;  // long operators: a second array of per-wavefront partials (FP64: r.r; MIXED: 1.Ap)
    double *x, *r, *s, *Ap;
    const double *b, *dinv;
    SP<double> *sp[2];   // small operators: the pairs (s, p) by iteration parity
    SP<float> *sp32[2];  // (iteration k's p, then its s, go into those of parity k)
    float *r32, *s32, *Ap32, *xc32;
    const float *dinv32;
    const float *az32;  // A 1 in FP32 (MIXED deflation)
    const struct AzList *azl;  // its nonzeros, when few (MIXED deflation)
    int deflate;        // MIXED: deflate the constant vector in the inner iteration
    const double *az;  // A 1 on the solved rows (MIXED)
    double *sc;        // S_COUNT scalars
    int *state, *iters;
    double *part;  // P_COUNT x kMaxRedBlocks partials; each array has one
                   // producer grid size and stays zero past it
    int precond;
    // the Jacobi inverse per tuple of the operator's dictionary (LEAN sweeps)
    const DictSel *dc_sel;
    const uint16_t *dc_id;
    const double *ddinv;
    const float *ddinv32;
    __device__ double *P(int k) const { return part + k * kMaxRedBlocks; }
};

// The state word is written by workgroup 0 of a kernel while the other
// workgroups of that kernel may be reading it, so every access is an atomic
// one (relaxed, device scope): a reader sees either the word an earlier
// kernel left (ordered by the kernel boundary) or the one workgroup 0 of
// its own kernel is writing.  Each writer makes both outcomes give the same
// result: the direction kernel stamps a convergence with its iteration, and
// a workgroup that reads its own kernel's stamp takes the convergence path
// every workgroup computes; a breakdown leaves the iterates undefined, so
// skipping work is harmless.  An atomic load is an ordered memory
// reference: the compiler issues it where it is written, together with the
// kernel's other early loads.
__device__ inline int state_load(const int *p) { return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
__device__ inline void state_store(int *p, int v) { __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
__device__ inline bool running(const PcgDev &d) { return state_load(d.state) == ST_RUN; }
// A word read at the top of a kernel and used only after its prologue: an
// atomic load (workgroup scope, relaxed: a plain load instruction) is an
// ordered memory reference, so the compiler issues it where it is written,
// together with the other loads, instead of sinking it to its first use.
__device__ inline double early_load(const double *p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}
__device__ inline int conv_stamp(int k) { return ST_CONV | (k << 2); }
__device__ inline bool leader() { return blockIdx.x == 0 && threadIdx.x == 0; }

__device__ inline double rho_slot(const PcgDev &d, int k) { return d.sc[S_RHO0 + (k & 1)]; }
// p.Ap partials of iteration k in the fused (small-operator) iteration
__device__ inline double *dn_part(const PcgDev &d, int k) { return d.P((k & 1) ? P_DN2 : P_DN); }
// 1.Ap partials of iteration k of the mixed fused iteration
__device__ inline double *sa_part(const PcgDev &d, int k) { return d.P((k & 1) ? P_SA2 : P_SA); }

// Deflation of the constant vector in the mixed inner iteration (deflated
// CG, Saad, Yeung, Erhel and Guyomarc'h, SIAM J. Sci. Comput. 21, 2000,
// with W = 1): the iteration uses w = P A p = A p - A1 (1.Ap)/(1.A1) in
// place of A p, so alpha = rho / (p.Ap - (1.Ap)^2 / (1.A1)) (1.Ap = A1.p:
// A symmetric on the solved rows).  The defect correction already applies
// the matching coarse step (x += c 1).  Off when 1.A1 is not positive and
// finite, like the coarse step.
__device__ inline bool deflating(const PcgDev &d, double zaz) { return d.deflate && zaz > 0.0 && isfinite(zaz); }
__device__ inline double m_denom(double dn, double sap, double zaz, bool dfl) {
    return dfl ? dn - sap * sap / zaz : dn;
}

// Rows a thread of a grid-stride update sweep has in flight: a LEAN row's
// two streams alone leave the memory idle (us per iteration with 1, 2, 4
// rows: mixed 256^3 205 / 197 / 211, FP64 200^3 171 / 167 / 167); a row of
// five streams does not gain (mixed 160^3 clustered 79.4 / 79.4 / 82.3).
template <bool LEAN>
constexpr int kSweepU = LEAN ? 2 : 1;
// LEAN sweeps (long iterations on an operator with a dictionary): the
// preconditioned residual s = Dinv r is not stored.  The direction sweep
// reads r instead of s and forms it again, with the inverse diagonal from
// the dictionary, so the update writes r alone: two vector streams of its
// five less.  The same expression on the same values: the same bits.
__device__ inline double s_of(double r, double di, bool precond) {
    if (!precond) return r;
    double si = 0.0;
    si = si + r * di;  // :99-105
    return si;
}
__device__ inline float s_of(float r, float di, bool precond) { return precond ? r * di : r; }
__device__ inline double dict_dinv(const PcgDev &d, int row, double) {
    return d.precond ? dict_one(d.dc_sel, d.dc_id, d.ddinv, row) : 0.0;
}
__device__ inline float dict_dinv(const PcgDev &d, int row, float) {
    return d.precond ? dict_one(d.dc_sel, d.dc_id, d.ddinv32, row) : 0.0f;
}

// ---- setup ---------------------------------------------------------------

// x = x0 (all), direction buffers = x0 outside the solved rows,
// Ap = (A x0)_i or x0_i on empty rows, r = b + (-1.0) Ap   (:55-70); p null:
// the directions are the pairs' (small operators)
template <int W>
__global__ __launch_bounds__(kBlock) void k_setup_resid(EllView A, PcgDev d, const double *__restrict__ x0, int n_all,
                                                        double *__restrict__ p, double *__restrict__ p2) {
    const int stride = gridDim.x * kBlock;
    for (int i = blockIdx.x * kBlock + threadIdx.x; i < n_all; i += stride) {
        d.x[i] = x0[i];
        if (i >= d.n && p) {
            p[i] = x0[i];
            p2[i] = x0[i];
        } else if (i >= d.n) {
            d.sp[0][i] = d.sp[1][i] = SP<double>{0.0, x0[i]};
        }
    }
    Operand<double> xo{x0};
    FOR_ROWS(d.n, row) {
        double sum;
        bool any = row_dot<W, double, double>(A, A.val, xo, row, sum);
        double t = any ? sum : x0[row];
        d.Ap[row] = t;
        d.r[row] = d.b[row] + -1.0 * t;
    }
}

// p = Dinv r (or r); partials of r.p, b.b, r.r  (:72-80)
__global__ __launch_bounds__(kBlock) void k_setup_dir(PcgDev d, double *__restrict__ p) {
    double rs = 0.0, bb = 0.0, rr = 0.0;
    FOR_ROWS(d.n, row) {
        double ri = d.r[row];
        double pi;
        if (d.precond) {
            pi = 0.0;
            pi = pi + ri * d.dinv[row];
        } else {
            pi = ri;
        }
        if (p)
            p[row] = pi;
        else
            d.sp[0][row].p = pi;
        rs = rs + ri * pi;
        bb = bb + d.b[row] * d.b[row];
        rr = rr + ri * ri;
    }
    double red[3] = {rs, bb, rr};
    block_reduce_n<3>(red);
    if (threadIdx.x == 0) {
        d.P(P_RS)[blockIdx.x] = red[0];
        d.P(P_BB)[blockIdx.x] = red[1];
        d.P(P_RR)[blockIdx.x] = red[2];
    }
}

// What the host reads at a poll: the scalars, the state word and the
// iteration count, by the workgroup that formed them last (flag null: not
// asked for).
struct Pub {
    double *sc;
    int *st;
    uint64_t *flag;
    uint64_t seq;
};
__device__ inline void publish(const PcgDev &d, const Pub &p) {
    if (!p.flag) return;
    __syncthreads();
    const int t = threadIdx.x;
    if (t >= 64) return;  // one wavefront: its stores come before its release
    if (t < S_COUNT) p.sc[t] = d.sc[t];
    if (t == S_COUNT) p.st[0] = state_load(d.state);
    if (t == S_COUNT + 1) p.st[1] = *d.iters;
    if (t == 0) publish_seq(p.flag, p.seq);
}

__global__ __launch_bounds__(64) void k_publish(PcgDev d, Pub pub) { publish(d, pub); }

// one workgroup: rho_0, b.b, r.r, the tolerance, the state word and the iteration count
__global__ __launch_bounds__(kBlock) void k_setup_fin(PcgDev d, double tol, Pub pub) {
    const double rho = sum_partials<RED_SUM>(d.P(P_RS), d.G);
    const double bb = sum_partials<RED_SUM>(d.P(P_BB), d.G);
    const double rr = sum_partials<RED_SUM>(d.P(P_RR), d.G);
    if (threadIdx.x == 0) {
        const double tol2 = tol > 0.0 ? tol * tol * bb : -1.0;
        d.sc[S_RHO0] = rho;
        d.sc[S_BB] = bb;
        d.sc[S_RR] = rr;
        d.sc[S_TOL2] = tol2;
        state_store(d.state, (tol > 0.0 && rr <= tol2) ? ST_CONV : ST_RUN);
        *d.iters = 0;
    }
    publish(d, pub);
}

// ---- FP64 iteration --------------------------------------------------------

// alpha of iteration k, stored by workgroup 0 of K2 of k (every workgroup
// of K2 forms the same value from the same partials), so that a later
// kernel reads one scalar instead of re-reducing the p.Ap partials
__device__ inline double alpha_slot(const PcgDev &d, int k) { return d.sc[S_ALPHA0 + (k & 1)]; }
__device__ inline void store_alpha(const PcgDev &d, int k, double alpha) {
    if (leader()) d.sc[S_ALPHA0 + (k & 1)] = alpha;
}

// A product operand that also keeps the value it reads at the row's own
// column (the p_i of p.Ap, which the row's diagonal entry reads anyway), so
// that the product does not load it a second time (FP64 product: 1.8%
// faster at 256^3; the FP32 product keeps the separate load, which measured
// faster there).
template <class T>
struct SelfOperand {
    const T *__restrict__ p;
    int row;
    mutable T self;
    mutable bool found;
    __device__ inline T at(int j) const {
        const T v = p[j];
        if (j == row) {
            self = v;
            found = true;
        }
        return v;
    }
};

// Kernel prologues.  SMALL (operators of at most 2^19 rows, where every
// thread holds at most one row and a kernel lasts a few microseconds): the
// state word, the scalars, the partials and the row's operands are requested
// together, so the kernel spends one memory round trip before its first
// store, and the direction update is fused into the product (two kernels
// per iteration).  Otherwise (long kernels, where that latency is hidden by
// the sweep) the state word is tested first, with a scalar load, and the
// partial arrays are summed one at a time, which keeps the register count,
// and with it the occupancy of the sweep, low.

// x += alpha_k p of the last iteration k (small operators)
__global__ __launch_bounds__(kBlock) void k_x_flush(PcgDev d, int k) {
    if (!running(d)) return;
    const double alpha = alpha_slot(d, k);
    const SP<double> *__restrict__ sp = d.sp[k & 1];
    FOR_ROWS(d.n, row) d.x[row] = d.x[row] + alpha * sp[row].p;  // :95
}

// Mid-size operators: up to kWideRows rows (mixed: kWideRows32) the products
// run in workgroups of 512 threads, past 2^20 rows 1024, that store one
// partial each, at most kMaxRedBlocks of them, which the update's prologue
// sums like any other: no fold kernel between.  us per iteration with the
// fold and without: FP64 clustered 81^3 29.5 / 27.7, 97^3 37.7 / 36.4, 112^3
// 44.3 / 43.6, 128^3 56.8 / 54.5; mixed 81^3 26.8 / 24.4, 97^3 30.0 / 28.4,
// 112^3 36.0 / 35.6, 128^3 44.9 / 45.2 (so not there); rows in scattered
// order 81^3 37.3 / 36.5 (1024 threads: 38.8, a last round of 7 of 519
// workgroups).  The FP64 products with the dictionary, whose wavefronts run
// for very different times, lose more to wide workgroups than the fold
// takes (128^3 42.0 / 46.4): they keep a fold, k_fold_wide, which forms the
// same partials in the same order, so every layout still gives the same bits.
constexpr int kWideRows = 1024 * kMaxRedBlocks, kWideRows32 = 3 << 19;
static int wide_of(int n) { return n <= 512 * kMaxRedBlocks ? 512 : 1024; }
template <int N, int M>
__device__ inline void wide_store(const PcgDev &d, int c, const double (&sh)[N][M]) {
    __syncthreads();
    const int t = threadIdx.x;
    if (t < M) {
        double v = 0.0;
#pragma unroll
        for (int q = 0; q < N / kWaves; ++q) {
            double w = sh[q * kWaves][t];
#pragma unroll
            for (int j = 1; j < kWaves; ++j) w = w + sh[q * kWaves + j][t];
            v = v + w;
        }
        d.P(t ? P_SA : P_DN)[c] = v;
    }
}

// K1: Ap = A p (empty rows keep Ap), p.Ap partials; one row per thread.
// Long operators: workgroups in dispatch order, one partial per wavefront
// (with the direction and update sweeps in dispatch order too, 2% faster
// per FP64 iteration at 256^3 than the XCD-contiguous order, which keeps
// the neighbour gathers in one XCD's L2).  The state word is tested after
// the row's loads instead of before them, taking its latency off the kernel's
// critical path (FP64 solve at 256^3: 1256 -> 1238 ms); a finished solve then still
// reads the operator, but stores nothing.  (The same reordering in the
// long direction and update sweeps made the solve slower: 1303 ms.)
// SYM: the slot values from the operator's symmetric form (stencil layout).
// NB: threads of a workgroup (more than kBlock: wide_store).
template <int W, int NB, bool SYM = false>
__device__ inline void iter_spmv(const EllView &A, const PcgDev &d, const double *__restrict__ p) {
    const int st = state_load(d.state);  // tested after the row's loads, before any store
    const int c = blockIdx.x;
    const int row = c * NB + threadIdx.x;
    double acc = 0.0, sum = 0.0, pr = 0.0;
    bool any = false;
    if (row < d.n) {
        const SelfOperand<double> po{p, row, 0.0, false};
        if constexpr (SYM)
            any = row_dot_sym<W, double, double>(A, A.val, A.sym, po, row, sum);
        else
            any = row_dot<W, double, double>(A, A.val, po, row, sum);
        if (!any) sum = d.Ap[row];  // empty row: Ap keeps its value
        pr = po.found ? po.self : p[row];
    }
    if (st != ST_RUN) return;
    if (row < d.n) {
        if (any) d.Ap[row] = sum;
        acc = pr * sum;
    }
    acc = wave_sum_63(acc);
    if constexpr (NB > kBlock) {
        __shared__ double sh[NB / 64][1];
        if ((threadIdx.x & 63) == 63) sh[threadIdx.x >> 6][0] = acc;
        wide_store(d, c, sh);
    } else {
        // one partial per wavefront: no barrier, each wavefront retires alone
        if ((threadIdx.x & 63) == 63) d.chunk[c * kWaves + (threadIdx.x >> 6)] = acc;
    }
}

template <int W, int NB>
__global__ __launch_bounds__(NB) void k_iter_spmv(EllView A, PcgDev d, const double *__restrict__ p) {
    iter_spmv<W, NB>(A, d, p);
}

// the first product of a small operator: p_0 from the pairs, XCD-contiguous
// order, one partial per chunk
template <int W>
__global__ __launch_bounds__(kBlock) void k_iter_spmv_small(EllView A, PcgDev d) {
    const int st = state_load(d.state);
    const int c = xcd_block(blockIdx.x, gridDim.x);
    const int row = c * kBlock + threadIdx.x;
    double pr = 0.0, sum = 0.0;
    bool any = false;
    if (row < d.n) {
        const PairOperand<double> po{d.sp[0]};
        pr = po.at(row);
        any = row_dot<W, double, double>(A, A.val, po, row, sum);
        if (!any) sum = d.Ap[row];  // empty row: Ap keeps its value
    }
    if (st != ST_RUN) return;
    if (any) d.Ap[row] = sum;
    double acc = row < d.n ? pr * sum : 0.0;
    acc = block_reduce<RED_SUM>(acc);
    if (threadIdx.x == 0) d.chunk[c] = acc;
}

template <int W, int NB>
__global__ __launch_bounds__(NB) void k_iter_spmv_sym(EllView A, PcgDev d, const double *__restrict__ p) {
    iter_spmv<W, NB, true>(A, d, p);
}

// K1 with the slot values from the dictionary.  The wavefront sums of a
// chunk's four slices are added here, in the order the fold adds them, and
// stored as one value per chunk (an 8-byte store per slice and sum took 12
// of 73 us in the FP32 product at 256^3): the same sums in the same order.
template <int R, int M>
__device__ inline void chunk_store(const PcgDev &d, const double (&sh)[4 * R][M]) {
    __syncthreads();
    const int t = threadIdx.x, c = dict_block(blockIdx.x, gridDim.x) * R + t / M;
    if (t < R * M && c < d.nchunk) {
        double v = 0.0;
#pragma unroll
        for (int j = 0; j < kWaves; ++j) v = v + sh[t / M * 4 + j][t % M];
        (t % M ? d.chunk_s : d.chunk)[c] = v;
    }
}

template <int SW, int R>
__global__ __launch_bounds__(kBlock) void k_iter_spmv_dict(EllView A, PcgDev d, const double *__restrict__ p) {
    __shared__ double sh[4 * R][1];
    const int st = state_load(d.state);
    dict_rows<true, R, SW, double, double>(A, A.val, d.n, p, [&](int row, bool ok, bool any, double sum, double own) {
        if (st != ST_RUN) return;
        if (ok && any) d.Ap[row] = sum;
        if (ok && !any) sum = d.Ap[row];  // empty row: Ap keeps its value
        const double acc = wave_sum_63(ok ? own * sum : 0.0);
        if ((threadIdx.x & 63) == 63) sh[(row >> 6) & (4 * R - 1)][0] = acc;
    });
    if (st != ST_RUN) return;
    chunk_store<R, 1>(d, sh);
}

// ---- small operators: prologue and epilogue sums ----------------------------
//
// M sums of at most 64 K (WAVE: every wavefront sums all of them by itself,
// no LDS and no barrier) or 256 K partials (each wavefront its share, one
// exchange), the same in every lane of every workgroup.  The loads are
// issued unconditionally at load(), early in a kernel: a slot past n is the
// array's last entry, a zero whenever n < kMaxRedBlocks.
constexpr int kSmallK = 8;  // partials per lane
constexpr int kWaveParts = 64 * kSmallK;

__device__ inline double lane_value(double v, int lane) {
    const long long b = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_readlane((int)b, lane);
    const int hi = __builtin_amdgcn_readlane((int)(b >> 32), lane);
    return __longlong_as_double(((long long)hi << 32) | (long long)(unsigned)lo);
}

template <int M, bool WAVE>
struct SmallSums {
    double v[M][kSmallK];
    __device__ inline void load(const double *const (&part)[M], int n) {
        const int step = WAVE ? 64 : kBlock, t = WAVE ? threadIdx.x & 63 : threadIdx.x;
#pragma unroll
        for (int m = 0; m < M; ++m)
#pragma unroll
            for (int k = 0; k < kSmallK; ++k) {
                const int i = t + k * step;
                v[m][k] = part[m][i < n ? i : kMaxRedBlocks - 1];
            }
    }
    __device__ inline void reduce(double (&out)[M]) {
        static_assert(M <= 2, "at most two sums");
        __shared__ double sh[kWaves][2];
        double acc[2] = {0.0, 0.0};
#pragma unroll
        for (int m = 0; m < M; ++m)
#pragma unroll
            for (int k = 0; k < kSmallK; ++k) acc[m] = acc[m] + v[m][k];
        const double t = M == 1 ? wave_sum_63(acc[0]) : wave_sum_two(acc[0], acc[1]);
        if (WAVE) {
            out[0] = lane_value(t, M == 1 ? 63 : 31);
            if (M > 1) out[M - 1] = lane_value(t, 63);
            return;
        }
        const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
        if (M == 1 ? lane == 63 : (lane & 31) == 31) sh[w][M == 1 ? 0 : lane >> 5] = t;
        __syncthreads();
#pragma unroll
        for (int m = 0; m < M; ++m) {
            double a = sh[0][m];
#pragma unroll
            for (int k = 1; k < kWaves; ++k) a = a + sh[k][m];
            out[m] = a;
        }
    }
};

// M sums over the workgroup, in thread 0 (sh: used nowhere else in the kernel)
template <int M>
__device__ inline void small_block_sum(double (&v)[M]) {
    static_assert(M <= 2, "at most two sums");
    __shared__ double sh[kWaves][2];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const double t = M == 1 ? wave_sum_63(v[0]) : wave_sum_two(v[0], v[M - 1]);
    if (M == 1 ? lane == 63 : (lane & 31) == 31) sh[w][M == 1 ? 0 : lane >> 5] = t;
    __syncthreads();
    if (threadIdx.x == 0)
#pragma unroll
        for (int m = 0; m < M; ++m) {
            v[m] = sh[0][m];
#pragma unroll
            for (int k = 1; k < kWaves; ++k) v[m] = v[m] + sh[k][m];
        }
}

// The operand row of the fused kernels, requested ahead where the layout
// lets the kernel know its width (W: as kernel_width).
template <int W, class T>
struct RowPre {
    StencilPre<(W < 0 ? -W : 1), T> st;
    EllPre<(W > 0 ? W : 1), T> el;
    __device__ inline void load(const EllView &A, const T *val, const SP<T> *sp, int row) {
        if constexpr (W < 0)
            stencil_row_pre<(W < 0 ? -W : 1), T>(A, val, sp, row, st);
        else if constexpr (W > 0)
            ell_row_pre<(W > 0 ? W : 1), T>(A, val, sp, row, el);
    }
    __device__ inline bool sum(const EllView &A, const T *val, const DirOperand<T> &x, int row, T &out) const {
        if constexpr (W < 0) {
            return stencil_row_fin<(W < 0 ? -W : 1), T>(A, val, x, row, st, out);
        } else if constexpr (W > 0) {
            out = T(0);
#pragma unroll
            for (int k = 0; k < (W > 0 ? W : 1); ++k)
                out = out + dir_at(el.g[k], el.c[k], x.beta, x.n) * el.v[k];
            return true;
        } else {
            return row_dot<0, T, T>(A, val, x, row, out);
        }
    }
};

// Small operators, k >= 1: K0 and K1 in one kernel over the product's grid
// (one row per thread).  rho_k, the convergence test, x += alpha_{k-1} p_{k-1}
// on the thread's row, p_k = 1.0 s + beta p_{k-1} into the other pairs,
// Ap = A p_k with p_k formed at every column read, and the p_k.Ap
// partials of iteration k (read by K2 of k while this kernel's own
// partials of k-1 stay intact: two partial arrays by parity).
// TOL: a solve with a tolerance (the r.r partials and the convergence
// test); without one (the reference's fixed iteration count) the prologue
// sums the rho partials only.
template <int W, bool TOL, bool WAVE>
__device__ inline void iter_dirprod(const EllView &A, const PcgDev &d, int k) {
    const SP<double> *__restrict__ old = d.sp[(k - 1) & 1];
    const int st = state_load(d.state);
    const int c = xcd_block(blockIdx.x, gridDim.x);
    const int row = c * kBlock + threadIdx.x;
    const bool own = row < d.n;
    double xo = 0.0;
    SP<double> me{0.0, 0.0};
    if (own) {
        xo = d.x[row];
        me = old[row];
    }
    const double tol2 = TOL ? early_load(d.sc + S_TOL2) : -1.0;
    const double rho_prev = early_load(d.sc + S_RHO0 + ((k - 1) & 1));
    const double alpha = early_load(d.sc + S_ALPHA0 + ((k - 1) & 1));  // alpha_{k-1}, as K2 of k-1 formed it (:93)
    constexpr int NS = TOL ? 2 : 1;
    SmallSums<NS, WAVE> ps;
    if constexpr (TOL)
        ps.load({d.P(P_RS), d.P(P_RR)}, d.G);
    else
        ps.load({d.P(P_RS)}, d.G);
    RowPre<W, double> q;
    if (own) q.load(A, A.val, old, row);
    double sums[NS];
    ps.reduce(sums);
    if (st != ST_RUN && st != conv_stamp(k)) return;
    if (TOL && tol2 >= 0.0 && sums[NS - 1] <= tol2) {  // every workgroup reaches the same decision
        if (own) d.x[row] = xo + alpha * me.p;
        if (leader()) state_store(d.state, conv_stamp(k));
        return;
    }
    const double beta = sums[0] / rho_prev;  // :107-109
    if (leader()) d.sc[S_RHO0 + (k & 1)] = sums[0];
    double pr = 0.0, sum = 0.0;
    if (own) {
        d.x[row] = xo + alpha * me.p;    // :95 of iteration k-1
        pr = 1.0 * me.s + beta * me.p;   // :113
        d.sp[k & 1][row].p = pr;
        if (q.sum(A, A.val, DirOperand<double>{old, beta, d.n}, row, sum))  // :87
            d.Ap[row] = sum;
        else
            sum = d.Ap[row];  // empty row: Ap keeps its value
    }
    double acc[1] = {own ? pr * sum : 0.0};
    small_block_sum<1>(acc);
    if (threadIdx.x == 0) dn_part(d, k)[c] = acc[0];
}

template <int W, bool TOL, bool WAVE>
__global__ __launch_bounds__(kBlock) void k_iter_dirprod(EllView A, PcgDev d, int k) {
    iter_dirprod<W, TOL, WAVE>(A, d, k);
}

// the per-wavefront partials of the long products, folded in index order:
// thread i sums chunk i's kWaves partials, each workgroup its 256 chunks
// into one of the Gdn partials of P_DN
__global__ __launch_bounds__(kBlock) void k_fold_dn(PcgDev d) {
    if (!running(d)) return;
    const int i = blockIdx.x * kBlock + threadIdx.x;
    double v = 0.0, sa = 0.0;
    if (i < d.nchunk) {
        const double *w = d.chunk + (size_t)i * d.wpc;
        for (int j = 0; j < d.wpc; ++j) v = v + w[j];
        if (d.deflate) {
            const double *ws = d.chunk_s + (size_t)i * d.wpc;
            for (int j = 0; j < d.wpc; ++j) sa = sa + ws[j];
        }
    }
    if (d.deflate) {
        double red[2] = {v, sa};
        block_reduce_n<2>(red);
        if (threadIdx.x == 0) {
            d.P(P_DN)[blockIdx.x] = red[0];
            d.P(P_SA)[blockIdx.x] = red[1];
        }
    } else {
        v = block_reduce<RED_SUM>(v);
        if (threadIdx.x == 0) d.P(P_DN)[blockIdx.x] = v;
    }
}

// wide_store's partials, of `per` chunks each, from those of the chunks (one
// per chunk).  (Their total from one workgroup instead, so that the update
// reads one number, was slower: FP64 128^3 42.4 / 44.0 us per iteration.)
__global__ __launch_bounds__(kBlock) void k_fold_wide(PcgDev d, int per) {
    if (!running(d)) return;
    const int i = blockIdx.x * kBlock + threadIdx.x, c0 = i * per;
    if (i >= d.Gdn) return;
    double v = 0.0;
    for (int q = 0; q < per; ++q)
        if (c0 + q < d.nchunk) v = v + d.chunk[c0 + q];
    d.P(P_DN)[i] = v;
}

// K2 (operators of at most 2^19 rows): alpha_k, r += (-alpha) Ap, s = Dinv r,
// partials of r.s and r.r; one row per thread, its operands requested before
// the prologue's sums
template <bool WAVE>
__global__ __launch_bounds__(kBlock) void k_iter_update(PcgDev d, int k) {
    const bool precond = d.precond != 0;
    const ThreadRows t(d.n);
    const bool own = t.valid();
    double ro = 0.0, apr = 0.0, di = 0.0;
    const int st = state_load(d.state);
    if (own) {
        ro = d.r[t.row];
        apr = d.Ap[t.row];
        if (precond) di = d.dinv[t.row];
    }
    const double rho = early_load(d.sc + S_RHO0 + (k & 1));
    SmallSums<1, WAVE> ps;
    ps.load({dn_part(d, k)}, d.Gdn);
    double sums[1];
    ps.reduce(sums);
    const double dn = sums[0];
    if (st != ST_RUN) return;
    const double alpha = rho / dn;
    if (dn == 0.0 || !isfinite(dn) || !isfinite(alpha)) {
        if (leader()) state_store(d.state, ST_BREAK);
        return;
    }
    store_alpha(d, k, alpha);
    const double malpha = -1.0 * alpha;
    double red[2] = {0.0, 0.0};
    if (own) {
        const double ri = ro + malpha * apr;  // :97
        d.r[t.row] = ri;
        double si;
        if (precond) {  // :99-105
            si = 0.0;
            si = si + ri * di;
        } else {
            si = ri;
        }
        d.sp[k & 1][t.row].s = si;
        red[0] = ri * si;
        red[1] = ri * ri;
    }
    small_block_sum<2>(red);
    if (threadIdx.x == 0) {
        d.P(P_RS)[blockIdx.x] = red[0];
        d.P(P_RR)[blockIdx.x] = red[1];
    }
    if (leader()) *d.iters = k + 1;
}

// ---- FP64 iteration on mid-size operators (2^19 to kRowsMin rows) ----------
//
// A sweep of 2048 (or fewer) workgroups striding over the rows in
// XCD-contiguous order, whose prologue re-reduces the previous kernel's
// partials (every workgroup forms the same scalars): three or four launches
// per iteration (direction, product, a fold where the product leaves more
// partials than a prologue sums, update).  At these sizes the three
// extra launches of the row-per-thread iteration cost more than its faster
// sweeps save (FP64 solve to 1e-10, grid-stride against row-per-thread:
// 128^3 94.9 against 107.0 ms, 160^3 205.8 / 227.7, 192^3 419.2 / 424.6;
// past the switch 224^3 834.0 / 776.4, 256^3 1418 / 1286).
constexpr int kRowsMin = 1 << 23;

// The x updates of the long iterations (x += alpha_k p_k, :95) are made two
// at a time by the direction sweep of every second iteration, which reads
// p_{k-1} anyway: x is read and written half as often for one more read of
// the direction before (two direction buffers by parity; the older one is
// the one being overwritten).  In order, so the same bits.  Nine streams
// instead of ten per two sweeps.
__device__ inline double x_two(double x, double a2, double p2, double a1, double p1) {
    const double t = x + a2 * p2;  // iteration k-2
    return t + a1 * p1;            // iteration k-1
}

// K0 (k >= 1): rho_k, the convergence test, beta, p_k = 1.0 s + beta p_{k-1}
// into pnew (which holds p_{k-2}); PAIR: the x updates of k-2 and k-1
template <bool LEAN, bool PAIR, int U>
__global__ __launch_bounds__(kBlock) void k_iter_dir(PcgDev d, const double *__restrict__ pold,
                                                    double *__restrict__ pnew, int k) {
    double *__restrict__ x = d.x;
    const double *__restrict__ s = LEAN ? d.r : d.s;
    const int st = state_load(d.state);
    struct In {
        double s, di, po, x, pp;
    };
    const auto load = [&](int row) {
        return In{s[row], LEAN ? dict_dinv(d, row, 0.0) : 0.0, pold[row], PAIR ? x[row] : 0.0, PAIR ? pnew[row] : 0.0};
    };
    AheadSweep<U, 1, decltype(load)> rows(d.n, load);
    rows.ahead();
    const double rho = sum_partials<RED_SUM>(d.P(P_RS), d.G);  // :107
    const double a1 = PAIR ? alpha_slot(d, k - 1) : 0.0, a2 = PAIR ? alpha_slot(d, k - 2) : 0.0;
    const double tol2 = d.sc[S_TOL2];
    if (st != ST_RUN && st != conv_stamp(k)) return;
    if (tol2 >= 0.0) {
        const double rr = sum_partials<RED_SUM>(d.P(P_RR), d.G);
        if (rr <= tol2) {  // every workgroup reaches the same decision
            if (leader()) state_store(d.state, conv_stamp(k));
            return;
        }
    }
    const double beta = rho / rho_slot(d, k - 1);  // :109
    if (leader()) d.sc[S_RHO0 + (k & 1)] = rho;
    rows.each([&](int row, const In &v) {
        const double si = LEAN ? s_of(v.s, v.di, d.precond != 0) : v.s;
        if (PAIR) x[row] = x_two(v.x, a2, v.pp, a1, v.po);
        pnew[row] = 1.0 * si + beta * v.po;  // :113
    });
}

// K2: alpha_k from the folded p.Ap partials, r += (-alpha) Ap, s = Dinv r,
// partials of r.s and r.r (one per workgroup); each row's operands are
// loaded together (one round trip per row)
template <bool LEAN, int U>
__global__ __launch_bounds__(kBlock) void k_iter_update_grid(PcgDev d, int k) {
    const int st = state_load(d.state);
    double *__restrict__ r = d.r, *__restrict__ s = d.s;
    const double *__restrict__ Ap = d.Ap, *__restrict__ dinv = d.dinv;
    const bool precond = d.precond != 0;
    struct In {
        double r, ap, di;
    };
    const auto load = [&](int row) {
        return In{r[row], Ap[row], LEAN ? dict_dinv(d, row, 0.0) : precond ? dinv[row] : 0.0};
    };
    AheadSweep<U, kSweepU<LEAN>, decltype(load)> rows(d.n, load);
    rows.ahead();
    double dsum[1];
    if (d.Gdn <= kBlock)  // one round of the uniform loop
        sum_partials_n<1>({d.P(P_DN)}, d.Gdn, dsum);
    else
        dsum[0] = sum_partials<RED_SUM>(d.P(P_DN), d.Gdn);
    const double dn = dsum[0];
    if (st != ST_RUN) return;
    const double alpha = rho_slot(d, k) / dn;  // :93
    if (dn == 0.0 || !isfinite(dn) || !isfinite(alpha)) {
        if (leader()) state_store(d.state, ST_BREAK);
        return;
    }
    store_alpha(d, k, alpha);
    const double malpha = -1.0 * alpha;
    double rs = 0.0, rr = 0.0;
    rows.each([&](int row, const In &v) {
        const double ri = v.r + malpha * v.ap;  // :97
        r[row] = ri;
        const double si = s_of(ri, v.di, precond);
        if (!LEAN) s[row] = si;
        rs = rs + ri * si;
        rr = rr + ri * ri;
    });
    double red[2] = {rs, rr};
    block_reduce_n<2>(red);
    if (threadIdx.x == 0) {
        d.P(P_RS)[blockIdx.x] = red[0];
        d.P(P_RR)[blockIdx.x] = red[1];
    }
    if (leader()) *d.iters = k + 1;
}

// ---- FP64 iteration on long operators (more than kRowsMin rows) -------------
//
// One row per thread over the whole operator, workgroups in dispatch order
// (consecutive 256-row chunks on consecutive XCDs, the whole chip streaming
// one narrow window of every array): the direction and update sweeps run
// at the pace of a plain stream of their access mix.  So many workgroups
// cannot each re-reduce the previous kernel's partials, so the scalars come
// from one-workgroup kernels instead:
//   K0  p = 1.0 s + beta p, x by two directions in turn (beta, alphas from slots)
//   K1  Ap = A p, per-wavefront p.Ap partials          (iter_spmv)
//   fold + F1: alpha = rho_k / (p.Ap)                  (breakdown test)
//   K2  r += (-alpha) Ap, s = Dinv r, per-wavefront r.s and r.r partials
//   fold + F2: rho_{k+1}, r.r, the convergence test, beta
// F2 stamps a convergence with the next iteration's index; the final flush
// then applies the x updates still due.

__device__ inline double ntload(const double *p) { return __builtin_nontemporal_load(p); }
__device__ inline void ntstore(double *p, double v) { __builtin_nontemporal_store(v, p); }

// K0 of iteration k >= 1 (as k_iter_dir)
template <bool LEAN, bool PAIR>
__global__ __launch_bounds__(kBlock) void k_iter_dir_rows(PcgDev d, const double *__restrict__ pold,
                                                         double *__restrict__ pnew, int k) {
    if (!running(d)) return;
    const int row = blockIdx.x * kBlock + threadIdx.x;
    if (row >= d.n) return;
    const double a1 = PAIR ? alpha_slot(d, k - 1) : 0.0, a2 = PAIR ? alpha_slot(d, k - 2) : 0.0;
    const double beta = d.sc[S_BETA];
    // nontemporal accesses: each array is streamed once per sweep (a plain
    // stream of this mix runs 8% faster with them on this device)
    const double sr = ntload((LEAN ? d.r : d.s) + row), po = ntload(pold + row);
    const double xo = PAIR ? ntload(d.x + row) : 0.0, pp = PAIR ? ntload(pnew + row) : 0.0;
    const double si = LEAN ? s_of(sr, dict_dinv(d, row, 0.0), d.precond != 0) : sr;
    if (PAIR) ntstore(d.x + row, x_two(xo, a2, pp, a1, po));
    ntstore(pnew + row, 1.0 * si + beta * po);  // :113
}

// the `per` partials of each of the nwg workgroups of a sweep (a, and b
// where not null), folded in index order into one partial per workgroup of
// this kernel, arrays ia and ib
__global__ __launch_bounds__(kBlock) void k_fold_two(PcgDev d, int nwg, int per, const double *__restrict__ a,
                                                    const double *__restrict__ b, int ia, int ib) {
    if (!running(d)) return;
    const int i = blockIdx.x * kBlock + threadIdx.x;
    double va = 0.0, vb = 0.0;
    if (i < nwg) {
        for (int j = 0; j < per; ++j) va = va + a[(size_t)i * per + j];
        if (b)
            for (int j = 0; j < per; ++j) vb = vb + b[(size_t)i * per + j];
    }
    double red[2] = {va, vb};
    block_reduce_n<2>(red);
    if (threadIdx.x == 0) {
        d.P(ia)[blockIdx.x] = red[0];
        if (b) d.P(ib)[blockIdx.x] = red[1];
    }
}

// F1 (one workgroup): alpha_k = rho_k / p.Ap, or a breakdown
__device__ inline void alpha_finish(const PcgDev &d, int k, double dn) {
    const double alpha = rho_slot(d, k) / dn;  // :93
    if (dn == 0.0 || !isfinite(dn) || !isfinite(alpha))
        state_store(d.state, ST_BREAK);
    else
        d.sc[S_ALPHA0 + (k & 1)] = alpha;
}

__global__ __launch_bounds__(kBlock) void k_alpha_fin(PcgDev d, int k) {
    if (!running(d)) return;
    const double dn = sum_partials<RED_SUM>(d.P(P_DN), d.Gdn);
    if (threadIdx.x == 0) alpha_finish(d, k, dn);
}

// K2 of iteration k: kUpdateRows slices per wavefront, their loads in flight
// together and their rows summed before the wavefront's two sums, which
// with one slice and two separate sums held the kernel to 4.7 TB/s (256^3
// with a dictionary: 86 -> 61 us, 6.6 TB/s; FP64 iteration at 256^3
// clustered 428 -> 421 us).
constexpr int kUpdateRows = 2;
template <bool LEAN>
__global__ __launch_bounds__(kBlock) void k_iter_update_rows(PcgDev d, int k) {
    if (!running(d)) return;
    const int wv = blockIdx.x * kWaves + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    const double malpha = -1.0 * alpha_slot(d, k);
    double rs = 0.0, rr = 0.0, ro[kUpdateRows], apr[kUpdateRows], di[kUpdateRows];
#pragma unroll
    for (int u = 0; u < kUpdateRows; ++u) {
        const int at = (wv * kUpdateRows + u) * 64 + lane, row = at < d.n ? at : d.n - 1;
        ro[u] = ntload(d.r + row);
        apr[u] = ntload(d.Ap + row);
        di[u] = !d.precond ? 0.0 : LEAN ? dict_one(d.dc_sel, d.dc_id, d.ddinv, row) : ntload(d.dinv + row);
    }
#pragma unroll
    for (int u = 0; u < kUpdateRows; ++u) {
        const int row = (wv * kUpdateRows + u) * 64 + lane;
        const double ri = ro[u] + malpha * apr[u];  // :97
        double si;
        if (d.precond) {  // :99-105
            si = 0.0;
            si = si + ri * di[u];
        } else {
            si = ri;
        }
        if (row < d.n) {
            ntstore(d.r + row, ri);
            if (!LEAN) ntstore(d.s + row, si);
            rs = rs + ri * si;
            rr = rr + ri * ri;
        }
    }
    // one partial per wavefront: no barrier
    const double t = wave_sum_two(rs, rr);
    if (lane == 31) d.chunk[wv] = t;
    if (lane == 63) d.chunk_s[wv] = t;
    if (leader()) *d.iters = k + 1;
}

// F2 (one workgroup) after K2 of iteration k - 1: rho_k, r.r, the
// convergence test (stamped with k), beta_k
__device__ inline void beta_finish(const PcgDev &d, int k, double rho, double rr) {
    const double tol2 = d.sc[S_TOL2];
    d.sc[S_RR] = rr;
    if (tol2 >= 0.0 && rr <= tol2) {
        state_store(d.state, conv_stamp(k));
        return;
    }
    d.sc[S_BETA] = rho / rho_slot(d, k - 1);  // :107-111
    d.sc[S_RHO0 + (k & 1)] = rho;
}

__global__ __launch_bounds__(kBlock) void k_beta_fin(PcgDev d, int k, int np) {
    if (!running(d)) return;
    double sums[2];
    sum_partials_n<2>({d.P(P_RS), d.P(P_RR)}, np, sums);
    if (threadIdx.x == 0) beta_finish(d, k, sums[0], sums[1]);
}


// The x updates still due when a long solve has stopped: of its `iters`
// iterations K0 of every even iteration k >= 2 has applied those before k
// (after a breakdown in iteration `iters`, whose K0 ran, that one's too).
// Directions by parity in pa (even) and pb.
__global__ __launch_bounds__(kBlock) void k_x_flush_pair(PcgDev d, const double *__restrict__ pa,
                                                        const double *__restrict__ pb) {
    const int it = *d.iters;
    if (it < 1) return;
    const bool broke = (state_load(d.state) & ST_MASK) == ST_BREAK;
    if (broke && !(it & 1)) return;
    const bool two = !(it & 1);
    const double a1 = alpha_slot(d, it - 1), a2 = two ? alpha_slot(d, it - 2) : 0.0;
    const double *__restrict__ p1 = ((it - 1) & 1) ? pb : pa;
    FOR_ROWS(d.n, row) {
        double x = d.x[row];
        if (two) x = x + a2 * pa[row];
        d.x[row] = x + a1 * p1[row];
    }
}

// one workgroup after the last iteration: the final convergence test on the
// r.r F2 left
__global__ __launch_bounds__(kBlock) void k_fin_rows(PcgDev d, Pub pub) {
    if (threadIdx.x == 0) {
        const double rr = d.sc[S_RR], tol2 = d.sc[S_TOL2];
        const int st = state_load(d.state);
        if ((st == ST_RUN || (st & ST_MASK) == ST_CONV) && tol2 >= 0.0 && rr <= tol2) state_store(d.state, ST_CONV);
    }
    publish(d, pub);
}

// one workgroup after the last iteration: r.r and the final convergence test
__global__ __launch_bounds__(kBlock) void k_fin(PcgDev d, Pub pub) {
    const double rr = sum_partials<RED_SUM>(d.P(P_RR), d.G);
    if (threadIdx.x == 0) {
        d.sc[S_RR] = rr;
        const double tol2 = d.sc[S_TOL2];
        if (state_load(d.state) == ST_RUN && tol2 >= 0.0 && rr <= tol2) state_store(d.state, ST_CONV);
    }
    publish(d, pub);
}

// ---- MIXED iteration (FP32 vectors and operator, FP64 dot accumulation) --------

// K0 (k >= 1): rho_k, beta (0 after a restart: the previous rho slot is
// +inf), p32 = s32 + beta p32 into pnew; PAIR: the correction updates
// xc += alpha p of iterations k-2 and k-1 (not yet folded by a defect
// correction), two at a time as in k_iter_dir
template <bool LEAN, bool PAIR, int U>
__global__ __launch_bounds__(kBlock) void k_m_dir(PcgDev d, const float *__restrict__ pold, float *__restrict__ pnew,
                                                 int k) {
    float *__restrict__ xc = d.xc32;
    const float *__restrict__ s = LEAN ? d.r32 : d.s32;
    const int st = state_load(d.state);
    struct In {
        float s, di, po, x, pp;
    };
    // nontemporal accesses: each array is streamed once per sweep (mixed
    // solve at 256^3 over four runs: 392-394 ms with them, 403-405 without;
    // the sweeps' own times are unchanged within noise)
    const auto load = [&](int row) {
        return In{__builtin_nontemporal_load(s + row), LEAN ? dict_dinv(d, row, 0.0f) : 0.0f,
                  __builtin_nontemporal_load(pold + row), PAIR ? __builtin_nontemporal_load(xc + row) : 0.0f,
                  PAIR ? __builtin_nontemporal_load(pnew + row) : 0.0f};
    };
    AheadSweep<U, 1, decltype(load)> rows(d.n, load);
    rows.ahead();
    const double rho = sum_partials<RED_SUM>(d.P(P_RS), d.G);
    const float a1 = PAIR ? (float)alpha_slot(d, k - 1) : 0.0f;  // as K2 formed them
    const float a2 = PAIR ? (float)alpha_slot(d, k - 2) : 0.0f;
    if (st != ST_RUN) return;
    const float beta = (float)(rho / rho_slot(d, k - 1));
    if (leader()) d.sc[S_RHO0 + (k & 1)] = rho;
    rows.each([&](int row, const In &v) {
        const float si = LEAN ? s_of(v.s, v.di, d.precond != 0) : v.s;
        if (PAIR) {
            const float t = v.x + a2 * v.pp;
            __builtin_nontemporal_store(t + a1 * v.po, xc + row);
        }
        __builtin_nontemporal_store(si + beta * v.po, pnew + row);
    });
}

// Small operators, k >= 1: k_m_dir and the FP32 product in one kernel (as
// iter_dirprod)
template <int W, bool WAVE>
__global__ __launch_bounds__(kBlock) void k_m_dirprod(EllView A, PcgDev d, int k, int pending) {
    const SP<float> *__restrict__ old = d.sp32[(k - 1) & 1];
    const int st = state_load(d.state);
    const int c = xcd_block(blockIdx.x, gridDim.x);
    const int row = c * kBlock + threadIdx.x;
    const bool own = row < d.n;
    float xo = 0.0f;
    SP<float> me{0.0f, 0.0f};
    if (own) {
        xo = d.xc32[row];
        me = old[row];
    }
    const double rho_prev = early_load(d.sc + S_RHO0 + ((k - 1) & 1));
    const double alpha = early_load(d.sc + S_ALPHA0 + ((k - 1) & 1));  // alpha_{k-1}, as K2 of k-1 formed it
    SmallSums<1, WAVE> ps;
    ps.load({d.P(P_RS)}, d.G);
    RowPre<W, float> q;
    if (own) q.load(A, A.val32, old, row);
    double sums[1];
    ps.reduce(sums);
    if (st != ST_RUN) return;
    const float a32 = pending ? (float)alpha : 0.0f;
    const float beta = (float)(sums[0] / rho_prev);
    if (leader()) d.sc[S_RHO0 + (k & 1)] = sums[0];
    double red[2] = {0.0, 0.0};
    if (own) {
        if (pending) d.xc32[row] = xo + a32 * me.p;
        const float pr = me.s + beta * me.p;
        d.sp32[k & 1][row].p = pr;
        float sum;
        q.sum(A, A.val32, DirOperand<float>{old, beta, d.n}, row, sum);
        d.Ap32[row] = sum;
        red[0] = (double)pr * (double)sum;
        red[1] = (double)sum;
    }
    small_block_sum<2>(red);
    if (threadIdx.x == 0) {
        dn_part(d, k)[c] = red[0];
        sa_part(d, k)[c] = red[1];
    }
}

// K1 in FP32 (the symmetric form of the slot values measured slower here,
// 121-131 against 118.5 us at 256^3, so the FP32 product keeps the full slot
// values).  No state test: the product's stores (Ap32, its partials) are
// read only by the fold and the update, which test it; and mixed iterations
// are queued only while the solve runs (convergence is decided at a defect
// correction, after which nothing is queued).
template <int W, int NB>
__global__ __launch_bounds__(NB) void k_m_spmv(EllView A, PcgDev d, const float *__restrict__ p) {
    const int c = xcd_block(blockIdx.x, gridDim.x);
    const int row = c * NB + threadIdx.x;
    double acc = 0.0, sa = 0.0;
    if (row < d.n) {
        // (a SelfOperand here measured 9% slower than the separate load)
        Operand<float> po{p};
        const float pr = p[row];
        float sum;
        row_dot<W, float, float>(A, A.val32, po, row, sum);
        d.Ap32[row] = sum;
        acc = (double)pr * (double)sum;
        sa = (double)sum;
    }
    const int lane = threadIdx.x & 63;
    acc = wave_sum_two(acc, sa);
    if constexpr (NB > kBlock) {
        __shared__ double sh[NB / 64][2];
        if ((lane & 31) == 31) sh[threadIdx.x >> 6][lane >> 5] = acc;
        wide_store(d, c, sh);
    } else {
        const int wv = c * kWaves + (threadIdx.x >> 6);
        if (lane == 31) d.chunk[wv] = acc;
        if (lane == 63) d.chunk_s[wv] = acc;
    }
}

// the first product of a small operator (as k_iter_spmv_small)
template <int W>
__global__ __launch_bounds__(kBlock) void k_m_spmv_small(EllView A, PcgDev d) {
    const int st = state_load(d.state);
    const int c = xcd_block(blockIdx.x, gridDim.x);
    const int row = c * kBlock + threadIdx.x;
    float pr = 0.0f, sum = 0.0f;
    if (row < d.n) {
        const PairOperand<float> po{d.sp32[0]};
        pr = po.at(row);
        row_dot<W, float, float>(A, A.val32, po, row, sum);
    }
    if (st != ST_RUN) return;
    double acc = 0.0, sa = 0.0;
    if (row < d.n) {
        d.Ap32[row] = sum;
        acc = (double)pr * (double)sum;
        sa = (double)sum;
    }
    double red[2] = {acc, sa};
    block_reduce_n<2>(red);
    if (threadIdx.x == 0) {
        d.chunk[c] = red[0];
        if (d.deflate) sa_part(d, 0)[c] = red[1];
    }
}

// (as k_iter_spmv_dict)
template <int SW, int R>
__global__ __launch_bounds__(kBlock) void k_m_spmv_dict(EllView A, PcgDev d, const float *__restrict__ p) {
    __shared__ double sh[4 * R][2];
    dict_rows<true, R, SW, float, float>(A, A.val32, d.n, p, [&](int row, bool ok, bool, float sum, float own) {
        if (ok) d.Ap32[row] = sum;
        const int lane = threadIdx.x & 63;
        const double acc = wave_sum_two(ok ? (double)own * (double)sum : 0.0, ok ? (double)sum : 0.0);
        if ((lane & 31) == 31) sh[(row >> 6) & (4 * R - 1)][lane >> 5] = acc;
    });
    chunk_store<R, 2>(d, sh);
}

template <bool LEAN, int U>
__global__ __launch_bounds__(kBlock) void k_m_update(PcgDev d, int k) {
    float *__restrict__ r = d.r32, *__restrict__ s = d.s32;
    const float *__restrict__ Ap = d.Ap32, *__restrict__ dinv = d.dinv32;
    const bool precond = d.precond != 0;
    double rs = 0.0, rr = 0.0;
    const int st = state_load(d.state);
    struct In {
        float r, ap, di;
    };
    const auto load = [&](int row) {
        return In{__builtin_nontemporal_load(r + row), __builtin_nontemporal_load(Ap + row),
                  LEAN      ? dict_dinv(d, row, 0.0f)
                  : precond ? __builtin_nontemporal_load(dinv + row)
                            : 0.0f};
    };
    AheadSweep<U, kSweepU<LEAN>, decltype(load)> rows(d.n, load);
    rows.ahead();
    // every prologue load issued before the first is used: 1.A1, the
    // list of A 1's nonzeros, and the p.Ap and 1.Ap partials (summed
    // together; alpha goes to its scalar slot, so later kernels need
    // not reproduce this sum)
    const double zaz = d.sc[S_ZAZ];
    const int naz_all = d.azl->count;
    int li[kAzList];
    float lv[kAzList];
#pragma unroll
    for (int j = 0; j < kAzList; ++j) {
        li[j] = d.azl->idx[j];
        lv[j] = d.azl->val[j];
    }
    double sums[2];
    if (d.Gdn <= kBlock)  // one round of the uniform loop (up to 256^3)
        sum_partials_n<2>({d.P(P_DN), d.P(P_SA)}, d.Gdn, sums);
    else  // all slots in one round trip
        sum_padded<2>({d.P(P_DN), d.P(P_SA)}, {d.Gdn, d.Gdn}, sums);
    if (st != ST_RUN) return;
    const bool dfl = deflating(d, zaz);
    const double sap = dfl ? sums[1] : 0.0;
    const double dn = m_denom(sums[0], sap, zaz, dfl);
    const double alpha = rho_slot(d, k) / dn;
    if (dn == 0.0 || !isfinite(dn) || !isfinite(alpha)) {
        if (leader()) state_store(d.state, ST_BREAK);
        return;
    }
    store_alpha(d, k, alpha);
    const float a32 = (float)alpha, c32 = dfl ? (float)(sap / zaz) : 0.0f;
    const float *__restrict__ az = d.az32;
    // A 1 from its list of nonzeros when it is short (the same values
    // as the dense array, without streaming it), else row by row
    const int naz = dfl ? naz_all : 0;
    const bool listed = naz <= kAzList;
#pragma unroll
    for (int j = 0; j < kAzList; ++j) li[j] = j < naz ? li[j] : -1;
    rows.each(
        [&](int row, const In &v) {
            float azr = 0.0f;
            if (dfl && !listed) {
                azr = az[row];
            } else {
                // rows compared with the list only in a chunk that holds a
                // listed row (a workgroup-uniform test per chunk)
                const int base = __builtin_amdgcn_readfirstlane(row - (int)threadIdx.x);
                bool hit = false;
#pragma unroll
                for (int j = 0; j < kAzList; ++j) hit = hit || (unsigned)(li[j] - base) < (unsigned)kBlock;
                if (hit)
#pragma unroll
                    for (int j = 0; j < kAzList; ++j) azr = row == li[j] ? lv[j] : azr;
            }
            const float wr = dfl ? v.ap - c32 * azr : v.ap;  // (P A p)_row
            const float ri = v.r - a32 * wr;
            __builtin_nontemporal_store(ri, r + row);
            const float si = precond ? ri * v.di : ri;
            if (!LEAN) __builtin_nontemporal_store(si, s + row);
            rs = rs + (double)ri * (double)si;
            rr = rr + (double)ri * (double)ri;
        });
    double red[2] = {rs, rr};
    block_reduce_n<2>(red);
    if (threadIdx.x == 0) {
        d.P(P_RS)[blockIdx.x] = red[0];
        d.P(P_RR)[blockIdx.x] = red[1];
    }
    if (leader()) *d.iters = k + 1;
}

// the update of a small operator (as k_iter_update)
template <bool WAVE>
__global__ __launch_bounds__(kBlock) void k_m_update_small(PcgDev d, int k) {
    const bool precond = d.precond != 0, want_az = d.deflate != 0;
    const ThreadRows t(d.n);
    const bool own = t.valid();
    float ro = 0.0f, apr = 0.0f, di = 0.0f, azr = 0.0f;
    const int st = state_load(d.state);
    if (own) {
        ro = d.r32[t.row];
        apr = d.Ap32[t.row];
        if (precond) di = d.dinv32[t.row];
        if (want_az) azr = d.az32[t.row];
    }
    const double rho = early_load(d.sc + S_RHO0 + (k & 1));
    const double zaz = early_load(d.sc + S_ZAZ);
    SmallSums<2, WAVE> ps;
    ps.load({dn_part(d, k), sa_part(d, k)}, d.Gdn);
    double sums[2];
    ps.reduce(sums);
    if (st != ST_RUN) return;
    const bool dfl = deflating(d, zaz);
    const double dn = m_denom(sums[0], sums[1], zaz, dfl);
    const double alpha = rho / dn;
    if (dn == 0.0 || !isfinite(dn) || !isfinite(alpha)) {
        if (leader()) state_store(d.state, ST_BREAK);
        return;
    }
    store_alpha(d, k, alpha);
    const float a32 = (float)alpha, c32 = dfl ? (float)(sums[1] / zaz) : 0.0f;
    double red[2] = {0.0, 0.0};
    if (own) {
        const float wr = dfl ? apr - c32 * azr : apr;  // (P A p)_row
        const float ri = ro - a32 * wr;
        d.r32[t.row] = ri;
        const float si = precond ? ri * di : ri;
        d.sp32[k & 1][t.row].s = si;
        red[0] = (double)ri * (double)si;
        red[1] = (double)ri * (double)ri;
    }
    small_block_sum<2>(red);
    if (threadIdx.x == 0) {
        d.P(P_RS)[blockIdx.x] = red[0];
        d.P(P_RR)[blockIdx.x] = red[1];
    }
    if (leader()) *d.iters = k + 1;
}

// the replaced s of a correction (or of the start, with the first direction
// p = s and a zero correction) into the pairs that the next iteration reads
__global__ __launch_bounds__(kBlock) void k_m_pairs(PcgDev d, SP<float> *__restrict__ sp, int first) {
    FOR_ROWS(d.n, row) {
        const float s = d.s32[row];
        sp[row].s = s;
        if (first) {
            sp[row].p = s;
            d.xc32[row] = 0.0f;
        }
    }
}

// k_m_fold of a small operator
__global__ __launch_bounds__(kBlock) void k_m_fold_small(PcgDev d, int k) {
    const float a32 = (float)alpha_slot(d, k);
    const SP<float> *__restrict__ sp = d.sp32[k & 1];
    FOR_ROWS(d.n, row) {
        const float xcv = d.xc32[row] + a32 * sp[row].p;
        d.x[row] = d.x[row] + (double)xcv;
        d.xc32[row] = 0.0f;
    }
}

// one workgroup: the FP32 recursive r.r for the host's correction test
__global__ __launch_bounds__(kBlock) void k_m_status(PcgDev d, Pub pub) {
    const double rr = sum_partials<RED_SUM>(d.P(P_RR), d.G);
    if (threadIdx.x == 0) d.sc[S_RR] = rr;
    publish(d, pub);
}

// x += xc, with the last iterations' pending updates xc += alpha p first
// (two: those of k-1 in p2 and k in p; one: that of k), xc = 0
__global__ __launch_bounds__(kBlock) void k_m_fold(PcgDev d, const float *__restrict__ p, const float *__restrict__ p2,
                                                  int k, int pending) {
    const float a1 = (float)alpha_slot(d, k), a2 = pending > 1 ? (float)alpha_slot(d, k - 1) : 0.0f;
    FOR_ROWS(d.n, row) {
        float xcv = d.xc32[row];
        if (pending > 1) xcv = xcv + a2 * p2[row];
        if (pending) xcv = xcv + a1 * p[row];
        d.x[row] = d.x[row] + (double)xcv;
        d.xc32[row] = 0.0f;
    }
}

// Defect correction, part 1: r = b - A x in FP64 (empty rows: x) and the
// partials of 1.r.
template <int W>
__global__ __launch_bounds__(kBlock) void k_m_resid(EllView A, PcgDev d) {
    double sr = 0.0;
    Operand<double> xo{d.x};
    FOR_ROWS(d.n, row) {
        double sum;
        bool any = row_dot<W, double, double>(A, A.val, xo, row, sum);
        double t = any ? sum : d.x[row];
        double ri = d.b[row] + -1.0 * t;
        d.r[row] = ri;
        sr = sr + ri;
    }
    sr = block_reduce<RED_SUM>(sr);
    if (threadIdx.x == 0) d.P(P_SUMR)[blockIdx.x] = sr;
}

// Part 2: the coarse step c = (1.r)/(1.A1) (skipped when off, or when 1.A1
// is not positive and finite): x += c, r -= c A1 on the solved rows; then
// r32 = r, s32 = Dinv r32, partials of r32.s32 and of the true r.r.
__global__ __launch_bounds__(kBlock) void k_m_coarse(PcgDev d, int use) {
    const double sr = sum_partials<RED_SUM>(d.P(P_SUMR), d.G);
    const double zaz = d.sc[S_ZAZ];
    double c = (use && zaz > 0.0 && isfinite(zaz)) ? sr / zaz : 0.0;
    if (!isfinite(c)) c = 0.0;
    double rs = 0.0, rr = 0.0;
    FOR_ROWS(d.n, row) {
        double ri = d.r[row];
        if (c != 0.0) {
            d.x[row] = d.x[row] + c;
            ri = ri - c * d.az[row];
            d.r[row] = ri;
        }
        float r32 = (float)ri;
        d.r32[row] = r32;
        float s32 = d.precond ? r32 * d.dinv32[row] : r32;
        d.s32[row] = s32;
        rs = rs + (double)r32 * (double)s32;
        rr = rr + ri * ri;
    }
    double red[2] = {rs, rr};
    block_reduce_n<2>(red);
    if (threadIdx.x == 0) {
        d.P(P_RS2)[blockIdx.x] = red[0];
        d.P(P_RR2)[blockIdx.x] = red[1];
    }
}

// One workgroup after k_m_resid: the replaced residual becomes the
// recursion's (its partials are copied over the FP32 ones); the direction is
// kept unless the recursive r.r had drifted below a hundredth of the true
// one, then the previous rho slot is set to +inf so the next beta is 0.
__global__ __launch_bounds__(kBlock) void k_m_corr_fin(PcgDev d, int k, int first, Pub pub) {
    const double rrt = sum_partials<RED_SUM>(d.P(P_RR2), d.G);
    const double rrec = first ? 0.0 : sum_partials<RED_SUM>(d.P(P_RR), d.G);
    __syncthreads();
    for (int i = threadIdx.x; i < d.G; i += kBlock) {
        d.P(P_RS)[i] = d.P(P_RS2)[i];
        d.P(P_RR)[i] = d.P(P_RR2)[i];
    }
    const double rs = first ? sum_partials<RED_SUM>(d.P(P_RS2), d.G) : 0.0;
    if (threadIdx.x == 0) {
        if (first) d.sc[S_RHO0] = rs;  // rho of iteration 0
        if (!first && rrt > 100.0 * rrec) d.sc[S_RHO0 + ((k - 1) & 1)] = INFINITY;
        d.sc[S_TRUE_RR] = rrt;
        d.sc[S_RR] = rrt;
        const double tol2 = d.sc[S_TOL2];
        if (state_load(d.state) == ST_RUN && tol2 >= 0.0 && rrt <= tol2) state_store(d.state, ST_CONV);
    }
    publish(d, pub);
}

// first direction p32 = s32, correction zero
__global__ __launch_bounds__(kBlock) void k_m_start(PcgDev d, float *__restrict__ p) {
    FOR_ROWS(d.n, row) {
        p[row] = d.s32[row];
        d.xc32[row] = 0.0f;
    }
}

__global__ __launch_bounds__(kBlock) void k_to32(int n, const double *__restrict__ a, float *__restrict__ b) {
    int i = blockIdx.x * kBlock + threadIdx.x;
    if (i < n) b[i] = (float)a[i];
}

__global__ __launch_bounds__(kBlock) void k_tuple_inv(int n, const double *__restrict__ diag, double *__restrict__ inv,
                                                      float *__restrict__ inv32) {
    const int i = blockIdx.x * kBlock + threadIdx.x;
    if (i >= n) return;
    const double v = 1.0 / diag[i];
    inv[i] = v;
    inv32[i] = (float)v;
}

// z = 1 on rows [0, n), 0 on [n, n_all); az = 0 on [0, n)
__global__ __launch_bounds__(kBlock) void k_ones(int n, int n_all, double *__restrict__ z, double *__restrict__ az,
                                                 AzList *azl) {
    int i = blockIdx.x * kBlock + threadIdx.x;
    if (i < n_all) z[i] = i < n ? 1.0 : 0.0;
    if (i < n) az[i] = 0.0;
    if (i == 0) azl->count = 0;
}

// az32 = (float) az, and the list of its nonzeros (entries past kAzList
// are only counted; the order of the entries does not matter, each row
// matches at most one)
__global__ __launch_bounds__(kBlock) void k_az32(int n, const double *__restrict__ az, float *__restrict__ az32,
                                                 AzList *azl) {
    const int i = blockIdx.x * kBlock + threadIdx.x;
    if (i >= n) return;
    const float v = (float)az[i];
    az32[i] = v;
    if (v != 0.0f) {
        const int slot = atomicAdd(&azl->count, 1);
        if (slot < kAzList) {
            azl->idx[slot] = i;
            azl->val[slot] = v;
        }
    }
}

// ---- the solve without allocations -------------------------------------------
//
// The workspace of one FP64 solve on an operator of at most kScratchRows
// rows lives in `scratch`, a file-scope device array (one copy per GPU, held
// until the process ends): r, Ap, Dinv (kScratchRows doubles each), the
// two arrays of pairs (s, p) (kScratchAll pairs each), the partial-sum arrays, the
// scalars and the state words.  Host code never passes `scratch` itself
// (in host code the name is a stand-in, not a device address): gip_init
// looks up its address on each device with hipGetSymbolAddress and keeps it
// in g_scratch, and the entry point builds its workspace from that pointer.
// Every call on a GPU shares its array; what must start at zero is cleared
// by a kernel at the start of each call, so calls that overlap on one GPU
// race.
constexpr int kScratchRows = 1 << 18;
constexpr int kScratchAll = (1 << 18) + (1 << 16);
constexpr size_t kScratchZero = (size_t)P_COUNT * kMaxRedBlocks + S_COUNT + 1;  // partials, scalars, state words
constexpr size_t kScratchDoubles = 3 * (size_t)kScratchRows + 4 * (size_t)kScratchAll + kScratchZero;
static __device__ __align__(256) double scratch[kScratchDoubles];
constexpr int kScratchDevices = 64;
static double *g_scratch[kScratchDevices];
static std::mutex g_scratch_mu;

// Called by gip_init with `device` current.
int pcg_scratch_setup(int device) {
    if (device < 0 || device >= kScratchDevices) return GIP_OK;  // no no-alloc solves on this device
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    if (g_scratch[device]) return GIP_OK;
    double *ptr = nullptr;
    GIP_HIP_TRY(hipGetSymbolAddress((void **)&ptr, HIP_SYMBOL(scratch)));
    g_scratch[device] = ptr;
    return GIP_OK;
}

__global__ __launch_bounds__(kBlock) void k_zero(size_t n, double *__restrict__ a) {
    const size_t i = (size_t)blockIdx.x * kBlock + threadIdx.x;
    if (i < n) a[i] = 0.0;
}

}  // namespace gip

using namespace gip;

struct gip_pcg {
    gip_ctx *ctx;
    const gip_mat *A;
    int n, n_all, grid;
    double *r, *p, *s, *Ap, *dinv;  // small operators: p and p2 are arrays of pairs (s, p), no s
    float *r32, *p32, *s32, *Ap32, *xc32, *dinv32;
    double *p2;   // second direction buffer (directions alternate by parity)
    float *p32b;  // its FP32 counterpart
    double *ddinv;   // the Jacobi inverse per tuple of the operator's dictionary
    float *ddinv32;  // (FP64, FP32), made from dictionary `dict_version`
    uint64_t dict_version;
    double *az;   // A 1 (MIXED coarse step)
    float *az32;  // its FP32 copy (MIXED deflation)
    AzList *azl;  // the FP32 copy's nonzeros, when few
    double *sc, *part, *chunk;
    int nchunk, gdn;
    bool fold;  // nchunk > kMaxRedBlocks: the chunk partials need the fold kernel;
                // otherwise the fused two-kernel iteration runs
    bool rows;  // fold and more than kRowsMin rows: the row-per-thread iteration
    int *state;    // state, iters
    // pinned coherent words the kernels publish to: scalars, then state and
    // count, and the sequence word; their device address; the last number
    double *h_pub, *h_pub_dev;
    uint64_t *h_flag, *h_flag_dev, *seq;
    uint64_t own_seq;
    hipEvent_t tev0, tev1;  // time_products: the sampled product launch
};

// Multiple of 8 (one share per XCD), at most kMaxRedBlocks (one partial each).
// The product kernels run one workgroup per 256-row chunk instead.
// Rows a thread of a mid-size sweep has, all requested before the prologue
// (AheadSweep); 0, one (small operators) or as many as come.  512 to 1024
// workgroups, two to four per CU, each with all its rows in flight, need a
// quarter of the prologues that 2048 workgroups of one or two rows repeat
// and leave no half-empty round.  us per iteration with 2048 workgroups, 4,
// 6 and 8 rows ahead: mixed 81^3 24.5 / 19.5 / 20.3 / 20.5, 97^3 28.4 / 24.1
// / 24.1 / 23.9, 112^3 35.5 / 34.5 / 31.4 / 30.9, 128^3 39.4 / - / - / 34.5;
// FP64 81^3 26.8 / 24.5 / 25.5 / 27.1, 97^3 31.9 / 30.0 / 31.0 / 32.3, 112^3
// 39.4 / 39.0 / 37.4 / 38.2, 128^3 42.6 / - / - / 40.9; clustered 81^3 27.7 /
// 25.4 / 25.1 / 26.1, 128^3 54.9 / - / - / 52.5.  Past 2^21 rows it no longer
// pays (160^3 mixed 68.5 / 70.4, FP64 80.8 / 83.1).
static int ahead_rows(int n) {
    const int nchunk = (n + kBlock - 1) / kBlock;
    return nchunk <= kMaxRedBlocks ? 0 : nchunk <= 4096 ? 4 : nchunk <= 8192 ? 8 : 0;
}
static int pcg_grid(int n) {
    const int u = ahead_rows(n), nchunk = ((n + kBlock - 1) / kBlock + (u ? u - 1 : 0)) / (u ? u : 1);
    int g = ((nchunk + 7) / 8) * 8;
    if (g > kMaxRedBlocks) g = kMaxRedBlocks;
    if (g < 8) g = 8;
    return g;
}

// Launch KERNEL<W> with W the operator's kernel width: a uniform ELL width
// (5..7), a stencil width (-7, -8), or 0 for the generic loops.
#define DISPATCH_WG(A, GRID, KERNEL, ...)                                     \
    do {                                                                        \
        switch (kernel_width(A)) {                                              \
            case 5: KERNEL<5><<<GRID, kBlock, 0, st>>>(__VA_ARGS__); break;      \
            case 6: KERNEL<6><<<GRID, kBlock, 0, st>>>(__VA_ARGS__); break;      \
            case 7: KERNEL<7><<<GRID, kBlock, 0, st>>>(__VA_ARGS__); break;      \
            case -7: KERNEL<-7><<<GRID, kBlock, 0, st>>>(__VA_ARGS__); break;    \
            case -8: KERNEL<-8><<<GRID, kBlock, 0, st>>>(__VA_ARGS__); break;    \
            default: KERNEL<0><<<GRID, kBlock, 0, st>>>(__VA_ARGS__); break;     \
        }                                                                       \
    } while (0)
// KERNEL<W, ARGS> over the chunks of a small operator
#define COMMA(A, B) A, B
#define DISPATCH_SMALL(A, KERNEL, ARGS, ...)                                              \
    do {                                                                                  \
        switch (kernel_width(A)) {                                                        \
            case 5: KERNEL<5, ARGS><<<S->nchunk, kBlock, 0, st>>>(__VA_ARGS__); break;    \
            case 6: KERNEL<6, ARGS><<<S->nchunk, kBlock, 0, st>>>(__VA_ARGS__); break;    \
            case 7: KERNEL<7, ARGS><<<S->nchunk, kBlock, 0, st>>>(__VA_ARGS__); break;    \
            case -7: KERNEL<-7, ARGS><<<S->nchunk, kBlock, 0, st>>>(__VA_ARGS__); break;  \
            case -8: KERNEL<-8, ARGS><<<S->nchunk, kBlock, 0, st>>>(__VA_ARGS__); break;  \
            default: KERNEL<0, ARGS><<<S->nchunk, kBlock, 0, st>>>(__VA_ARGS__); break;   \
        }                                                                                 \
    } while (0)
#define DISPATCH_W(A, KERNEL, ...) DISPATCH_WG(A, S->grid, KERNEL, __VA_ARGS__)
// the product of a long iteration, KERNEL or (FP64) its _sym form, in
// workgroups of kWide or kBlock threads
#define WIDTHS(KERNEL, GRID, NB, P)                                                \
    switch (kernel_width(A)) {                                                     \
        case 5: KERNEL<5, NB><<<GRID, NB, 0, st>>>(v, d, P); break;                \
        case 6: KERNEL<6, NB><<<GRID, NB, 0, st>>>(v, d, P); break;                \
        case 7: KERNEL<7, NB><<<GRID, NB, 0, st>>>(v, d, P); break;                \
        case -7: KERNEL<-7, NB><<<GRID, NB, 0, st>>>(v, d, P); break;              \
        case -8: KERNEL<-8, NB><<<GRID, NB, 0, st>>>(v, d, P); break;              \
        default: KERNEL<0, NB><<<GRID, NB, 0, st>>>(v, d, P); break;               \
    }
#define SYM_WIDTHS(KERNEL, GRID, NB, P)                                            \
    if (kernel_width(A) == -7)                                                     \
        KERNEL<-7, NB><<<GRID, NB, 0, st>>>(v, d, P);                              \
    else                                                                           \
        KERNEL<-8, NB><<<GRID, NB, 0, st>>>(v, d, P);
#define SYM_PRODUCT(KERNEL, P)                                                     \
    do {                                                                           \
        if (wide == 1024) {                                                        \
            SYM_WIDTHS(KERNEL, nwide, 1024, P)                                     \
        } else if (wide) {                                                         \
            SYM_WIDTHS(KERNEL, nwide, 512, P)                                      \
        } else {                                                                   \
            SYM_WIDTHS(KERNEL, S->nchunk, kBlock, P)                               \
        }                                                                          \
    } while (0)
#define ROW_PRODUCT(KERNEL, P)                                                     \
    do {                                                                           \
        if (wide == 1024) {                                                        \
            WIDTHS(KERNEL, nwide, 1024, P)                                         \
        } else if (wide) {                                                         \
            WIDTHS(KERNEL, nwide, 512, P)                                          \
        } else {                                                                   \
            WIDTHS(KERNEL, S->nchunk, kBlock, P)                                   \
        }                                                                          \
    } while (0)

#define LEAN_LAUNCH(KERNEL, GRID, ...)                                                \
    do {                                                                              \
        if (lean)                                                                     \
            KERNEL<true><<<GRID, kBlock, 0, st>>>(__VA_ARGS__);                       \
        else                                                                          \
            KERNEL<false><<<GRID, kBlock, 0, st>>>(__VA_ARGS__);                      \
    } while (0)

static PcgDev make_dev(gip_pcg *S, const double *b, double *x, int precond) {
    PcgDev d;
    d.n = S->n;
    d.G = S->grid;
    d.nchunk = S->nchunk;
    d.wpc = kWaves;
    d.Gdn = S->gdn;
    d.chunk = S->fold ? S->chunk : S->part + P_DN * kMaxRedBlocks;
    d.chunk_s = S->fold ? S->chunk + (size_t)S->nchunk * kWaves : nullptr;
    d.az32 = S->az32;
    d.azl = S->azl;
    d.deflate = 0;
    d.x = x;
    d.r = S->r;
    d.s = S->s;
    d.Ap = S->Ap;
    d.b = b;
    d.dinv = S->dinv;
    d.sp[0] = reinterpret_cast<SP<double> *>(S->p);
    d.sp[1] = reinterpret_cast<SP<double> *>(S->p2);
    d.sp32[0] = reinterpret_cast<SP<float> *>(S->p32);
    d.sp32[1] = reinterpret_cast<SP<float> *>(S->p32b);
    d.r32 = S->r32;
    d.s32 = S->s32;
    d.Ap32 = S->Ap32;
    d.xc32 = S->xc32;
    d.dinv32 = S->dinv32;
    d.az = S->az;
    d.sc = S->sc;
    d.state = S->state;
    d.iters = S->state + 1;
    d.part = S->part;
    d.precond = precond;
    d.dc_sel = S->A->d_dict_sel;
    d.dc_id = S->A->d_dict_id;
    d.ddinv = S->ddinv;
    d.ddinv32 = S->ddinv32;
    return d;
}

extern "C" {

int gip_pcg_create(gip_ctx *c, const gip_mat *A, int32_t n_all, gip_pcg **out) {
    if (!c || !A || !out || n_all < A->nrows) return set_error(GIP_EINVAL, "gip_pcg_create: bad argument");
    // one stream orders the operator's value updates and the solves
    if (A->ctx != c) return set_error(GIP_EINVAL, "gip_pcg_create: operator belongs to another context");
    if (n_all < A->cols_needed) return set_error(GIP_EINVAL, "gip_pcg_create: vectors shorter than the operator's columns");
    if (A->format != GIP_FMT_ELL && A->format != GIP_FMT_CSR && A->format != GIP_FMT_STENCIL)
        return set_error(GIP_EINVAL, "gip_pcg_create: operator must be ELL, stencil or CSR");
    gip_pcg *S = new (std::nothrow) gip_pcg();
    if (!S) return set_error(GIP_ENOMEM, "gip_pcg_create: allocation failed");
    S->ctx = c;
    S->A = A;
    S->n = A->nrows;
    S->n_all = n_all;
    S->grid = pcg_grid(A->nrows);
    S->nchunk = std::max(1, (A->nrows + kBlock - 1) / kBlock);
    // up to kMaxRedBlocks chunks (2^19 rows) the next kernels read the
    // per-chunk partials directly; beyond, a fold kernel sums each run of
    // 256 chunks first
    S->fold = S->nchunk > kMaxRedBlocks;
    S->rows = S->fold && S->n > kRowsMin;
    S->gdn = S->fold ? (S->nchunk + kBlock - 1) / kBlock : S->nchunk;
    if (S->gdn > kMaxRedBlocks) {
        delete S;
        return set_error(GIP_EINVAL, "gip_pcg_create: more rows than the product partials cover (2^27)");
    }
    size_t n = (size_t)std::max(1, A->nrows);
    size_t na = (size_t)std::max(1, n_all);  // directions are SpMV inputs: ghost columns included
    hipError_t e = hipSetDevice(c->device);
    auto dalloc = [&](void **p, size_t bytes) {
        if (e == hipSuccess) e = hipMalloc(p, bytes);
    };
    dalloc((void **)&S->r, n * 8);
    const size_t pb = S->fold ? 8 : sizeof(SP<double>);
    dalloc((void **)&S->p, na * pb);
    dalloc((void **)&S->p2, na * pb);
    if (S->fold) dalloc((void **)&S->s, n * 8);
    dalloc((void **)&S->Ap, n * 8);
    dalloc((void **)&S->dinv, n * 8);
    dalloc((void **)&S->sc, S_COUNT * 8);
    dalloc((void **)&S->part, (size_t)P_COUNT * kMaxRedBlocks * 8);
    if (S->fold) dalloc((void **)&S->chunk, (size_t)S->nchunk * kWaves * 2 * 8);  // p.Ap, then 1.Ap
    dalloc((void **)&S->state, 2 * sizeof(int));
    if (e == hipSuccess) e = hipHostMalloc((void **)&S->h_pub, kHostBlock * 8, hipHostMallocCoherent);
    if (e == hipSuccess) e = hipHostGetDevicePointer((void **)&S->h_pub_dev, S->h_pub, 0);
    if (e == hipSuccess) {
        memset(S->h_pub, 0, kHostBlock * 8);
        S->h_flag = reinterpret_cast<uint64_t *>(S->h_pub + kSeqSlot);
        S->h_flag_dev = reinterpret_cast<uint64_t *>(S->h_pub_dev + kSeqSlot);
        S->seq = &S->own_seq;
    }
    if (e == hipSuccess) e = hipMemsetAsync(S->sc, 0, S_COUNT * 8, c->stream);
    // partial slots past each producer's grid stay zero for sum_padded
    if (e == hipSuccess) e = hipMemsetAsync(S->part, 0, (size_t)P_COUNT * kMaxRedBlocks * 8, c->stream);
    if (e == hipSuccess) e = hipMemsetAsync(S->state, 0, 2 * sizeof(int), c->stream);
    if (e != hipSuccess) {
        int rc = hip_fail(e, "gip_pcg_create");
        gip_pcg_destroy(S);
        return rc;
    }
    int rc = A->diag_missing ? GIP_OK : gip_mat_diag_inv(A, S->dinv);
    if (!rc && S->fold && mat_dict_ok(A)) {
        // the same inverse, once per tuple (the diagonal is part of the tuple)
        const int nd = A->dict_n;
        e = hipMalloc((void **)&S->ddinv, (size_t)nd * 8);
        if (e == hipSuccess) e = hipMalloc((void **)&S->ddinv32, (size_t)nd * 4);
        if (e == hipSuccess) {
            k_tuple_inv<<<(nd + kBlock - 1) / kBlock, kBlock, 0, c->stream>>>(nd, A->d_dict_diag, S->ddinv, S->ddinv32);
            e = hipGetLastError();
            S->dict_version = A->dict_version;
        }
        if (e != hipSuccess) rc = hip_fail(e, "gip_pcg_create dictionary");
    }
    if (!rc) {
        e = hipStreamSynchronize(c->stream);
        if (e != hipSuccess) rc = hip_fail(e, "gip_pcg_create sync");
    }
    if (rc) {
        gip_pcg_destroy(S);
        return rc;
    }
    *out = S;
    return GIP_OK;
}

int gip_pcg_destroy(gip_pcg *S) {
    if (!S) return GIP_OK;
    hipSetDevice(S->ctx->device);
    hipStreamSynchronize(S->ctx->stream);
    void *ptrs[] = {S->r,    S->p,      S->s,  S->Ap, S->dinv, S->r32,   S->p32,  S->s32,  S->Ap32,
                    S->xc32, S->dinv32, S->az, S->sc, S->part, S->chunk, S->state, S->p2, S->p32b, S->az32, S->azl,
                    S->ddinv, S->ddinv32};
    for (void *p : ptrs)
        if (p) hipFree(p);
    if (S->h_pub) hipHostFree(S->h_pub);
    if (S->tev0) hipEventDestroy(S->tev0);
    if (S->tev1) hipEventDestroy(S->tev1);
    delete S;
    return GIP_OK;
}

static int ensure_mixed(gip_pcg *S) {
    if (S->r32) return GIP_OK;
    const gip_mat *A = S->A;
    if (((A->format == GIP_FMT_ELL || A->format == GIP_FMT_STENCIL) && !A->d_ell_val32) ||
        (A->format == GIP_FMT_CSR && !A->d_val32))
        return set_error(GIP_EINVAL, "mixed precision needs an operator created with GIP_MAT_FP32");
    size_t n = (size_t)std::max(1, S->n), na = (size_t)std::max(1, S->n_all);
    float **bufs[] = {&S->r32, &S->s32, &S->Ap32, &S->xc32, &S->dinv32};
    for (float **b : bufs) GIP_HIP_TRY(hipMalloc(b, n * 4));
    GIP_HIP_TRY(hipMalloc(&S->az, n * 8));
    GIP_HIP_TRY(hipMalloc(&S->az32, n * 4));
    GIP_HIP_TRY(hipMalloc(&S->azl, sizeof(AzList)));
    GIP_HIP_TRY(hipMemsetAsync(S->azl, 0, sizeof(AzList), S->ctx->stream));
    // the FP32 direction is an SpMV input: ghost columns included, and zero
    // there (the correction leaves the ghost values of x unchanged)
    const size_t pb = S->fold ? 4 : sizeof(SP<float>);
    GIP_HIP_TRY(hipMalloc(&S->p32, na * pb));
    GIP_HIP_TRY(hipMemsetAsync(S->p32, 0, na * pb, S->ctx->stream));
    GIP_HIP_TRY(hipMalloc(&S->p32b, na * pb));
    GIP_HIP_TRY(hipMemsetAsync(S->p32b, 0, na * pb, S->ctx->stream));
    if (S->n) {
        k_to32<<<(S->n + kBlock - 1) / kBlock, kBlock, 0, S->ctx->stream>>>(S->n, S->dinv, S->dinv32);
        GIP_LAUNCH_CHECK("dinv32");
    }
    return GIP_OK;
}

// az = A 1 over the solved rows and 1.A1 into S_ZAZ, from A's current
// values (one product and one reduction per mixed solve); the FP64
// direction buffer serves as the vector 1 before the setup overwrites it.
static int coarse_setup(gip_pcg *S) {
    gip_ctx *c = S->ctx;
    if (S->n_all == 0) return GIP_OK;
    double *z = S->p;
    k_ones<<<(S->n_all + kBlock - 1) / kBlock, kBlock, 0, c->stream>>>(S->n, S->n_all, z, S->az, S->azl);
    GIP_LAUNCH_CHECK("coarse vector");
    int rc = spmv_launch(c, S->A, z, S->az, 1.0, 0.0, 0, nullptr);
    if (!rc) rc = launch_reduce(c, RED_SUM, S->n, S->az, z, S->sc + S_ZAZ);
    if (!rc && S->n) {
        k_az32<<<(S->n + kBlock - 1) / kBlock, kBlock, 0, c->stream>>>(S->n, S->az, S->az32, S->azl);
        GIP_LAUNCH_CHECK("coarse vector fp32");
    }
    return rc;
}

static_assert(S_COUNT + 2 <= kPubWords, "published words");
static int *h_state(gip_pcg *S) { return reinterpret_cast<int *>(S->h_pub + S_COUNT); }

// what the next kernel to publish stores, and the wait for it
static Pub next_pub(gip_pcg *S) {
    return Pub{S->h_pub_dev, reinterpret_cast<int *>(S->h_pub_dev + S_COUNT), S->h_flag_dev, ++*S->seq};
}
static int wait_pub(gip_pcg *S) { return wait_published(S->ctx, S->h_flag, *S->seq); }

constexpr int kFixedPoll = 4096;

// The solve on a solver's workspace (allocated by gip_pcg_create, or the
// no-alloc scratch); arguments already checked.
static int pcg_solve_impl(gip_pcg *S, const double *b, double *x, const double *x0, const gip_pcg_opts *o,
                          gip_pcg_stats *stats) {
    gip_ctx *c = S->ctx;
    hipStream_t st = c->stream;
    const gip_mat *A = S->A;
    const bool mixed = o->precision == GIP_PCG_MIXED;
    if (mixed) {
        int rc = ensure_mixed(S);
        if (rc) return rc;
    }
    if (mixed) {
        int rc = coarse_setup(S);
        if (rc) return rc;
    }
    // the dictionary of a stencil operator's slot values, where it has one, before
    // either form of the stored values; in FP32 from 2^21 rows on, below
    // which the values stay in the caches (us per iteration without and with
    // it: FP64 81^3 30.9 / 27.9, 97^3 37.9 / 31.5, 128^3 58.5 / 46.6, 256^3
    // 423.7 / 324.1; mixed 97^3 31.5 / 32.3, 128^3 45.0 / 42.3, 256^3
    // 250.8 / 211.1)
    const bool dict = S->fold && A->st_w >= 7 && (mixed ? mat_dict_ok32(A) && S->n >= 1 << 21 : mat_dict_ok(A));
    // else the symmetric form of a 7- or 8-slot operator for the FP64 products
    // of the long iterations (made and checked here after a change of values;
    // the no-alloc solve never has those iterations)
    bool sym = false;
    if (!mixed && dict) {
        const_cast<gip_mat *>(A)->sym_due = A->val_version + 1;
    } else if (!mixed && S->fold && (kernel_width(A) == -7 || kernel_width(A) == -8)) {
        int rc = mat_sym_prepare(c, const_cast<gip_mat *>(A), &sym);
        if (rc) return rc;
    }
    // ... and its inverse diagonal, while the solver's (taken when it was
    // created) is the one of the operator's present values.  us per
    // iteration with s stored and not: FP64 128^3 46.6 / 43.5, 200^3 195 /
    // 165, 256^3 324 / 300; mixed 256^3 211 / 197, but 200^3 117 / 122: where
    // slices need their rows' ids, those and the record cost the FP32 sweeps
    // what s and Dinv did.
    const bool lean = dict && (!mixed || !A->dict_ids) &&
                      (!o->precond || (S->ddinv && S->dict_version == A->dict_version));
    PcgDev d = make_dev(S, b, x, o->precond ? 1 : 0);
    if (dict) d.wpc = 1;
    const int wide = S->fold && S->n <= (mixed ? kWideRows32 : kWideRows) ? wide_of(S->n) : 0;
    const int nwide = wide ? (S->n + wide - 1) / wide : 0;
    if (wide) d.Gdn = nwide;
    auto fold = [&]() {  // between a long product and its update
        if (!wide)
            k_fold_dn<<<S->gdn, kBlock, 0, st>>>(d);
        else if (dict)
            k_fold_wide<<<(nwide + kBlock - 1) / kBlock, kBlock, 0, st>>>(d, wide / kBlock);
    };
    EllView v = view(A);
    const int pollk = o->poll > 0 ? o->poll : 16;
    const int use_coarse = o->coarse >= 0 ? 1 : 0;
    d.deflate = mixed && use_coarse;
    // small operators: few enough partials for every wavefront to sum them all
    const bool wave = S->grid <= kWaveParts;
    // direction of iteration k: two buffers by parity
    auto pdir = [&](int k) { return (k & 1) ? S->p2 : S->p; };
    auto pdir32 = [&](int k) { return (k & 1) ? S->p32b : S->p32; };
    // the instance of a long sweep: LEAN, whether a direction sweep makes the
    // pending x updates, and (not the row-per-thread ones) the rows a thread
    // requests ahead
#define DIR_LAUNCH(KERNEL, GRID, PAIR, ...)                        \
    do {                                                           \
        if (lean && (PAIR))                                        \
            KERNEL<true, true><<<GRID, kBlock, 0, st>>>(__VA_ARGS__);   \
        else if (lean)                                             \
            KERNEL<true, false><<<GRID, kBlock, 0, st>>>(__VA_ARGS__);  \
        else if (PAIR)                                             \
            KERNEL<false, true><<<GRID, kBlock, 0, st>>>(__VA_ARGS__);  \
        else                                                       \
            KERNEL<false, false><<<GRID, kBlock, 0, st>>>(__VA_ARGS__); \
    } while (0)
#define AHEAD_DIR(KERNEL, U, PAIR, ...)                                      \
    do {                                                                     \
        if (lean && (PAIR))                                                  \
            KERNEL<true, true, U><<<S->grid, kBlock, 0, st>>>(__VA_ARGS__);  \
        else if (lean)                                                       \
            KERNEL<true, false, U><<<S->grid, kBlock, 0, st>>>(__VA_ARGS__); \
        else if (PAIR)                                                       \
            KERNEL<false, true, U><<<S->grid, kBlock, 0, st>>>(__VA_ARGS__); \
        else                                                                 \
            KERNEL<false, false, U><<<S->grid, kBlock, 0, st>>>(__VA_ARGS__);\
    } while (0)
#define SWEEP_DIR(KERNEL, PAIR, ...)                   \
    do {                                               \
        if (ahead == 4)                                \
            AHEAD_DIR(KERNEL, 4, PAIR, __VA_ARGS__);   \
        else if (ahead == 8)                           \
            AHEAD_DIR(KERNEL, 8, PAIR, __VA_ARGS__);   \
        else                                           \
            AHEAD_DIR(KERNEL, 0, PAIR, __VA_ARGS__);   \
    } while (0)
#define AHEAD_UPDATE(KERNEL, U)                                     \
    do {                                                            \
        if (lean)                                                   \
            KERNEL<true, U><<<S->grid, kBlock, 0, st>>>(d, k);      \
        else                                                        \
            KERNEL<false, U><<<S->grid, kBlock, 0, st>>>(d, k);     \
    } while (0)
#define SWEEP_UPDATE(KERNEL)            \
    do {                                \
        if (ahead == 4)                 \
            AHEAD_UPDATE(KERNEL, 4);    \
        else if (ahead == 8)            \
            AHEAD_UPDATE(KERNEL, 8);    \
        else                            \
            AHEAD_UPDATE(KERNEL, 0);    \
    } while (0)
    const int ahead = ahead_rows(S->n);
    // time_products: events around one product launch (k >= 1) per host
    // poll, read after the poll's synchronisation
    const bool timing = o->time_products != 0;
    if (timing && !S->tev0) {
        GIP_HIP_TRY(hipEventCreate(&S->tev0));
        GIP_HIP_TRY(hipEventCreate(&S->tev1));
    }
    std::vector<float> samples;
    bool armed = false;  // a sampled pair is recorded and not read yet
    auto sample_begin = [&](int k) {
        const bool on = timing && !armed && k > 0;
        if (on) hipEventRecord(S->tev0, st);
        return on;
    };
    auto sample_end = [&](bool on) {
        if (on) {
            hipEventRecord(S->tev1, st);
            armed = true;
        }
    };
    auto sample_read = [&]() {  // after a wait for the host's poll
        float ms = 0.0f;
        if (armed) hipEventSynchronize(S->tev1);
        if (armed && hipEventElapsedTime(&ms, S->tev0, S->tev1) == hipSuccess) samples.push_back(ms);
        armed = false;
    };
    // setup, GIP_LinearSolver.h:55-80
    double *const dir0 = S->fold ? S->p : nullptr;  // small operators: the pairs in d
    DISPATCH_W(A, k_setup_resid, v, d, x0, S->n_all, dir0, S->p2);
    k_setup_dir<<<S->grid, kBlock, 0, st>>>(d, dir0);
    const bool fixed = !mixed && !(o->tol > 0.0);
    k_setup_fin<<<1, kBlock, 0, st>>>(d, o->tol, fixed || mixed ? Pub{} : next_pub(S));
    GIP_LAUNCH_CHECK("pcg setup");
    int corrections = 0, rc;
    // FP64 with a fixed iteration count (tol <= 0): nothing can stop the
    // solve early but a breakdown, after which every queued kernel returns
    // at once, so the iterations are queued and the host reads the state
    // once, at the end (on long runs every kFixedPoll iterations: 200,000 of a
    // small operator that breaks down at once queued 1.0 s of kernels)
    if (fixed)
        h_state(S)[0] = ST_RUN;
    else if (!mixed && (rc = wait_pub(S)))
        return rc;
    if (!mixed) {
        int k = 0;  // iterations queued
        while (k < o->maxit && h_state(S)[0] == ST_RUN) {
            int chunk = std::min(fixed ? kFixedPoll : pollk, o->maxit - k);
            for (int j = 0; j < chunk; ++j, ++k) {
                if (S->fold && !S->rows) {
                    if (k > 0) SWEEP_DIR(k_iter_dir, k >= 2 && !(k & 1), d, pdir(k - 1), pdir(k), k);
                    const bool smp = sample_begin(k);
                    if (dict)
                        DICT_LAUNCH(k_iter_spmv_dict, A->st_w, S->nchunk, st, v, d, pdir(k));
                    else if (sym)
                        SYM_PRODUCT(k_iter_spmv_sym, pdir(k));
                    else
                        ROW_PRODUCT(k_iter_spmv, pdir(k));
                    sample_end(smp);
                    fold();
                    SWEEP_UPDATE(k_iter_update_grid);
                } else if (S->fold) {
                    // (partials: p.Ap in chunk, then r.s in chunk and r.r in chunk_s)
                    if (k > 0) DIR_LAUNCH(k_iter_dir_rows, S->nchunk, k >= 2 && !(k & 1), d, pdir(k - 1), pdir(k), k);
                    const bool smp = sample_begin(k);
                    if (dict)
                        DICT_LAUNCH(k_iter_spmv_dict, A->st_w, S->nchunk, st, v, d, pdir(k));
                    else if (sym)
                        SYM_PRODUCT(k_iter_spmv_sym, pdir(k));
                    else
                        ROW_PRODUCT(k_iter_spmv, pdir(k));
                    sample_end(smp);
                    k_fold_two<<<S->gdn, kBlock, 0, st>>>(d, S->nchunk, d.wpc, d.chunk, nullptr, P_DN, P_DN);
                    k_alpha_fin<<<1, kBlock, 0, st>>>(d, k);
                    const int uwg = (S->nchunk + kUpdateRows - 1) / kUpdateRows, ufold = (uwg + kBlock - 1) / kBlock;
                    LEAN_LAUNCH(k_iter_update_rows, uwg, d, k);
                    k_fold_two<<<ufold, kBlock, 0, st>>>(d, uwg, kWaves, d.chunk, d.chunk_s, P_RS, P_RR);
                    k_beta_fin<<<1, kBlock, 0, st>>>(d, k + 1, ufold);
                } else {
                    const bool smp = sample_begin(k);
                    const bool tol = o->tol > 0.0;  // without one (fixed iteration count): no r.r test
                    if (k == 0)
                        DISPATCH_WG(A, S->nchunk, k_iter_spmv_small, v, d);
                    else if (wave && tol)
                        DISPATCH_SMALL(A, k_iter_dirprod, COMMA(true, true), v, d, k);
                    else if (wave)
                        DISPATCH_SMALL(A, k_iter_dirprod, COMMA(false, true), v, d, k);
                    else if (tol)
                        DISPATCH_SMALL(A, k_iter_dirprod, COMMA(true, false), v, d, k);
                    else
                        DISPATCH_SMALL(A, k_iter_dirprod, COMMA(false, false), v, d, k);
                    sample_end(smp);
                    if (wave)
                        k_iter_update<true><<<S->grid, kBlock, 0, st>>>(d, k);
                    else
                        k_iter_update<false><<<S->grid, kBlock, 0, st>>>(d, k);
                }
            }
            GIP_LAUNCH_CHECK("pcg iteration");
            if (!fixed || k < o->maxit) {
                k_publish<<<1, 64, 0, st>>>(d, next_pub(S));
                GIP_LAUNCH_CHECK("pcg poll");
                if ((rc = wait_pub(S))) return rc;
                sample_read();
            }
        }
        if (S->fold) {
            if (k > 0) k_x_flush_pair<<<S->grid, kBlock, 0, st>>>(d, S->p, S->p2);
        } else if (k > 0) {
            k_x_flush<<<S->grid, kBlock, 0, st>>>(d, k - 1);
        }
        if (S->rows)
            k_fin_rows<<<1, kBlock, 0, st>>>(d, next_pub(S));
        else
            k_fin<<<1, kBlock, 0, st>>>(d, next_pub(S));
        GIP_LAUNCH_CHECK("pcg final test");
        if ((rc = wait_pub(S))) return rc;
    } else {
        // FP64 residual of x0 (with the coarse step), FP32 copies, first direction
        DISPATCH_W(A, k_m_resid, v, d);
        k_m_coarse<<<S->grid, kBlock, 0, st>>>(d, use_coarse);
        k_m_corr_fin<<<1, kBlock, 0, st>>>(d, 0, 1, next_pub(S));
        if (S->fold)
            k_m_start<<<S->grid, kBlock, 0, st>>>(d, S->p32);
        else
            k_m_pairs<<<S->grid, kBlock, 0, st>>>(d, d.sp32[0], 1);
        GIP_LAUNCH_CHECK("mixed setup");
        if ((rc = wait_pub(S))) return rc;
        double last_rr = S->h_pub[S_TRUE_RR];
        const double it = o->inner_tol > 0.0 ? o->inner_tol : 0.1;
        const double inner2 = it * it;
        int k = 0, pending = 0;  // pending: the correction updates not yet applied (at most two)
        while (k < o->maxit && h_state(S)[0] == ST_RUN) {
            int chunk = std::min(pollk, o->maxit - k);
            for (int j = 0; j < chunk; ++j, ++k) {
                if (S->fold) {
                    if (k > 0) SWEEP_DIR(k_m_dir, pending == 2, d, pdir32(k - 1), pdir32(k), k);
                    pending = pending == 2 ? 1 : pending + 1;
                    const bool smp = sample_begin(k);
                    if (dict)
                        DICT_LAUNCH(k_m_spmv_dict, A->st_w, S->nchunk, st, v, d, pdir32(k));
                    else
                        ROW_PRODUCT(k_m_spmv, pdir32(k));
                    sample_end(smp);
                    fold();
                    SWEEP_UPDATE(k_m_update);
                } else {
                    const bool smp = sample_begin(k);
                    if (k == 0)
                        DISPATCH_WG(A, S->nchunk, k_m_spmv_small, v, d);
                    else if (wave)
                        DISPATCH_SMALL(A, k_m_dirprod, true, v, d, k, pending);
                    else
                        DISPATCH_SMALL(A, k_m_dirprod, false, v, d, k, pending);
                    sample_end(smp);
                    if (wave)
                        k_m_update_small<true><<<S->grid, kBlock, 0, st>>>(d, k);
                    else
                        k_m_update_small<false><<<S->grid, kBlock, 0, st>>>(d, k);
                    pending = 1;
                }
            }
            k_m_status<<<1, kBlock, 0, st>>>(d, next_pub(S));
            GIP_LAUNCH_CHECK("mixed iteration");
            if ((rc = wait_pub(S))) return rc;
            sample_read();
            if (h_state(S)[0] != ST_RUN) break;
            const double rr32 = S->h_pub[S_RR], tol2 = S->h_pub[S_TOL2];
            const bool near_target = tol2 >= 0.0 && rr32 <= tol2;
            if (rr32 <= inner2 * last_rr || near_target || k >= o->maxit) {
                if (S->fold)
                    k_m_fold<<<S->grid, kBlock, 0, st>>>(d, pdir32(k - 1), pdir32(k), k - 1, pending);
                else
                    k_m_fold_small<<<S->grid, kBlock, 0, st>>>(d, k - 1);
                pending = 0;
                DISPATCH_W(A, k_m_resid, v, d);
                k_m_coarse<<<S->grid, kBlock, 0, st>>>(d, use_coarse);
                k_m_corr_fin<<<1, kBlock, 0, st>>>(d, k, 0, next_pub(S));
                if (!S->fold) k_m_pairs<<<S->grid, kBlock, 0, st>>>(d, d.sp32[(k - 1) & 1], 0);
                GIP_LAUNCH_CHECK("mixed correction");
                ++corrections;
                if ((rc = wait_pub(S))) return rc;
                last_rr = S->h_pub[S_TRUE_RR];
            }
        }
    }
    sample_read();
    int status = GIP_OK;
    const int fin = h_state(S)[0] & ST_MASK;
    if (fin == ST_BREAK)
        status = GIP_EBREAKDOWN;
    else if (o->tol > 0.0 && fin != ST_CONV)
        status = GIP_ENOCONV;
    if (stats) {
        stats->iters = h_state(S)[1];
        stats->corrections = corrections;
        const double bb = S->h_pub[S_BB], rr = S->h_pub[S_RR];
        stats->relres = bb > 0.0 ? std::sqrt(rr / bb) : std::sqrt(rr);
        stats->status = status;
        stats->product_samples = (int32_t)samples.size();
        stats->product_ms = 0.0;
        if (!samples.empty()) {  // median (a launch that found the solve finished is short)
            std::nth_element(samples.begin(), samples.begin() + samples.size() / 2, samples.end());
            stats->product_ms = samples[samples.size() / 2];
        }
    }
    return status == GIP_EBREAKDOWN ? set_error(GIP_EBREAKDOWN, "PCG breakdown (p.Ap == 0 or non-finite step)") : GIP_OK;
}

int gip_pcg_solve(gip_pcg *S, const double *b, double *x, const double *x0, const gip_pcg_opts *o, gip_pcg_stats *stats) {
    if (!S || !b || !x || !x0 || !o || o->maxit < 0) return set_error(GIP_EINVAL, "gip_pcg_solve: bad argument");
    if (o->precond && S->A->diag_missing) return set_error(GIP_EINVAL, "gip_pcg_solve: Jacobi needs every diagonal entry");
    return pcg_solve_impl(S, b, x, x0, o, stats);
}

int gip_pcg_solve_noalloc(gip_ctx *c, const gip_mat *A, int32_t n_all, const double *b, double *x, const double *x0,
                          const gip_pcg_opts *o, gip_pcg_stats *stats) {
    if (!c || !A || !b || !x || !x0 || !o || o->maxit < 0)
        return set_error(GIP_EINVAL, "gip_pcg_solve_noalloc: bad argument");
    if (A->ctx != c) return set_error(GIP_EINVAL, "gip_pcg_solve_noalloc: operator belongs to another context");
    if (o->precision != GIP_PCG_FP64) return set_error(GIP_EINVAL, "gip_pcg_solve_noalloc: FP64 only");
    if (o->time_products) return set_error(GIP_EINVAL, "gip_pcg_solve_noalloc: no product timing");
    if (A->format != GIP_FMT_ELL && A->format != GIP_FMT_CSR && A->format != GIP_FMT_STENCIL)
        return set_error(GIP_EINVAL, "gip_pcg_solve_noalloc: operator must be ELL, stencil or CSR");
    if (A->nrows > kScratchRows || n_all > kScratchAll)
        return set_error(GIP_EINVAL, "gip_pcg_solve_noalloc: at most 262144 rows and 327680 vector entries");
    if (n_all < A->nrows || n_all < A->cols_needed)
        return set_error(GIP_EINVAL, "gip_pcg_solve_noalloc: vectors shorter than the operator's columns");
    if (o->precond && A->diag_missing)
        return set_error(GIP_EINVAL, "gip_pcg_solve_noalloc: Jacobi needs every diagonal entry");
    double *base = (c->device >= 0 && c->device < kScratchDevices) ? g_scratch[c->device] : nullptr;
    if (!base) return set_error(GIP_EINVAL, "gip_pcg_solve_noalloc: no scratch on this device (gip_init sets it up)");
    GIP_HIP_TRY(hipSetDevice(c->device));
    gip_pcg S{};
    S.ctx = c;
    S.A = A;
    S.n = A->nrows;
    S.n_all = n_all;
    S.grid = pcg_grid(A->nrows);
    S.nchunk = std::max(1, (A->nrows + kBlock - 1) / kBlock);
    S.fold = false;  // at most 1024 chunks: the fused two-kernel iteration
    S.gdn = S.nchunk;
    S.r = base;
    S.Ap = S.r + kScratchRows;
    S.dinv = S.Ap + kScratchRows;
    S.p = S.dinv + kScratchRows;
    S.p2 = S.p + 2 * (size_t)kScratchAll;
    double *zero = S.p2 + 2 * (size_t)kScratchAll;
    S.part = zero;
    S.sc = S.part + (size_t)P_COUNT * kMaxRedBlocks;
    S.state = reinterpret_cast<int *>(S.sc + S_COUNT);
    S.h_pub = c->h_result + kPubSlot;
    S.h_pub_dev = c->h_result_dev + kPubSlot;
    S.h_flag = reinterpret_cast<uint64_t *>(c->h_result + kPubSeqSlot);
    S.h_flag_dev = reinterpret_cast<uint64_t *>(c->h_result_dev + kPubSeqSlot);
    S.seq = &c->pub_seq;
    // partial slots past each producer's grid, the scalars and the state
    // words start at zero (a previous call may have left other values)
    k_zero<<<(unsigned)((kScratchZero + kBlock - 1) / kBlock), kBlock, 0, c->stream>>>(kScratchZero, zero);
    GIP_LAUNCH_CHECK("gip_pcg_solve_noalloc: clear");
    if (!A->diag_missing) {
        int rc = gip_mat_diag_inv(A, S.dinv);
        if (rc) return rc;
    }
    return pcg_solve_impl(&S, b, x, x0, o, stats);
}

}  // extern "C"
