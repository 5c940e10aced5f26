// Device helpers shared by the SpMV, PCG and batch kernels: a read-only
// view of an operator, the product operand, the stored-order row sum, and
// the XCD-contiguous row sweep.
#pragma once

#include <hip/hip_runtime.h>

#include "gip_internal.h"

namespace gip {

struct EllView {
    int fmt;  // GIP_FMT_ELL / GIP_FMT_CSR / GIP_FMT_STENCIL
    const int32_t *soff, *col, *rp;
    const double *val;
    const float *val32;
    // stencil layout
    const int32_t *st_off, *st_tcol;
    const StencilHdr *st_hdr;
    const StencilTail *st_tail;
    int st_w, tail_base, cmax;
    int ell_lg;  // sliced ELL: log2 of the rows per slice
    // symmetric form of the slot values (null when not in use)
    const int8_t *st_code;
    const double *sym;
    int sym_nu, sym_stride;  // arrays of sym_stride values (every slice's rows), one after another
    int sym_d[kSymMaxD];
    // dictionary of the slot values (null when there is none)
    const DictRec *dc_rec;
    const uint16_t *dc_id;
    const double *dc_tab, *dc_soa;
    const float *dc_tab32, *dc_soa32;
    int dc_n, dc_ids;
};

static EllView view(const gip_mat *A) {
    EllView v{};
    const bool packed = A->format == GIP_FMT_ELL || A->format == GIP_FMT_STENCIL;
    v.fmt = A->format;
    v.soff = A->d_slice_off;
    v.col = A->format == GIP_FMT_ELL ? A->d_ell_col : A->d_col;
    v.rp = A->d_rowptr;
    v.val = packed ? A->d_ell_val : A->d_val;
    v.val32 = packed ? A->d_ell_val32 : A->d_val32;
    v.st_off = A->d_st_off;
    v.st_tcol = A->d_st_tcol;
    v.st_hdr = A->d_st_hdr;
    v.st_tail = A->d_st_tail;
    v.st_w = A->st_w;
    v.tail_base = (int)A->st_tail_base;
    v.cmax = A->cols_needed > 0 ? A->cols_needed - 1 : 0;
    v.ell_lg = A->ell_lg;
    v.st_code = A->d_st_code;
    v.sym = A->sym_ok > 0 ? A->d_sym_val : nullptr;
    v.sym_nu = A->sym_nu;
    v.sym_stride = A->nslices * 64;
    for (int j = 0; j < kSymMaxD; ++j) v.sym_d[j] = A->sym_d[j];
    if (mat_dict_ok(A)) {
        v.dc_rec = A->d_dict_rec;
        v.dc_id = A->d_dict_id;
        v.dc_tab = A->d_dict_tab;
        v.dc_soa = A->d_dict_soa;
        v.dc_tab32 = A->d_dict_tab32;
        v.dc_soa32 = A->d_dict_soa32;
        v.dc_n = A->dict_n;
        v.dc_ids = A->dict_ids;
    }
    return v;
}

// Kernel template width of an operator: W > 0 uniform-width ELL, W < 0 the
// stencil layout with -W slots, 0 the generic loops.
static inline int kernel_width(const gip_mat *A) {
    if (A->format == GIP_FMT_ELL) return A->uniform_width;
    if (A->format == GIP_FMT_STENCIL) return -A->st_w;
    return 0;
}

// Operator metadata is read through the constant address space: no kernel
// writes an operator that it multiplies by, so a wavefront-uniform index
// gives a scalar load even where the kernel has stored results before it
// (inside a loop over rows the compiler could not prove that by itself).
template <class T>
using const_as = const __attribute__((address_space(4))) T;
template <class T>
__device__ inline const_as<T> *as_const(const T *p) {
    return (const_as<T> *)(uintptr_t)p;
}

// Workgroup b of G is placed on XCD b % 8 by the dispatcher; renumber the
// workgroups so that each XCD sweeps one contiguous range of rows and the
// neighbour gathers of a row range stay in that XCD's L2.
__device__ inline int xcd_block(int b, int G) {
    const int x = b & 7, idx = b >> 3, q = G >> 3, r = G & 7;
    return x * q + (x < r ? x : r) + idx;
}

// Runs of 8 consecutive chunks on one XCD, the runs in dispatch order: the
// whole chip still sweeps one narrow window of the vectors, and of a chunk's
// neighbours a mesh line away (one or a few chunks) most are in the same L2.
// Workgroups past the last whole group of 8 runs keep their place.
__device__ inline int xcd_run_block(int b, int G) {
    if (b >= (G & ~63)) return b;
    return (b & ~63) | ((b & 7) << 3) | ((b >> 3) & 7);
}

// The input vector of a product.  The row sums take any operand type with
// at(j) (the PCG also forms a direction on the fly as its operand).
template <class T>
struct Operand {
    const T *__restrict__ p;
    __device__ inline T at(int j) const { return p[j]; }
};

// The tail of a row in a slice of kind 2 (empty rows, or rows of several
// tail entries), located through the slice header's lane masks; false for
// an empty row.
template <class T, class V, class X>
__device__ inline bool stencil_tail_hdr(const EllView &A, const V *__restrict__ val, const X &x, int s, int row,
                                        T &sum) {
    const StencilHdr *h = A.st_hdr + s;
    const uint64_t bit = 1ull << (row & 63), below = bit - 1ull;
    if (h->empty & bit) return false;  // empty row: left untouched
    int t = h->tsoff;
    for (int j = 0; j < kStencilMaxTail; ++j) {
        const uint64_t mj = h->m[j];
        if (!(mj & bit)) break;
        const int e = t + __popcll(mj & below);
        sum = sum + x.at(A.st_tcol[e]) * val[A.tail_base + e];
        t += __popcll(mj);
    }
    return true;
}

// A slice's only tail entry (record kind 3): its lane, column and position
// are wavefront-uniform, so its value and operand are loads every lane of
// the wavefront shares, issued without waiting for a per-lane index.
template <class T, class V, class X>
__device__ inline void stencil_tail_one(const EllView &A, const V *__restrict__ val, const X &x, const StencilTail &tl,
                                        int row, T &sum) {
    const int lane_t = (tl.kind >> 8) & 63;
    const V tv = val[A.tail_base + tl.tsoff];
    const T xt = x.at((int)(uint32_t)tl.m0);
    if ((row & 63) == lane_t) sum = sum + xt * tv;
}

// A slice's tail record, in scalar loads.
__device__ inline StencilTail tail_rec(const_as<StencilTail> *t) {
    StencilTail r;
    r.tsoff = t->tsoff;
    r.kind = t->kind;
    r.m0 = t->m0;
    return r;
}

// The tail of a row after its slots (false for an empty row): a compact
// 16-byte record per slice; the 80-byte header only for the rare slices
// with empty rows or rows of several tail entries.
template <class T, class V, class X>
__device__ inline bool stencil_tail(const EllView &A, const V *__restrict__ val, const X &x, const StencilTail &tl,
                                    int s, int row, T &sum) {
    const int kind = tl.kind & 0xff;
    if (kind == 3) {
        stencil_tail_one(A, val, x, tl, row, sum);
    } else if (kind == 1) {
        const uint64_t bit = 1ull << (row & 63);
        if (tl.m0 & bit) {
            const int e = tl.tsoff + __popcll(tl.m0 & (bit - 1ull));
            sum = sum + x.at(A.st_tcol[e]) * val[A.tail_base + e];
        }
    } else if (kind == 2) {
        return stencil_tail_hdr(A, val, x, s, row, sum);
    }
    return true;
}

// Stencil-layout row sum: the slots in order (column row + offset, clamped
// into the vector for slots the row lacks, whose value is 0), then the
// row's tail in stored order.  The wavefront's 64 rows are one slice, so
// the slice's offsets and header are wavefront-uniform (scalar loads); a
// tail entry's position follows from the header's lane masks.
template <int SW, class T, class V, class X>
__device__ inline bool stencil_row(const EllView &A, const V *__restrict__ val, const X &x, int row, T &sum) {
    const int w = SW > 0 ? SW : A.st_w;
    const int s = __builtin_amdgcn_readfirstlane(row >> 6);
    const_as<int32_t> *off = as_const(A.st_off) + (size_t)s * w;
    const V *vs = val + (size_t)s * w * 64 + (row & 63);
    if (SW > 0) {
        int c[SW > 0 ? SW : 1];
        V v[SW > 0 ? SW : 1];
#pragma unroll
        for (int k = 0; k < SW; ++k) {
            const int cc = row + off[k];
            c[k] = cc < 0 ? 0 : (cc > A.cmax ? A.cmax : cc);
            v[k] = __builtin_nontemporal_load(&vs[64 * k]);
        }
#pragma unroll
        for (int k = 0; k < SW; ++k) sum = sum + x.at(c[k]) * v[k];
    } else {
        for (int k = 0; k < w; ++k) {
            const int cc = row + off[k];
            sum = sum + x.at(cc < 0 ? 0 : (cc > A.cmax ? A.cmax : cc)) * vs[64 * k];
        }
    }
    return stencil_tail(A, val, x, tail_rec(as_const(A.st_tail) + s), s, row, sum);
}

// Stencil-layout row sum over the symmetric form of the slot values
// (gip_layout.h, plan_symmetric): the same values in the same order as
// stencil_row, a slot of offset -d taking its value from row - d's slot of
// offset +d.  The slice's 8 slot codes are one scalar load.
template <int SW, class T, class V, class X>
__device__ inline bool stencil_row_sym(const EllView &A, const V *__restrict__ val, const V *__restrict__ sym,
                                       const X &x, int row, T &sum) {
    const int s = __builtin_amdgcn_readfirstlane(row >> 6);
    const size_t stride = (size_t)A.sym_stride;
    const_as<int32_t> *off = as_const(A.st_off) + (size_t)s * SW;
    const uint64_t codes = as_const(reinterpret_cast<const uint64_t *>(A.st_code))[s];
    int c[SW];
    V v[SW];
#pragma unroll
    for (int k = 0; k < SW; ++k) {
        const int cc = row + off[k];
        c[k] = cc < 0 ? 0 : (cc > A.cmax ? A.cmax : cc);
        // array and row of the slot's value from the (scalar) code, so that
        // every slot is one unconditional load, issued before any sum
        const int code = (int)(int8_t)(codes >> (8 * k));
        const bool lower = code >= kSymLower;
        const int j = lower ? code - kSymLower : (code < 0 ? 0 : code);
        const int d = !lower ? 0 : j == 0 ? A.sym_d[0] : j == 1 ? A.sym_d[1] : j == 2 ? A.sym_d[2] : A.sym_d[3];
        const int pr = row - d, prc = pr < 0 ? 0 : pr;
        const V u = sym[(size_t)j * stride + prc];
        v[k] = (code < 0 || pr < 0) ? V(0) : u;
    }
#pragma unroll
    for (int k = 0; k < SW; ++k) sum = sum + x.at(c[k]) * v[k];
    return stencil_tail(A, val, x, tail_rec(as_const(A.st_tail) + s), s, row, sum);
}

__device__ inline const double *dict_tab(const EllView &A, double) { return A.dc_tab; }
__device__ inline const float *dict_tab(const EllView &A, float) { return A.dc_tab32; }
__device__ inline const double *dict_soa(const EllView &A, double) { return A.dc_soa; }
__device__ inline const float *dict_soa(const EllView &A, float) { return A.dc_soa32; }

// a[i] at a 32-bit byte offset from a wavefront-uniform address: one load
// instruction with a scalar base, no vector address arithmetic.
template <class T>
__device__ inline T at_byte(const T *a, uint32_t byte) {
    return *reinterpret_cast<const T *>(reinterpret_cast<const char *>(a) + byte);
}

// One value per tuple (the inverse diagonal, say) for a row.
template <class V>
__device__ inline V dict_one(const DictSel *sel, const uint16_t *ids, const V *tuple_val, int row) {
    const_as<DictSel> *r = as_const(sel) + __builtin_amdgcn_readfirstlane(row >> 6);
    const int a = r->a, b = r->b;
    if (b < 0) return tuple_val[a + ids[row]];
    const V va = as_const(tuple_val)[a], vb = as_const(tuple_val)[b];
    return ((r->mask >> (row & 63)) & 1ull) ? vb : va;
}

// A wavefront-uniform value that is loaded by this point: the compiler
// would otherwise move a load down to its first use, into whichever branch
// that is, and string the loads out one round trip after another.
template <class T>
__device__ inline void loaded(T v) {
    asm volatile("" ::"s"(v));
}

__device__ inline DictRec dict_rec(const EllView &A, int s) {
    const_as<DictRec> *r = as_const(A.dc_rec) + s;
    DictRec q;
#pragma unroll
    for (int k = 0; k < kStencilMaxW; ++k) q.off[k] = r->off[k];
    q.a = r->a;
    q.b = r->b;
    q.mask = r->mask;
    q.col[0] = r->col[0];
    q.col[1] = r->col[1];
    q.pos = r->pos;
    q.flags = r->flags;
    return q;
}

// v of the lane before (CTRL 0x138) or after (0x130) this one; the
// wavefront's first (last) lane takes `edge`.
template <int CTRL>
__device__ inline float lane_next(float v, float edge) {
    return __int_as_float(
        __builtin_amdgcn_update_dpp(__float_as_int(edge), __float_as_int(v), CTRL, 0xf, 0xf, false));
}
template <int CTRL>
__device__ inline double lane_next(double v, double edge) {
    const long long b = __double_as_longlong(v), e = __double_as_longlong(edge);
    const int lo = __builtin_amdgcn_update_dpp((int)e, (int)b, CTRL, 0xf, 0xf, false);
    const int hi = __builtin_amdgcn_update_dpp((int)(e >> 32), (int)(b >> 32), CTRL, 0xf, 0xf, false);
    return __longlong_as_double(((long long)hi << 32) | (long long)(unsigned)lo);
}

// The operands of a fast slice: the slots' (LINE: those of the row's own
// line from the wavefront's own operands, see dict_line, and the line's
// neighbours past the slice) and the tail's.
template <int SW, class T, class V>
struct DictX {
    T x[SW], before, after, xt[2];
    V tv[2];
    int tc;  // many tails: the lane's tail column (-1: none), its value in vt
    V vt;
};

// MANY: the slice may have more than two tail entries (kDictMany).
template <bool LINE, bool MANY, int SW, class T, class V>
__device__ inline void dict_x_load(const EllView &A, const V *__restrict__ val, const T *__restrict__ x,
                                   const DictRec &r, int s, int lane, uint32_t at, DictX<SW, T, V> &q) {
#pragma unroll
    for (int k = 0; k < SW; ++k) {
        if (LINE && k >= 2 && k <= 4) continue;
        if (LINE && k == 7 && (r.flags & kDictFree)) continue;
        q.x[k] = at_byte(x + r.off[k], at);
    }
    if (LINE) {
        q.x[3 % SW] = at_byte(x, at);
        q.before = as_const(x)[s * 64 - 1];
        q.after = as_const(x)[s * 64 + 64];
    }
    if (MANY) {
        q.tc = -1;
        q.vt = V(0);
        if ((r.flags & 3u) == kDictMany) {
            const uint64_t m = (uint32_t)r.col[0] | (uint64_t)(uint32_t)r.col[1] << 32, bit = 1ull << lane;
            if (m & bit) {
                const int e = __popcll(m & (bit - 1ull));
                q.tc = A.st_tcol[r.pos - A.tail_base + e];
                q.vt = val[r.pos + e];
            }
            q.xt[0] = q.xt[1] = T(0);
            q.tv[0] = q.tv[1] = V(0);
            return;
        }
    }
    q.xt[0] = as_const(x)[r.col[0]];
    q.xt[1] = as_const(x)[r.col[1]];
    q.tv[0] = as_const(val)[r.pos];
    q.tv[1] = as_const(val)[r.pos + (int)((r.flags >> 1) & 1u)];
}

template <bool LINE, bool MANY, int SW, class T, class V>
__device__ inline void dict_x_loaded(const DictX<SW, T, V> &q) {
    if (LINE) {
        loaded(q.before);
        loaded(q.after);
    }
    if (MANY) return;
    loaded(q.xt[0]);
    loaded(q.tv[0]);
    loaded(q.xt[1]);
    loaded(q.tv[1]);
}

template <int SW, class T, class V>
__device__ inline void dict_line(const DictRec &r, DictX<SW, T, V> &q) {
    const T c = q.x[3 % SW];
    q.x[2 % SW] = lane_next<0x138>(c, q.before);
    q.x[4 % SW] = lane_next<0x130>(c, q.after);
    if (SW > 7 && (r.flags & kDictFree)) q.x[7 % SW] = c;
}

template <bool MANY, int SW, class T, class V>
__device__ inline T dict_tail(const T *__restrict__ x, const DictRec &r, const DictX<SW, T, V> &q, int lane, T sum) {
    const uint32_t nt = r.flags & 3u;
    if (MANY && nt == kDictMany) {
        if (q.tc >= 0) sum = sum + x[q.tc] * q.vt;
    } else if (nt) {
        if (lane == (int)((r.flags >> 8) & 63u)) sum = sum + q.xt[0] * q.tv[0];
        if (nt == 2 && lane == (int)((r.flags >> 16) & 63u)) sum = sum + q.xt[1] * q.tv[1];
    }
    return sum;
}

// Any other slice: everything loaded where it is used.
template <int SW, class T, class V>
__device__ inline bool dict_row_slow(const EllView &A, const V *__restrict__ val, const T *__restrict__ x,
                                     const DictRec &r, int s, int row, T &sum) {
    const int id = r.b < 0 ? r.a + A.dc_id[row] : ((r.mask >> (row & 63)) & 1ull) ? r.b : r.a;
    T xv[SW];
    V v[SW];
#pragma unroll
    for (int k = 0; k < SW; ++k) {
        const int cc = row + r.off[k];
        xv[k] = x[cc < 0 ? 0 : (cc > A.cmax ? A.cmax : cc)];
        v[k] = dict_soa(A, V(0))[(size_t)k * A.dc_n + id];
    }
    sum = T(0);
#pragma unroll
    for (int k = 0; k < SW; ++k) sum = sum + xv[k] * v[k];
    return stencil_tail(A, val, Operand<T>{x}, tail_rec(as_const(A.st_tail) + s), s, row, sum);
}

// Row sums with the slot values from the dictionary, R 256-row chunks per
// workgroup: the stored values, bit for bit, in the stored order.
// use(row, ok, any, sum, own) takes a row's sum, called by whole wavefronts
// for every slice of every chunk, a thread's rows in ascending order (ok: the
// row exists; any: it is not empty; own: with OWN, the operand at the row's
// own column, which a vector shorter than the rows may not have).
//
// With the slot values gone a product is bound by the bytes it keeps in
// flight, so a wavefront takes R slices at once: their 64-byte records in
// scalar loads, then every load of the R slices before the first is waited
// for.  Slots are loads from a scalar base (no vector address arithmetic: a
// hundred vector instructions per wavefront take as long as streaming x and
// y), the two neighbours on the row's own line come from the neighbouring
// lanes (their cache lines would be requested again while in flight), and a
// slice of at most two tuples multiplies by scalars: tuple a in all lanes,
// then tuple b in the lanes of the mask (selecting values per lane took
// three instructions per value).  Slices of more tuples gather slot by slot
// through their rows' ids, which ascend along a mesh line, so the gathers
// mostly share cache lines.
// Workgroups start in the middle of the operator and wrap around: the slices
// that take several round trips (corners and edges of the mesh, a partial
// last slice) lie in its first and last planes, where they would hold up
// the kernel's end.
__device__ inline int dict_block(int b, int G) {
    const int c = xcd_run_block(b, G) + ((G >> 1) & ~63);
    return c < G ? c : c - G;
}

template <bool OWN, bool LINE, bool TUPLES, int R, int SW, class T, class V, class USE>
__device__ inline void dict_rows_fast(const EllView &A, const V *__restrict__ val, const T *__restrict__ x,
                                      const DictRec (&r)[R], const int (&ids)[R], int s0, int lane,
                                      const USE &use) {
    DictX<SW, T, V> q[R];
    V v[TUPLES ? 1 : R][SW];
    // plain products keep their rows' numbers for the stores (formed again
    // there, the products at 256^3 take 99.2 instead of 97.7 us, in FP32 53.5
    // instead of 50.1); the solver's form them again (269.9 instead of 267.2
    // us per FP64 iteration with them kept)
    int rows[R];
#pragma unroll
    for (int u = 0; u < R; ++u) {
        const int s = s0 + u, row = s * 64 + lane;
        rows[u] = row;
        dict_x_load<LINE, !TUPLES, SW, T, V>(A, val, x, r[u], s, lane, (uint32_t)row * (uint32_t)sizeof(T), q[u]);
        if (!TUPLES) {
            const int id = r[u].b < 0 ? r[u].a + ids[u] : ((r[u].mask >> lane) & 1ull) ? r[u].b : r[u].a;
#pragma unroll
            for (int k = 0; k < SW; ++k)
                v[u % (TUPLES ? 1 : R)][k] =
                    at_byte(dict_soa(A, V(0)) + (size_t)k * A.dc_n, (uint32_t)id * (uint32_t)sizeof(V));
        }
    }
#pragma unroll
    for (int u = 0; u < R; ++u) dict_x_loaded<LINE, !TUPLES, SW, T, V>(q[u]);
#pragma unroll
    for (int u = 0; u < R; ++u) {
        const int row = OWN ? (s0 + u) * 64 + lane : rows[u];
        if (LINE) dict_line<SW, T, V>(r[u], q[u]);
        T sum = T(0);
        if (TUPLES) {
            const_as<V> *ta = as_const(dict_tab(A, V(0))) + (size_t)r[u].a * 8;
            const_as<V> *tb = as_const(dict_tab(A, V(0))) + (size_t)r[u].b * 8;
#pragma unroll
            for (int k = 0; k < SW; ++k) sum = sum + q[u].x[k] * ta[k];
            if (r[u].mask) {
                if ((r[u].mask >> lane) & 1ull) {
                    sum = T(0);
#pragma unroll
                    for (int k = 0; k < SW; ++k) sum = sum + q[u].x[k] * tb[k];
                }
            }
        } else {
#pragma unroll
            for (int k = 0; k < SW; ++k) sum = sum + q[u].x[k] * v[u % (TUPLES ? 1 : R)][k];
        }
        sum = dict_tail<!TUPLES, SW, T, V>(x, r[u], q[u], lane, sum);
        use(row, true, true, sum, !OWN ? T(0) : LINE ? q[u].x[3 % SW] : x[row]);
    }
}

template <bool OWN, int R, int SW, class T, class V, class USE>
__device__ inline void dict_rows(const EllView &A, const V *__restrict__ val, int nrows, const T *__restrict__ x,
                                 const USE &use) {
    const int ns = (nrows + 63) >> 6, lane = threadIdx.x & 63;
    const int s0 =
        (dict_block(blockIdx.x, gridDim.x) * 4 + __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6)) * R;
    const int nw = (nrows + kBlock - 1) / kBlock * (kBlock / 64);  // wavefronts of whole chunks
    if (s0 >= nw) return;
    DictRec r[R];
    int id[R];
    const bool ids = A.dc_ids != 0;
#pragma unroll
    for (int u = 0; u < R; ++u) {
        const int s = min(s0 + u, ns - 1);
        r[u] = dict_rec(A, s);
        id[u] = ids ? A.dc_id[min(s * 64 + lane, nrows - 1)] : 0;
    }
    uint32_t all = s0 + R - 1 < ns ? ~0u : 0u;
    int least = 0;
#pragma unroll
    for (int u = 0; u < R; ++u) {
#pragma unroll
        for (int k = 0; k < SW; ++k) loaded(r[u].off[k]);
        loaded(r[u].a);
        loaded(r[u].b);
        loaded(r[u].mask);
        loaded(r[u].col[0]);
        loaded(r[u].col[1]);
        loaded(r[u].pos);
        loaded(r[u].flags);
        all &= r[u].flags;
        least = min(least, (r[u].flags & 3u) == kDictMany ? -1 : r[u].b);
    }
    if (SW >= kDictLineW && (all & kDictLine)) {
        if (least >= 0)
            dict_rows_fast<OWN, true, true, R, SW, T, V>(A, val, x, r, id, s0, lane, use);
        else
            dict_rows_fast<OWN, true, false, R, SW, T, V>(A, val, x, r, id, s0, lane, use);
    } else if (all & kDictFast) {
        dict_rows_fast<OWN, false, false, R, SW, T, V>(A, val, x, r, id, s0, lane, use);
    } else {
#pragma unroll 1
        for (int u = 0; u < R; ++u) {
            const int s = s0 + u, row = s * 64 + lane;
            const bool ok = row < nrows;
            if (s >= nw) return;
            T sum = T(0), own = T(0);
            bool any = false;
            if (ok) {
                if (OWN) own = x[row];
                any = dict_row_slow<SW, T, V>(A, val, x, dict_rec(A, s), s, row, sum);
            }
            use(row, ok, any, sum, own);
        }
    }
}

// Two slices per wavefront from 2^22 rows on: at 256^3 the FP32 product
// takes 51 instead of 62 us (FP64 97 / 101), at 128^3 8.8 / 9.8 (13.4 / 12.2),
// at 97^3 7.9 / 7.3 (12.3 / 10.8): with one slice the short kernels fill the
// chip better, with two the long ones keep more loads in flight.
static inline bool dict_two(int nrows) { return nrows >= 1 << 22; }

// Launch KERNEL<7 or 8, slices per wavefront> over `chunks` 256-row chunks
#define DICT_LAUNCH(KERNEL, W, CHUNKS, ST, ...)                                    \
    do {                                                                           \
        const int ch__ = (CHUNKS);                                                 \
        if (dict_two(ch__ * kBlock)) {                                             \
            if ((W) == 7)                                                          \
                KERNEL<7, 2><<<(ch__ + 1) / 2, kBlock, 0, ST>>>(__VA_ARGS__);      \
            else                                                                   \
                KERNEL<8, 2><<<(ch__ + 1) / 2, kBlock, 0, ST>>>(__VA_ARGS__);      \
        } else if ((W) == 7) {                                                     \
            KERNEL<7, 1><<<ch__, kBlock, 0, ST>>>(__VA_ARGS__);                    \
        } else {                                                                   \
            KERNEL<8, 1><<<ch__, kBlock, 0, ST>>>(__VA_ARGS__);                    \
        }                                                                          \
    } while (0)

template <int W, class T, class V, class X>
__device__ inline bool row_dot_sym(const EllView &A, const V *__restrict__ val, const V *__restrict__ sym,
                                   const X &x, int row, T &sum) {
    static_assert(W < 0, "the symmetric form is a stencil layout");
    sum = T(0);
    return stencil_row_sym<-W, T, V, X>(A, val, sym, x, row, sum);
}

// ---- one row of a small operator, requested ahead ---------------------------
//
// The fused direction-product of the small operators forms its operand
// 1.0 s + beta p at every column it reads, with a beta that its prologue has
// yet to sum.  What the row needs from memory does not depend on beta, so
// all of it is requested before the prologue waits: the operator's row, then
// the (s, p) pairs at its columns, kept side by side so that a column is one
// load, the tail's among them.  (With the operand gathered after the sums
// and s and p apart, a kernel cost one to three round trips more: us per
// FP64 iteration, fixed count, 32^3 9.6 -> 7.1, 46^3 11.1 -> 9.3, 80^3 27.3
// -> 23.8; the irregular 60^3 in sliced ELL 20.9 -> 16.9.)

template <class T>
struct alignas(2 * sizeof(T)) SP {
    T s, p;
};

constexpr int kPreTail = 3;  // tail entries of a row requested ahead

template <int SW, class T>
struct StencilPre {
    int c[SW], tc[kPreTail];  // columns (tail: -1 none)
    T v[SW], tv[kPreTail];
    SP<T> g[SW], tg[kPreTail];
    int slice;
    bool empty, more;  // an empty row; tails beyond kPreTail in the slice (summed from the header)
};

template <int SW, class T>
__device__ inline void stencil_row_pre(const EllView &A, const T *__restrict__ val, const SP<T> *__restrict__ sp,
                                       int row, StencilPre<SW, T> &q) {
    const int s = __builtin_amdgcn_readfirstlane(row >> 6);
    const_as<int32_t> *off = as_const(A.st_off) + (size_t)s * SW;
    const T *vs = val + (size_t)s * SW * 64 + (row & 63);
    const StencilTail tl = tail_rec(as_const(A.st_tail) + s);
#pragma unroll
    for (int k = 0; k < SW; ++k) {
        const int cc = row + off[k];
        q.c[k] = cc < 0 ? 0 : (cc > A.cmax ? A.cmax : cc);
        q.v[k] = __builtin_nontemporal_load(&vs[64 * k]);
    }
#pragma unroll
    for (int k = 0; k < SW; ++k) q.g[k] = sp[q.c[k]];
    q.slice = s;
    q.empty = q.more = false;
#pragma unroll
    for (int j = 0; j < kPreTail; ++j) {
        q.tc[j] = -1;
        q.tv[j] = T(0);
    }
    const int kind = tl.kind & 0xff;
    const uint64_t bit = 1ull << (row & 63), below = bit - 1ull;
    if (kind == 3) {
        if ((row & 63) == ((tl.kind >> 8) & 63)) {
            q.tc[0] = (int)(uint32_t)tl.m0;
            q.tv[0] = val[A.tail_base + tl.tsoff];
        }
    } else if (kind) {
        const_as<StencilHdr> *h = as_const(A.st_hdr) + s;
        int t = tl.tsoff;
        uint64_t m = tl.m0;
#pragma unroll
        for (int j = 0; j < kPreTail; ++j) {
            if (m & bit) {
                const int e = t + __popcll(m & below);
                q.tc[j] = A.st_tcol[e];
                q.tv[j] = val[A.tail_base + e];
            }
            if (kind == 1) break;
            t += __popcll(m);
            m = h->m[j + 1];
            if (!m) break;
            if (j + 1 == kPreTail) q.more = true;
        }
        if (kind == 2) q.empty = (h->empty & bit) != 0;
    }
#pragma unroll
    for (int j = 0; j < kPreTail; ++j)
        if (q.tc[j] >= 0) q.tg[j] = sp[q.tc[j]];
}

// the direction at column j (past the solved rows, ghost columns, it keeps
// its value), as the direction update computes it on the solved rows
__device__ inline double dir_at(const SP<double> &q, int j, double beta, int n) {
    return j < n ? 1.0 * q.s + beta * q.p : q.p;
}
__device__ inline float dir_at(const SP<float> &q, int j, float beta, int n) {
    return j < n ? q.s + beta * q.p : q.p;
}

template <class T>
struct DirOperand {
    const SP<T> *__restrict__ sp;
    T beta;
    int n;
    __device__ inline T at(int j) const { return dir_at(sp[j], j, beta, n); }
};

// the p of the pairs (the first iteration's operand)
template <class T>
struct PairOperand {
    const SP<T> *__restrict__ sp;
    __device__ inline T at(int j) const { return sp[j].p; }
};

template <int SW, class T>
__device__ inline bool stencil_row_fin(const EllView &A, const T *__restrict__ val, const DirOperand<T> &x, int row,
                                       const StencilPre<SW, T> &q, T &sum) {
    sum = T(0);
#pragma unroll
    for (int k = 0; k < SW; ++k) sum = sum + dir_at(q.g[k], q.c[k], x.beta, x.n) * q.v[k];
    if (q.more) return stencil_tail_hdr(A, val, x, q.slice, row, sum);
#pragma unroll
    for (int j = 0; j < kPreTail; ++j)
        if (q.tc[j] >= 0) sum = sum + dir_at(q.tg[j], q.tc[j], x.beta, x.n) * q.tv[j];
    return !q.empty;
}

// uniform sliced ELL of W entries per row
template <int W, class T>
struct EllPre {
    int c[W];
    T v[W];
    SP<T> g[W];
};

template <int W, class T>
__device__ inline void ell_row_pre(const EllView &A, const T *__restrict__ val, const SP<T> *__restrict__ sp, int row,
                                   EllPre<W, T> &q) {
    const int lg = A.ell_lg;
    const int base = A.soff[row >> lg] + (row & ((1 << lg) - 1));
#pragma unroll
    for (int k = 0; k < W; ++k) {
        q.c[k] = __builtin_nontemporal_load(&A.col[base + (k << lg)]);
        q.v[k] = __builtin_nontemporal_load(&val[base + (k << lg)]);
    }
#pragma unroll
    for (int k = 0; k < W; ++k) q.g[k] = sp[q.c[k]];
}

// Row sum in stored order; returns false for an empty row.
template <int W, class T, class V, class X>
__device__ inline bool row_dot(const EllView &A, const V *__restrict__ val, const X &x, int row, T &sum) {
    sum = T(0);
    if (W < 0) {
        return stencil_row<(W < 0 ? -W : 0), T, V, X>(A, val, x, row, sum);
    } else if (W == 0 && A.fmt == GIP_FMT_STENCIL) {
        return stencil_row<0, T, V, X>(A, val, x, row, sum);
    } else if (W > 0) {
        const int lg = A.ell_lg;
        const int base = A.soff[row >> lg] + (row & ((1 << lg) - 1));
        int c[W > 0 ? W : 1];
        V v[W > 0 ? W : 1];
#pragma unroll
        for (int k = 0; k < W; ++k) {
            c[k] = __builtin_nontemporal_load(&A.col[base + (k << lg)]);
            v[k] = __builtin_nontemporal_load(&val[base + (k << lg)]);
        }
#pragma unroll
        for (int k = 0; k < W; ++k) sum = sum + x.at(c[k]) * v[k];
        return true;
    } else if (A.fmt == GIP_FMT_ELL) {
        const int lg = A.ell_lg;
        const int s = row >> lg, base = A.soff[s] + (row & ((1 << lg) - 1));
        const int width = (A.soff[s + 1] - A.soff[s]) >> lg;
        bool any = false;
        for (int k = 0; k < width; ++k) {
            const int cc = A.col[base + (k << lg)];
            if (cc < 0) break;
            sum = sum + x.at(cc) * val[base + (k << lg)];
            any = true;
        }
        return any;
    } else {
        const int jb = A.rp[row], je = A.rp[row + 1];
        for (int j = jb; j < je; ++j) sum = sum + x.at(A.col[j]) * val[j];
        return jb != je;
    }
}

// Rows of workgroup b: each XCD (b % 8) sweeps a contiguous range of
// 256-row chunks, its workgroups taking the chunks in turn.
struct RowSweep {
    int c, c1, step;
    __device__ RowSweep(int n) {
        const int nchunk = (n + kBlock - 1) / kBlock;
        const int x = blockIdx.x & 7, local = blockIdx.x >> 3;
        step = gridDim.x >> 3;
        c = (int)((int64_t)nchunk * x / 8) + local;
        c1 = (int)((int64_t)nchunk * (x + 1) / 8);
    }
};

#define FOR_ROWS(n, row)                                          \
    for (RowSweep rs__(n); rs__.c < rs__.c1; rs__.c += rs__.step) \
        for (int row = rs__.c * kBlock + (int)threadIdx.x; row < (rs__.c + 1) * kBlock && row < (n); row = (n))

// FOR_ROWS with U rows' loads in flight: load(row) requests a row's operands
// (called for every lane: a row past the sweep is read as the last row),
// use(row, operands) takes them; a thread's rows in the same order.
template <int U, class LOAD, class USE>
__device__ inline void sweep_rows(int n, const LOAD &load, const USE &use) {
    if constexpr (U == 1) {
        FOR_ROWS(n, row) use(row, load(row));
        return;
    }
    RowSweep rs(n);
    for (; rs.c < rs.c1; rs.c += U * rs.step) {
        decltype(load(0)) v[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int c = rs.c + u * rs.step, row = c * kBlock + (int)threadIdx.x;
            v[u] = load(c < rs.c1 && row < n ? row : n - 1);
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int c = rs.c + u * rs.step, row = c * kBlock + (int)threadIdx.x;
            if (c < rs.c1 && row < n) use(row, v[u]);
        }
    }
}

// A sweep whose rows can be requested ahead: U > 0, at most U rows per
// thread, all of them by ahead(), which a kernel calls before its prologue,
// and each() takes them; U = 0, each() sweeps with V rows in flight.  load
// and use as for sweep_rows.
template <int U, int V, class LOAD>
struct AheadSweep {
    const LOAD &load;
    int n;
    RowSweep rs;
    decltype(load(0)) v[U > 0 ? U : 1];
    __device__ AheadSweep(int n_, const LOAD &l) : load(l), n(n_), rs(n_) {}
    __device__ int row(int u) const { return (rs.c + u * rs.step) * kBlock + (int)threadIdx.x; }
    __device__ bool own(int u) const { return rs.c + u * rs.step < rs.c1 && row(u) < n; }
    __device__ inline void ahead() {
#pragma unroll
        for (int u = 0; u < U; ++u) v[u] = load(own(u) ? row(u) : n - 1);
    }
    template <class USE>
    __device__ inline void each(const USE &use) const {
        if constexpr (U == 0) {
            sweep_rows<V>(n, load, use);
            return;
        }
#pragma unroll
        for (int u = 0; u < U; ++u)
            if (own(u)) use(row(u), v[u]);
    }
};

// The one row of a thread, over at least as many workgroups as there are
// chunks, in RowSweep's order, so that a kernel can request its operands
// before its prologue.
struct ThreadRows {
    RowSweep rs;
    int row, n;
    __device__ explicit ThreadRows(int n_) : rs(n_), n(n_) { row = rs.c * kBlock + (int)threadIdx.x; }
    __device__ bool valid() const { return rs.c < rs.c1 && row < n; }
};

}  // namespace gip
