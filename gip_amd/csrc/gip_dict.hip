// Dictionary of a stencil operator's slot values.
//
// The operators of a uniform mesh repeat a few values: the rows of the 256^3
// Laplacian hold 18 different tuples of slot values (7157 at 255^3, whose
// face distances differ in their last bits), in 0.94 GB of stored slots.
// The dictionary keeps the distinct tuples once (bit for bit; a tuple is a
// row's slot values and its diagonal value) and says per 64-row slice which
// tuples its rows hold, so a product streams its vectors and a 64-byte
// record per slice, with 2 more bytes per row where a slice holds more than
// two tuples, instead of 8 bytes per stored slot.
//
// The FP64 product of the Laplacian by stored slots and by dictionary: 128^3
// 30.3 / 12.2 us, 200^3 118 / 58, 255^3 255 / 142, 256^3 223 / 97 (x and y
// once are 268 MB, 47 us as a copy; a bare seven-point sum of scalar
// constants with no records takes 70); FP32 256^3 104 / 51.
//
// It is made on the device when the operator's values are set from the host:
// every row's tuple is hashed into an open-addressing table whose entry
// keeps the lowest row that holds the tuple; the rows kept, in ascending
// order, number the tuples (deterministic whatever order the inserts ran
// in); every row's values are then compared with its tuple's, so a hash
// collision refuses the dictionary instead of changing a value.
#include <algorithm>
#include <vector>

#include "gip_internal.h"

namespace gip {

namespace {

// Smallest operator a dictionary is made for: below it the values stay in
// the caches between products (64^3: 4.9 us with the stored slots, 5.2 with
// the dictionary; 97^3: 17.1 and 10.8).
constexpr int kDictMinRows = 1 << 18;
// Tuples allowed: at most one per kDictRatio rows (a table of 64 bytes per
// tuple then stays under the 8 bytes per row of one vector), 2^19 in all.
constexpr int kDictRatio = 8;
constexpr int kDictMax = 1 << 19;
// Rows and columns a dictionary product addresses with 32-bit byte offsets.
constexpr int kDictMaxRows = 1 << 28;
constexpr int kDictProbe = 64;  // slots tried before the insert gives up
constexpr int kMaxW = kStencilMaxW + 1;  // slot values and the diagonal

struct DictTable {
    uint64_t *key;  // hash of the tuple, 0: free
    int32_t *row;   // lowest row holding it
    int32_t *id;    // its number
    uint32_t mask;  // slots - 1
    int32_t *count; // [0] tuples inserted, [1] raised when the dictionary does not fit, [2] tuples listed, then -1 when
                    // some slice needs its rows' ids
    int32_t cap;
};

template <class T>
__device__ inline T dict_load(const T *p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

__device__ inline uint64_t dict_mix(uint64_t h, uint64_t v) {
    h = (h ^ v) * 0x9e3779b97f4a7c15ull;
    return h ^ (h >> 29);
}

// the bits of row r's tuple
__device__ inline void dict_tuple(int w, const double *val, const double *diag, int r, uint64_t (&t)[kMaxW]) {
    const size_t base = (size_t)(r >> 6) * w * 64 + (r & 63);
#pragma unroll
    for (int k = 0; k < kStencilMaxW; ++k) t[k] = k < w ? (uint64_t)__double_as_longlong(val[base + 64 * (size_t)k]) : 0;
    t[kStencilMaxW] = (uint64_t)__double_as_longlong(diag[r]);
}

__device__ inline uint64_t dict_hash(const uint64_t (&t)[kMaxW]) {
    uint64_t h = 0x243f6a8885a308d3ull;
#pragma unroll
    for (int k = 0; k < kMaxW; ++k) h = dict_mix(h, t[k]);
    h ^= h >> 32;
    return h ? h : 1;
}

// slot of a hash that has been inserted, or -1
__device__ inline int dict_find(const DictTable &T, uint64_t h) {
    uint32_t s = (uint32_t)h & T.mask;
    for (int i = 0; i < kDictProbe; ++i, s = (s + 1) & T.mask) {
        const uint64_t k = T.key[s];
        if (k == h) return (int)s;
        if (k == 0) return -1;
    }
    return -1;
}

__global__ __launch_bounds__(kBlock) void k_dict_clear(DictTable T) {
    const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
    if (i <= T.mask) {
        T.key[i] = 0;
        T.row[i] = INT32_MAX;
    }
    if (i < 3) T.count[i] = 0;
}

// One row per thread.  Plain atomic loads come first: once a tuple is known
// its later rows cost two cached reads and no atomic update.
__global__ __launch_bounds__(kBlock) void k_dict_insert(DictTable T, int n, int w, const double *__restrict__ val,
                                                        const double *__restrict__ diag) {
    const int r = blockIdx.x * kBlock + threadIdx.x;
    if (r >= n || dict_load(T.count + 1)) return;
    uint64_t t[kMaxW];
    dict_tuple(w, val, diag, r, t);
    const uint64_t h = dict_hash(t);
    uint32_t s = (uint32_t)h & T.mask;
    for (int i = 0; i < kDictProbe; ++i, s = (s + 1) & T.mask) {
        uint64_t k = dict_load(T.key + s);
        if (k == 0) {
            k = atomicCAS((unsigned long long *)T.key + s, 0ull, (unsigned long long)h);
            if (k == 0) {
                if (atomicAdd(T.count, 1) >= T.cap) atomicOr(T.count + 1, 1);
                k = h;
            }
        }
        if (k == h) {
            if (dict_load(T.row + s) > r) atomicMin(T.row + s, r);
            return;
        }
    }
    atomicOr(T.count + 1, 1);
}

__global__ __launch_bounds__(kBlock) void k_dict_list(DictTable T, int32_t *__restrict__ rows) {
    const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
    if (i > T.mask || T.key[i] == 0) return;
    const int at = atomicAdd(T.count + 2, 1);
    if (at < T.cap) rows[at] = T.row[i];
}

// tuple i is the one of row rows[i]: its values in both table orders, its
// number into the hash table (nothing past the slots in use: 0)
__global__ __launch_bounds__(kBlock) void k_dict_fill(DictTable T, int nd, int w, const int32_t *__restrict__ rows,
                                                      const double *__restrict__ val, const double *__restrict__ diag,
                                                      double *__restrict__ tab, double *__restrict__ soa,
                                                      double *__restrict__ ddiag) {
    const int i = blockIdx.x * kBlock + threadIdx.x;
    if (i >= nd) return;
    uint64_t t[kMaxW];
    dict_tuple(w, val, diag, rows[i], t);
    const int s = dict_find(T, dict_hash(t));
    if (s < 0)
        atomicOr(T.count + 1, 1);
    else
        T.id[s] = i;
#pragma unroll
    for (int k = 0; k < kStencilMaxW; ++k) {
        const double v = __longlong_as_double((long long)t[k]);
        tab[(size_t)i * 8 + k] = v;
        if (k < w) soa[(size_t)k * nd + i] = v;
    }
    ddiag[i] = __longlong_as_double((long long)t[kStencilMaxW]);
}

// One wavefront per slice: each row's tuple (its bits compared with the
// dictionary's), then the slice's record.  Rows past the end count as the
// slice's first row.
__global__ __launch_bounds__(kBlock) void k_dict_assign(DictTable T, int n, int ns, int nd, int w,
                                                        const double *__restrict__ val,
                                                        const double *__restrict__ diag,
                                                        const double *__restrict__ tab,
                                                        const double *__restrict__ ddiag,
                                                        const int32_t *__restrict__ off,
                                                        const StencilTail *__restrict__ tail,
                                                        const StencilHdr *__restrict__ hdr,
                                                        const int32_t *__restrict__ tcol, int tail_base, int cmax,
                                                        DictRec *__restrict__ rec, DictSel *__restrict__ sel,
                                                        uint16_t *__restrict__ ids) {
    const int r = blockIdx.x * kBlock + threadIdx.x, sl = r >> 6, lane = r & 63;
    if (sl >= ns) return;  // whole wavefronts
    int id = -1;
    bool bad = false;
    if (r < n) {
        uint64_t t[kMaxW];
        dict_tuple(w, val, diag, r, t);
        const int s = dict_find(T, dict_hash(t));
        id = s < 0 ? 0 : T.id[s];
        bad = s < 0;
#pragma unroll
        for (int k = 0; k < kStencilMaxW; ++k)
            bad = bad || (uint64_t)__double_as_longlong(tab[(size_t)id * 8 + k]) != t[k];
        bad = bad || (uint64_t)__double_as_longlong(ddiag[id]) != t[kStencilMaxW];
    }
    const int first = __shfl(id, 0, 64);
    if (id < 0) id = first;
    const uint64_t same = __ballot(id == first);
    int a = first, b = first;
    uint64_t mask = 0;
    if (~same) {
        const int other = __shfl(id, __builtin_ctzll(~same), 64);
        const uint64_t second = __ballot(id == other);
        if ((same | second) == ~0ull) {
            b = other;
            mask = second;
        } else {
            int lo = id, hi = id;
#pragma unroll
            for (int off = 32; off > 0; off >>= 1) {
                lo = min(lo, __shfl_xor(lo, off, 64));
                hi = max(hi, __shfl_xor(hi, off, 64));
            }
            bad = bad || hi - lo > 0xffff;
            a = lo;
            b = -1;
            if (r < n) ids[r] = (uint16_t)(id - lo);
        }
    }
    bool out = r >= n;  // not a fast slice: a row missing, a slot's column outside the vector
    for (int k = 0; k < w; ++k) {
        const int64_t cc = (int64_t)r + off[(size_t)sl * w + k];
        out = out || cc < 0 || cc > cmax;
    }
    const bool slow = __ballot(out) != 0;
    if (lane == 0) {
        DictRec q{};
        for (int k = 0; k < w; ++k) q.off[k] = off[(size_t)sl * w + k];
        q.a = a;
        q.b = b;
        q.mask = mask;
        const StencilTail t = tail[sl];
        const int kind = t.kind & 0xff;
        bool fits = kind == 0;
        if (kind == 3) {
            q.flags = 1u | (uint32_t)((t.kind >> 8) & 63) << 8;
            q.col[0] = (int32_t)(uint32_t)t.m0;
            q.pos = tail_base + t.tsoff;
            fits = true;
        } else if (kind == 1 && __popcll(t.m0) == 2) {
            q.flags = 2u | (uint32_t)__builtin_ctzll(t.m0) << 8 | (uint32_t)(63 - __builtin_clzll(t.m0)) << 16;
            q.col[0] = tcol[t.tsoff];
            q.col[1] = tcol[t.tsoff + 1];
            q.pos = tail_base + t.tsoff;
            fits = true;
        } else if (kind == 2 && hdr[sl].empty == 0 && __popcll(hdr[sl].m[0]) == 1 && hdr[sl].m[2] == 0) {
            // one row of two entries
            const uint32_t l = (uint32_t)__builtin_ctzll(hdr[sl].m[0]);
            q.flags = 2u | l << 8 | l << 16;
            q.col[0] = tcol[t.tsoff];
            q.col[1] = tcol[t.tsoff + 1];
            q.pos = tail_base + t.tsoff;
            fits = true;
        } else if (kind == 1) {
            q.flags = kDictMany;
            q.col[0] = (int32_t)(uint32_t)t.m0;
            q.col[1] = (int32_t)(uint32_t)(t.m0 >> 32);
            q.pos = tail_base + t.tsoff;
            fits = true;
        }
        if (fits && !slow) {
            q.flags |= kDictFast;
            if (w >= kDictLineW && q.off[2] == -1 && q.off[3] == 0 && q.off[4] == 1) q.flags |= kDictLine;
        }
        if (w > 7 && q.off[7] == 0) q.flags |= kDictFree;
        if (b < 0) T.count[2] = -1;  // some slice needs its rows' ids
        rec[sl] = q;
        sel[sl] = DictSel{a, b, mask};
    }
    if (bad) atomicOr(T.count + 1, 1);
}

__global__ __launch_bounds__(kBlock) void k_dict_f32(int64_t n, const double *__restrict__ a, float *__restrict__ b) {
    const int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x;
    if (i < n) b[i] = (float)a[i];
}

inline int blocks(int64_t n) { return (int)((n + kBlock - 1) / kBlock); }

}  // namespace

void mat_dict_free(gip_mat *A) {
    void *ptrs[] = {A->d_dict_rec, A->d_dict_sel, A->d_dict_id, A->d_dict_tab, A->d_dict_soa, A->d_dict_diag, A->d_dict_tab32,
                    A->d_dict_soa32};
    for (void *p : ptrs)
        if (p) hipFree(p);
    A->d_dict_rec = nullptr;
    A->d_dict_sel = nullptr;
    A->d_dict_id = nullptr;
    A->d_dict_tab = A->d_dict_soa = A->d_dict_diag = nullptr;
    A->d_dict_tab32 = A->d_dict_soa32 = nullptr;
    A->dict_n = 0;
}

// The caller's stream has been waited for (gip_mat_create,
// gip_mat_set_values); waits for it again before it returns.
int mat_dict_build(gip_ctx *c, gip_mat *A) {
    mat_dict_free(A);
    const int n = A->nrows, w = A->st_w;
    if (A->format != GIP_FMT_STENCIL || n < kDictMinRows || n > kDictMaxRows || A->cols_needed > kDictMaxRows ||
        w < 1 || w > kStencilMaxW) return GIP_OK;
    hipStream_t st = c->stream;
    DictTable T{};
    T.cap = std::min(n / kDictRatio, kDictMax);
    uint32_t slots = 1024;
    while (slots < 4u * (uint32_t)T.cap) slots *= 2;
    T.mask = slots - 1;
    char *work = nullptr;
    int32_t *d_rows = nullptr;
    // memory that is not there is no error: the operator stays as it is
    if (hipMalloc(&work, (size_t)slots * 16 + 64) != hipSuccess) {
        (void)hipGetLastError();
        return GIP_OK;
    }
    T.key = reinterpret_cast<uint64_t *>(work);
    T.row = reinterpret_cast<int32_t *>(work + (size_t)slots * 8);
    T.id = T.row + slots;
    T.count = T.id + slots;
    k_dict_clear<<<blocks(slots), kBlock, 0, st>>>(T);
    k_dict_insert<<<blocks(n), kBlock, 0, st>>>(T, n, w, A->d_ell_val, A->d_diag);
    int32_t cnt[3] = {0, 1, 0};
    hipError_t e = hipGetLastError();
    auto counts = [&]() {
        if (e == hipSuccess) e = hipMemcpyAsync(cnt, T.count, sizeof cnt, hipMemcpyDeviceToHost, st);
        if (e == hipSuccess) e = hipStreamSynchronize(st);
    };
    counts();
    const int nd = cnt[0];
    bool ok = e == hipSuccess && !cnt[1] && nd > 0 && nd <= T.cap;
    bool room = true;
    auto get = [&](auto **p, size_t count) {
        if (ok && room && hipMalloc(p, count * sizeof **p) != hipSuccess) {
            (void)hipGetLastError();
            *p = nullptr;
            room = false;
        }
    };
    get(&d_rows, (size_t)nd);
    get(&A->d_dict_rec, (size_t)A->nslices);
    get(&A->d_dict_sel, (size_t)A->nslices);
    get(&A->d_dict_id, (size_t)n);
    get(&A->d_dict_tab, (size_t)nd * 8);
    get(&A->d_dict_soa, (size_t)nd * w);
    get(&A->d_dict_diag, (size_t)nd);
    if (A->d_ell_val32) {
        get(&A->d_dict_tab32, (size_t)nd * 8);
        get(&A->d_dict_soa32, (size_t)nd * w);
    }
    ok = ok && room;
    if (ok) {
        std::vector<int32_t> rows((size_t)nd);
        k_dict_list<<<blocks(slots), kBlock, 0, st>>>(T, d_rows);
        e = hipMemcpyAsync(rows.data(), d_rows, sizeof(int32_t) * nd, hipMemcpyDeviceToHost, st);
        if (e == hipSuccess) e = hipStreamSynchronize(st);
        std::sort(rows.begin(), rows.end());
        if (e == hipSuccess) e = hipMemcpyAsync(d_rows, rows.data(), sizeof(int32_t) * nd, hipMemcpyHostToDevice, st);
        if (e == hipSuccess) {
            k_dict_fill<<<blocks(nd), kBlock, 0, st>>>(T, nd, w, d_rows, A->d_ell_val, A->d_diag, A->d_dict_tab,
                                                       A->d_dict_soa, A->d_dict_diag);
            k_dict_assign<<<blocks((int64_t)A->nslices * 64), kBlock, 0, st>>>(
                T, n, A->nslices, nd, w, A->d_ell_val, A->d_diag, A->d_dict_tab, A->d_dict_diag, A->d_st_off,
                A->d_st_tail, A->d_st_hdr, A->d_st_tcol, (int)A->st_tail_base, std::max(0, A->cols_needed - 1), A->d_dict_rec,
                A->d_dict_sel, A->d_dict_id);
            if (A->d_dict_tab32) {
                k_dict_f32<<<blocks((int64_t)nd * 8), kBlock, 0, st>>>((int64_t)nd * 8, A->d_dict_tab, A->d_dict_tab32);
                k_dict_f32<<<blocks((int64_t)nd * w), kBlock, 0, st>>>((int64_t)nd * w, A->d_dict_soa, A->d_dict_soa32);
            }
            e = hipGetLastError();
        }
        counts();  // also: `rows` has been read
        ok = e == hipSuccess && !cnt[1];
    }
    if (d_rows) hipFree(d_rows);
    hipFree(work);
    if (!ok) mat_dict_free(A);
    if (e != hipSuccess) return hip_fail(e, "dictionary of the slot values");
    if (ok) {
        A->dict_n = nd;
        A->dict_ids = cnt[2] < 0;
        A->dict_version = A->val_version + 1;
        if (w >= kDictLineW) mat_sym_free(A);  // the solves read the dictionary in their place
    }
    return GIP_OK;
}

}  // namespace gip
