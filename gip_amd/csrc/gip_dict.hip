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

#include "gip_internal.h"

namespace gip {

namespace {

// Smallest operator a dictionary is made for: below it the values stay in
// the caches between products (us with the stored slots and with the
// dictionary: 64^3, the smallest, 5.0 / 4.6, 72^3 7.2 / 5.4, 97^3 16.7 / 9.9).
constexpr int kDictMinRows = 1 << 18;
// FP32 values, half of that, stay there longer (65^3 4.4 / 4.4, 81^3 4.7 /
// 5.1, 97^3 6.8 / 6.8, 104^3 8.5 / 8.8, 112^3 9.9 / 9.3; slices of at most
// two tuples 128x64x64 4.3 / 4.4, 128x128x80 9.0 / 6.7): smallest operators
// whose FP32 products read the dictionary, and where slices need ids.
constexpr int kDictMinRows32 = 1 << 20, kDictMinIds32 = 5 << 18;
// Tuples allowed: at most one per kDictRatio rows (a table of 64 bytes per
// tuple then stays under the 8 bytes per row of one vector), 2^19 in all.
constexpr int kDictRatio = 8;
constexpr int kDictMax = 1 << 19;
// Rows and columns a dictionary product addresses with 32-bit byte offsets.
constexpr int kDictMaxRows = 1 << 28;
// A slice of more than two tuples gathers each slot's values through its rows'
// ids: as many cache lines of 16 FP64 tuples as its rows have tuples in.  On
// average over the slices at most 32 of them (FP32 products: 12), past which
// the gathers take longer than streaming the stored values.  us at 128^3 of
// the product and the PCG iteration, rows scaled from k values at random, by
// lines per slice; stored FP64 29.8 and 62.9, FP32 13.9 and 48.2:
//   lines      5.9    9.9   17.5   29.4   42.0   51.1
//   FP64      17.8   19.7   21.4   25.5   34.4   44.3
//   FP64 PCG  51.0   52.5   54.6   59.1   70.0   81.5
//   FP32      12.0   13.2   15.0   16.2   18.7   37.7
//   mixed     46.6   47.2   49.2   52.6   60.3   70.2
constexpr int kDictLines = 32, kDictLines32 = 12;
constexpr int kDictProbe = 64;  // slots tried before the insert gives up
constexpr int kMaxW = kStencilMaxW + 1;  // slot values and the diagonal

struct DictTable {
    uint64_t *key;  // hash of the tuple, 0: free
    int32_t *row;   // lowest row holding it
    int32_t *id;    // its number
    uint32_t mask;  // slots - 1
    int32_t *count; // [0] tuples inserted, [1] raised when the dictionary does not fit, [2] raised when some slice needs
                    // its rows' ids, [3] the lines of those slices
    int32_t cap;
    uint64_t *first;  // per slice: the rows that are the lowest of their tuple
    int32_t *before;  // how many of those the slices before it in its run of kDictScan slices have
    int32_t *run;     // and how many the runs before
};

template <class T>
__device__ inline T dict_load(const T *p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// a word of the table that may be an earlier one: an atomic update follows
// wherever that would matter
template <class T>
__device__ inline T dict_hint(const T *p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
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

__global__ __launch_bounds__(kBlock) void k_dict_clear(DictTable T, int ns) {
    const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
    if (i < (uint32_t)ns) T.first[i] = 0;
    if (i <= T.mask) {
        T.key[i] = 0;
        T.row[i] = INT32_MAX;
    }
    if (i < 4) T.count[i] = 0;
}

// One row per thread, of which the lowest of each tuple in a wavefront goes to
// the table (the wavefront's first kDictSame tuples are told apart by their
// hashes, lanes past those go for themselves).  Run over every kDictEvery-th
// workgroup first, then over all of them, whose tuples are nearly all known by
// then and cost two cached reads.  With every row in one launch going for
// itself, the rows in flight at the start (2^19, whatever the operator's
// size) met the same few free slots, one atomic update after another, 2.5
// ms; a counter update for each new tuple took as long on an operator
// without repetition.  us now: uniform 97^3 87, 128^3 39, 256^3 270; no
// two rows alike 97^3 350, 128^3 535, 256^3 610.
constexpr int kDictSame = 4, kDictEvery = 16;
__global__ __launch_bounds__(kBlock) void k_dict_insert(DictTable T, int n, int w, const double *__restrict__ val,
                                                        const double *__restrict__ diag, int every) {
    const int r = blockIdx.x * every * kBlock + threadIdx.x, lane = threadIdx.x & 63;
    uint64_t h = 0;
    bool todo = r < n && dict_load(T.count + 1) == 0;
    if (todo) {
        uint64_t t[kMaxW];
        dict_tuple(w, val, diag, r, t);
        h = dict_hash(t);
    }
    bool mine = todo;
    for (int i = 0; i < kDictSame; ++i) {
        const uint64_t left = __ballot(todo);
        if (!left) break;
        const int first = __builtin_ctzll(left);
        const bool same = h == (uint64_t)__shfl((unsigned long long)h, first, 64);
        mine = mine && (!todo || !same || lane == first);
        todo = todo && !same;
    }
    bool added = false, lost = mine;
    uint32_t s = (uint32_t)h & T.mask;
    for (int i = 0; mine && i < kDictProbe; ++i, s = (s + 1) & T.mask) {
        uint64_t k = dict_hint(T.key + s);
        if (k == 0) {
            k = atomicCAS((unsigned long long *)T.key + s, 0ull, (unsigned long long)h);
            added = k == 0;
            if (added) k = h;
        }
        if (k == h) {
            if (dict_hint(T.row + s) > r) atomicMin(T.row + s, r);
            lost = false;
            break;
        }
    }
    const uint64_t news = __ballot(added), bad = __ballot(lost);
    if (lane) return;
    const int more = __popcll(news);
    if ((more && atomicAdd(T.count, more) + more > T.cap) || bad) atomicOr(T.count + 1, 1);
}

// the lowest row of every tuple into its slice's mask
__global__ __launch_bounds__(kBlock) void k_dict_mark(DictTable T) {
    const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
    if (i > T.mask || T.key[i] == 0) return;
    const int r = T.row[i];
    atomicOr((unsigned long long *)T.first + (r >> 6), 1ull << (r & 63));
}

// inclusive scan of one value per thread of a workgroup of kDictScan
constexpr int kDictScan = 1024;
__device__ inline int dict_scan(int v, int32_t (&sh)[kDictScan]) {
    const int t = threadIdx.x;
    sh[t] = v;
    __syncthreads();
    for (int off = 1; off < kDictScan; off *= 2) {
        const int o = t >= off ? sh[t - off] : 0;
        __syncthreads();
        sh[t] += o;
        __syncthreads();
    }
    return sh[t];
}

// The marked rows before each slice within its run of kDictScan slices, and
// the runs' totals; then, by one workgroup, the totals before each run.
__global__ __launch_bounds__(kDictScan) void k_dict_scan(DictTable T, int ns) {
    __shared__ int32_t sh[kDictScan];
    const int s = blockIdx.x * kDictScan + threadIdx.x;
    const int own = s < ns ? __popcll(T.first[s]) : 0, sum = dict_scan(own, sh);
    if (s < ns) T.before[s] = sum - own;
    if (threadIdx.x == kDictScan - 1) T.run[blockIdx.x] = sum;
}
__global__ __launch_bounds__(kDictScan) void k_dict_runs(DictTable T, int nrun) {
    __shared__ int32_t sh[kDictScan];
    int base = 0;
    for (int r0 = 0; r0 < nrun; r0 += kDictScan) {
        const int r = r0 + threadIdx.x, own = r < nrun ? T.run[r] : 0, sum = dict_scan(own, sh);
        if (r < nrun) T.run[r] = base + sum - own;
        base += sh[kDictScan - 1];
        __syncthreads();
    }
}

// The tuples, numbered by their lowest rows: their values in both table
// orders (nothing past the slots in use: 0).  (The numbers from a sort on the
// host, with a copy each way, took 0.5 to 1 ms on 97^3 with 10^4 tuples.)
__global__ __launch_bounds__(kBlock) void k_dict_fill(DictTable T, int nd, int w, const double *__restrict__ val,
                                                      const double *__restrict__ diag, double *__restrict__ tab,
                                                      double *__restrict__ soa, double *__restrict__ ddiag) {
    const uint32_t s = blockIdx.x * kBlock + threadIdx.x;
    if (s > T.mask || T.key[s] == 0) return;
    const int r = T.row[s];
    const int sl = r >> 6;
    const int i = T.run[sl / kDictScan] + T.before[sl] + __popcll(T.first[sl] & ((1ull << (r & 63)) - 1ull));
    T.id[s] = i;
    if (i >= nd) return;
    uint64_t t[kMaxW];
    dict_tuple(w, val, diag, r, t);
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
        if (b < 0) T.count[2] = 1;
        rec[sl] = q;
        sel[sl] = DictSel{a, b, mask};
    }
    if (bad) atomicOr(T.count + 1, 1);
}

__global__ __launch_bounds__(kBlock) void k_dict_f32(int64_t n, const double *__restrict__ a, float *__restrict__ b) {
    const int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x;
    if (i < n) b[i] = (float)a[i];
}

// The cache lines (16 FP64 tuples) that the slices with ids gather from, by
// a few workgroups, one update each.
constexpr int kDictLineGrid = 512;
__global__ __launch_bounds__(kBlock) void k_dict_lines(DictTable T, int n, int ns, const DictSel *__restrict__ sel,
                                                       const uint16_t *__restrict__ ids) {
    __shared__ int32_t sh[kBlock / 64];
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    int lines = 0;
    for (int s = blockIdx.x * (kBlock / 64) + wv; s < ns; s += gridDim.x * (kBlock / 64)) {
        if (sel[s].b >= 0) continue;
        const int r = s * 64 + lane;
        const int line = r < n ? (sel[s].a + ids[r]) >> 4 : -1;
        uint64_t left = __ballot(r < n);
        while (left) {
            const int of = __shfl(line, __builtin_ctzll(left), 64);
            left &= ~__ballot(line == of);
            ++lines;
        }
    }
    if (lane == 0) sh[wv] = lines;
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int k = 1; k < kBlock / 64; ++k) lines += sh[k];
        if (lines) atomicAdd(T.count + 3, lines);
    }
}

// the counters to the host
__global__ void k_dict_report(const int32_t *__restrict__ count, int32_t *__restrict__ host) {
    if (threadIdx.x < 4) host[threadIdx.x] = count[threadIdx.x];
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
    A->dict_n = A->dict_room = 0;
}

// The operator's arrays for nd tuples (kept while they are large enough: made
// anew for every change of values, allocating and freeing them took 0.6 ms);
// false when memory is not there.
static bool dict_arrays(gip_mat *A, int nd) {
    bool room = true;
    auto get = [&](auto **p, size_t count) {
        if (!room || *p) return;
        if (hipMalloc(p, count * sizeof **p) != hipSuccess) {
            (void)hipGetLastError();
            *p = nullptr;
            room = false;
        }
    };
    if (A->dict_room && nd > A->dict_room) mat_dict_free(A);
    if (A->dict_room) return true;
    get(&A->d_dict_rec, (size_t)A->nslices);
    get(&A->d_dict_sel, (size_t)A->nslices);
    get(&A->d_dict_id, (size_t)A->nrows);
    get(&A->d_dict_tab, (size_t)nd * 8);
    get(&A->d_dict_soa, (size_t)nd * A->st_w);
    get(&A->d_dict_diag, (size_t)nd);
    if (A->d_ell_val32 && A->st_w >= kDictLineW && A->nrows >= kDictMinRows32) {
        get(&A->d_dict_tab32, (size_t)nd * 8);
        get(&A->d_dict_soa32, (size_t)nd * A->st_w);
    }
    if (room) A->dict_room = nd;
    return room;
}

// scratch: device memory of `bytes` bytes to work in (gip_mat_set_values has
// the values it copied; too little: allocated).  Waits for the stream before
// it returns.
int mat_dict_build(gip_ctx *c, gip_mat *A, void *scratch, size_t bytes) {
    A->dict_n = 0;
    const int n = A->nrows, w = A->st_w;
    // products of 1 and 5 slots have no dictionary kernels (spmv_launch)
    if (A->format != GIP_FMT_STENCIL || n < kDictMinRows || n > kDictMaxRows || A->cols_needed > kDictMaxRows ||
        w < 2 || w > kStencilMaxW || w == 5 || A->no_dict || A->vals_captured) {
        mat_dict_free(A);
        return GIP_OK;
    }
    hipStream_t st = c->stream;
    DictTable T{};
    T.cap = std::min(n / kDictRatio, kDictMax);
    uint32_t slots = 1024;
    while (slots < 4u * (uint32_t)T.cap) slots *= 2;
    T.mask = slots - 1;
    // memory that is not there is no error: the operator stays as it is
    const int ns = A->nslices, nrun = (ns + kDictScan - 1) / kDictScan;
    const size_t need = (size_t)slots * 16 + 64 + (size_t)ns * 12 + (size_t)nrun * 4;
    char *own = nullptr;
    if ((!A->h_dict && hipHostMalloc((void **)&A->h_dict, 4 * sizeof(int32_t), hipHostMallocCoherent) != hipSuccess) ||
        (bytes < need && hipMalloc(&own, need) != hipSuccess)) {
        (void)hipGetLastError();
        mat_dict_free(A);
        return GIP_OK;
    }
    char *const work = own ? own : static_cast<char *>(scratch);
    T.key = reinterpret_cast<uint64_t *>(work);
    T.first = T.key + slots;
    T.row = reinterpret_cast<int32_t *>(T.first + ns);
    T.id = T.row + slots;
    T.before = T.id + slots;
    T.run = T.before + ns;
    T.count = T.run + nrun;
    // the counters reach the host by a kernel's store: with copies from the
    // device among them, the next copy to it ran at half its speed (0.45 GB of
    // values 25.5 ms instead of 14.8)
    int32_t *report = nullptr, cnt[4] = {0, 1, 0, 0};
    hipError_t e = hipHostGetDevicePointer((void **)&report, A->h_dict, 0);
    auto counts = [&]() {
        if (e != hipSuccess) return;
        k_dict_report<<<1, 64, 0, st>>>(T.count, report);
        e = hipGetLastError();
        if (e == hipSuccess) e = hipStreamSynchronize(st);
        for (int k = 0; k < 4; ++k) cnt[k] = A->h_dict[k];
    };
    if (e == hipSuccess) {
        const int every = kDictEvery;
        k_dict_clear<<<blocks(std::max((int64_t)slots, (int64_t)ns)), kBlock, 0, st>>>(T, ns);
        k_dict_insert<<<(blocks(n) + every - 1) / every, kBlock, 0, st>>>(T, n, w, A->d_ell_val, A->d_diag, every);
        k_dict_insert<<<blocks(n), kBlock, 0, st>>>(T, n, w, A->d_ell_val, A->d_diag, 1);
        counts();
    }
    const int nd = cnt[0];
    bool ok = e == hipSuccess && !cnt[1] && nd > 0 && nd <= T.cap && dict_arrays(A, nd);
    if (ok) {
        k_dict_mark<<<blocks(slots), kBlock, 0, st>>>(T);
        k_dict_scan<<<nrun, kDictScan, 0, st>>>(T, ns);
        k_dict_runs<<<1, kDictScan, 0, st>>>(T, nrun);
        k_dict_fill<<<blocks(slots), kBlock, 0, st>>>(T, nd, w, A->d_ell_val, A->d_diag, A->d_dict_tab, A->d_dict_soa,
                                                      A->d_dict_diag);
        k_dict_assign<<<blocks((int64_t)ns * 64), kBlock, 0, st>>>(
            T, n, ns, nd, w, A->d_ell_val, A->d_diag, A->d_dict_tab, A->d_dict_diag, A->d_st_off, A->d_st_tail,
            A->d_st_hdr, A->d_st_tcol, (int)A->st_tail_base, std::max(0, A->cols_needed - 1), A->d_dict_rec,
            A->d_dict_sel, A->d_dict_id);
        if (A->d_dict_tab32) {
            k_dict_f32<<<blocks((int64_t)nd * 8), kBlock, 0, st>>>((int64_t)nd * 8, A->d_dict_tab, A->d_dict_tab32);
            k_dict_f32<<<blocks((int64_t)nd * w), kBlock, 0, st>>>((int64_t)nd * w, A->d_dict_soa, A->d_dict_soa32);
        }
        k_dict_lines<<<kDictLineGrid, kBlock, 0, st>>>(T, n, ns, A->d_dict_sel, A->d_dict_id);
        counts();
        ok = e == hipSuccess && !cnt[1] && cnt[3] <= (int64_t)kDictLines * ns;
    }
    if (own) hipFree(own);
    if (!ok) mat_dict_free(A);
    if (e != hipSuccess) return hip_fail(e, "dictionary of the slot values");
    if (ok) {
        A->dict_n = nd;
        A->dict_ids = cnt[2] != 0;
        A->dict_32 = A->d_dict_soa32 && n >= (A->dict_ids ? kDictMinIds32 : kDictMinRows32) &&
                     cnt[3] <= (int64_t)kDictLines32 * ns;
        A->dict_version = A->val_version + 1;
        if (w >= kDictLineW) mat_sym_free(A);  // the solves read the dictionary in their place
    }
    return GIP_OK;
}

}  // namespace gip
