// Internal declarations shared by the HIP translation units of libgip_hip.
#pragma once

#include <hip/hip_runtime.h>

#include <atomic>
#include <cstdint>
#include <mutex>
#include <string>

#include "gip_hip.h"
#include "gip_layout.h"
#include "gip_wait.h"

namespace gip {

int set_error(int code, const std::string &msg);
int hip_fail(hipError_t e, const char *what);

#define GIP_HIP_TRY(expr)                                   \
    do {                                                    \
        hipError_t e__ = (expr);                            \
        if (e__ != hipSuccess) return gip::hip_fail(e__, #expr); \
    } while (0)

#define GIP_LAUNCH_CHECK(name)                                         \
    do {                                                               \
        hipError_t e__ = hipGetLastError();                            \
        if (e__ != hipSuccess) return gip::hip_fail(e__, name);        \
    } while (0)

constexpr int kBlock = 256;        // threads per workgroup for streaming kernels
constexpr int kMaxRedBlocks = 2048; // partial sums per reduction

// All a product needs to know about a 64-row slice of an operator with a
// dictionary, in one cache line (one scalar load): the slot offsets; which
// tuples its rows hold (b >= 0: tuple b in the lanes of `mask`, tuple a in
// the others; b < 0: row r holds tuple a + dict_id[r]); up to two tail
// entries, their columns, the position of the first value in the value
// storage (0 where there is none: a valid one) and, in `flags`, their
// number and lanes (two of one lane in their order); or, for more than two rows of one tail entry each
// (number 3), `col` as the mask of their lanes.
struct DictRec {
    int32_t off[kStencilMaxW];
    int32_t a, b;
    uint64_t mask;
    int32_t col[2];
    int32_t pos;
    uint32_t flags;  // bits 0-1: tail entries; 8-13 and 16-21: their lanes
};
// The tuples of a slice alone, for the sweeps that need only the diagonal's
// (the four slices of a workgroup's chunk share a cache line).
struct DictSel {
    int32_t a, b;
    uint64_t mask;
};
// kDictFast: a full slice (64 rows of the operator) whose slots need no
// clamp and whose tail the record describes.  kDictLine: slots 2, 3 and 4
// of it are the offsets -1, 0 and 1.  kDictFree: slot 7 is unused (offset
// 0, values 0).
constexpr uint32_t kDictFast = 1u << 24, kDictFree = 1u << 25, kDictLine = 1u << 26;
constexpr uint32_t kDictMany = 3u;
constexpr int kDictLineW = 7;  // slots from which a slice can be one of these
static_assert(sizeof(DictRec) == 64, "slice dictionary record layout");

}  // namespace gip

struct gip_ctx {
    int device;
    hipStream_t stream;
    double *d_partials;     // kMaxRedBlocks * 4 doubles of reduction partials (one per workgroup)
    double *h_result;       // pinned, coherent host block: reduction results at 0, the no-alloc
                            // solve's published words at kPubSlot, sequence words at kSeqSlot
    double *h_result_dev;   // its device address: the finalize kernels store the result there
    uint64_t seq, pub_seq;  // last sequence numbers asked for
    std::mutex sync_mu;     // gip_sync: numbers are given out in the order of the launches
    uint64_t sync_seq;
    std::atomic<bool> published;  // a result was waited for since the stream was last drained (wait_published, drain)
    int num_cu;
};

struct gip_mat {
    gip_ctx *ctx;
    int32_t nrows, ncols, nnz;
    int32_t cols_needed;  // largest column index + 1
    int32_t format;
    int32_t lanes;  // CSR: lanes per row (1, 2, 4, 8)
    // CSR (kept for every format: value get/set, transposed products, diagonal)
    int32_t *d_rowptr;
    int32_t *d_col;
    double *d_val;
    float *d_val32;
    // sliced ELL with H = 2^ell_lg rows per slice (32, 64 or 128): slice s
    // covers rows [H s, H s + H); entry k of row H s + l sits at
    // slice_off[s] + H k + l; padding has col = -1.
    int32_t ell_lg;
    int32_t nslices;
    int32_t uniform_width; // > 0 when every slice has this width and no padding
    int64_t ell_stored;
    int32_t *d_slice_off; // nslices + 1
    int32_t *d_ell_col;
    double *d_ell_val;
    float *d_ell_val32;
    int32_t *d_csr2ell;   // CSR nnz index -> position in d_ell_val (ELL and stencil)
    // stencil layout (gip_layout.h): slice s, slot k holds the entry of
    // column row + off[s W + k] of each of its 64 rows, value at
    // d_ell_val[(s W + k) 64 + lane] (0 where a row lacks that column); a
    // row's remaining entries, in stored order, form its tail, located
    // through the slice header (lane masks per tail rank); tail values at
    // d_ell_val[tail_base + t], columns d_st_tcol[t].
    int32_t st_w;
    int64_t st_tail_base;
    int32_t st_tail_nnz;
    int32_t *d_st_off;        // nslices * st_w
    gip::StencilHdr *d_st_hdr;    // nslices (read for kind-2 slices only)
    gip::StencilTail *d_st_tail;  // nslices
    int32_t *d_st_tcol;    // st_tail_nnz
    // symmetric form of the slot values (gip_layout.h, plan_symmetric), used
    // by the FP64 PCG's product: sym_nu arrays of nslices * 64 values (0: the
    // layout has none), sym_d the paired offsets, made and checked on the
    // device from the slot values at the first solve after a change of the
    // values (val_version)
    int32_t sym_nu;
    int32_t sym_d[gip::kSymMaxD];
    int64_t sym_own_slots;  // slots of offsets >= 0 over all slices
    int8_t *d_st_code;  // nslices * 8 slot codes
    uint64_t val_version;
    double *d_sym_val;
    int32_t *d_sym_flag;
    uint64_t sym_version;  // val_version + 1 the symmetric values were made from (0: never)
    int32_t sym_ok;        // 1: in use, -1: the values are not symmetric
    uint64_t sym_due;      // val_version + 1 of a solve that read the dictionary in its place
    // dictionary of the slot values (gip_dict.hip): the distinct tuples of a
    // row's slot values and diagonal, dict_n of them (0: none), current while
    // dict_version == val_version + 1
    int32_t dict_n, dict_room;  // dict_room: tuples the arrays have room for
    bool no_dict;        // GIP_MAT_NO_DICT
    bool vals_captured;  // a captured graph may change the values unseen: no form made from them is used any more
    uint64_t dict_version;
    gip::DictRec *d_dict_rec;  // per slice: which tuples its rows hold
    gip::DictSel *d_dict_sel;
    uint16_t *d_dict_id;       // per row, read for slices of more than two tuples
    int32_t dict_ids;          // there are such slices
    bool dict_32;              // FP32 products read it too
    double *d_dict_tab, *d_dict_soa, *d_dict_diag;  // tuples, 8 per row of the table; slot by slot; a_ii
    float *d_dict_tab32, *d_dict_soa32;
    int32_t *h_dict;  // pinned: the build's counters
    // a_ii per row (the stored values of a DIAG operator), for Jacobi; for
    // the other layouts refreshed from d_diag_src (each row's last diagonal
    // entry's position in the value storage, -1 for none) when values change
    double *d_diag;
    int32_t *d_diag_src;
    int32_t diag_missing;
    // lazily built transpose: structure once, values refreshed per use
    gip_mat *transpose;
    int32_t *d_tsrc;  // per transposed entry: position in this operator's value storage
    int32_t *d_tdst;  // per transposed entry: position in the transpose's value storage
};

namespace gip {
int reduce_grid(int n);

// Words a kernel hands to the host: it stores them in pinned coherent
// memory, then the sequence number (a system-scope release), and the host
// waits for that number instead of copying the words and draining the
// stream: a dot product of 97,336 entries returns in 11.9 us instead of
// 16.9, and a solver's poll costs one short kernel instead of copies and a
// synchronisation.  Work queued before the kernel has completed when the
// number arrives.
constexpr int kHostBlock = 64, kPubSlot = 8, kPubWords = 24, kSeqSlot = 40, kPubSeqSlot = 48, kSyncSlot = 56;  // doubles
int wait_published(gip_ctx *c, const uint64_t *flag, uint64_t want);
hipError_t drain(gip_ctx *c);  // hipStreamSynchronize
__device__ inline void publish_seq(uint64_t *flag, uint64_t seq) {
    __hip_atomic_store(flag, seq, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}
// Makes (once per version of the values) and checks the symmetric form of
// a stencil operator's slot values; *ok is true when the PCG's product may
// read them.  Allocates on first use.
int mat_sym_prepare(gip_ctx *c, gip_mat *A, bool *ok);
// Frees the symmetric arrays (made again when a solve needs them).
void mat_sym_free(gip_mat *A);
// Makes the dictionary of a stencil operator's slot values from its current
// values where it pays (dict_n stays 0 otherwise), and frees it.
int mat_dict_build(gip_ctx *c, gip_mat *A, void *scratch, size_t bytes);
void mat_dict_free(gip_mat *A);
inline bool mat_dict_ok(const gip_mat *A) {
    return A->dict_n > 0 && !A->vals_captured && A->dict_version == A->val_version + 1;
}
inline bool mat_dict_ok32(const gip_mat *A) { return mat_dict_ok(A) && A->dict_32; }
inline bool capturing(hipStream_t st) {
    hipStreamCaptureStatus s = hipStreamCaptureStatusNone;
    return hipStreamIsCapturing(st, &s) != hipSuccess || s != hipStreamCaptureStatusNone;
}
// ... for a product that is launched now.  A captured one reads the stored
// values: its replays take those of their own time, and the dictionary of
// today is freed when the values change.
inline bool mat_dict_now(const gip_mat *A, hipStream_t st) { return mat_dict_ok(A) && !capturing(st); }
inline bool mat_dict_now32(const gip_mat *A, hipStream_t st) { return mat_dict_ok32(A) && !capturing(st); }
// values that the device writes (gip_dcsrmv_vals)
inline void mat_values_change(gip_mat *A, hipStream_t st) {
    ++A->val_version;
    if (!A->vals_captured && capturing(st)) A->vals_captured = true;
}
// Looks up the no-alloc PCG scratch array's address on `device` (current);
// called once per device by gip_init.
int pcg_scratch_setup(int device);
}
