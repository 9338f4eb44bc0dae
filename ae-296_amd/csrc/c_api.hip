// extern "C" surface of libmlora_hip.so (declared in include/mlora.h): argument
// validation on the host, then one or two kernel launches on the caller's stream.
// No allocation, no synchronisation, no state kept between calls.
#include <cstdarg>
#include <cstdio>
#include <cstring>
#include <mutex>

#include "../../include/mlora.h"
#include "mlora_args.hpp"

namespace {

thread_local char g_err[512] = "";

int fail(int code, const char *fmt, ...)
{
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(g_err, sizeof(g_err), fmt, ap);
    va_end(ap);
    return code;
}

bool aligned16(const void *p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

int log2_exact(int v)
{
    for (int s = 0; s < 31; s++)
        if ((1 << s) == v) return s;
    return -1;
}

int check_pool(mlora::PoolView &pv, const int32_t *page_tbl, const int32_t *rank, const float *scaling,
               int n_adapters, int max_pages, int page_rows, int64_t n_pages, int max_rank)
{
    const int32_t *a_tbl = page_tbl, *b_tbl = page_tbl;
    const int64_t n_pages_a = n_pages, n_pages_b = n_pages;
    if (!page_tbl || !rank || !scaling) return fail(MLORA_EINVAL, "page table, rank and scaling must not be NULL");
    if (n_adapters <= 0) return fail(MLORA_EINVAL, "n_adapters must be positive (got %d)", n_adapters);
    const int shift = log2_exact(page_rows);
    if (shift < 0 || page_rows > 64) return fail(MLORA_EINVAL, "page_rows must be a power of two in 1..64 (got %d)", page_rows);
    if (max_pages <= 0) return fail(MLORA_EINVAL, "max_pages must be positive (got %d)", max_pages);
    if (max_rank < 1 || max_rank > MLORA_MAX_RANK) return fail(MLORA_ERANGE, "max_rank must be in 1..%d (got %d)", MLORA_MAX_RANK, max_rank);
    if ((int64_t)max_pages * page_rows < max_rank)
        return fail(MLORA_ERANGE, "max_pages * page_rows = %lld cannot hold max_rank %d", (long long)max_pages * page_rows, max_rank);
    if (n_pages <= 0) return fail(MLORA_EINVAL, "n_pages must be positive");
    if (n_pages_a * page_rows > 0x7fffffffLL || n_pages_b * page_rows > 0x7fffffffLL)
        return fail(MLORA_ERANGE, "a rows slab may hold at most 2^31-1 rows");
    pv.a_tbl = a_tbl; pv.b_tbl = b_tbl; pv.rank = rank; pv.scaling = scaling;
    pv.n_adapters = n_adapters; pv.max_pages = max_pages; pv.page_shift = shift;
    pv.uniform_rank = 0; pv.uniform_scale = 0.f;
    pv.n_rows_a = n_pages_a * page_rows; pv.n_rows_b = n_pages_b * page_rows;
    pv.a_dense_stride = 0; pv.b_dense_stride = 0;
    return MLORA_OK;
}

// Device memory for mlora_bgmv_multi_noalloc: the fp32 intermediate of the two-launch decode form, for
// callers that cannot allocate.  Every GPU the library runs on holds its own copy of the array at its own
// address until the process ends; host code only ever uses the per-device address looked up below, never
// the array's name (which on the host is a stand-in, not a device address).
constexpr size_t SCRATCH_BYTES = MLORA_NOALLOC_SCRATCH_BYTES;
__device__ __align__(256) unsigned char scratch[SCRATCH_BYTES];

constexpr int SCRATCH_MAX_DEVICES = 64;
std::mutex g_scratch_mu;
void *g_scratch_ptr[SCRATCH_MAX_DEVICES] = {};

// Address of the current device's copy of `scratch` (looked up once per device); nullptr + error text on failure.
void *scratch_of_current_device()
{
    int dev = -1;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) { fail(MLORA_ELAUNCH, "hipGetDevice failed: %s", hipGetErrorString(e)); return nullptr; }
    if (dev < 0 || dev >= SCRATCH_MAX_DEVICES) { fail(MLORA_ERANGE, "device ordinal %d outside [0, %d)", dev, SCRATCH_MAX_DEVICES); return nullptr; }
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    if (!g_scratch_ptr[dev]) {
        void *ptr = nullptr;
        e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
        if (e != hipSuccess || !ptr) {
            fail(MLORA_ELAUNCH, "hipGetSymbolAddress(scratch) failed on device %d: %s", dev, hipGetErrorString(e));
            return nullptr;
        }
        g_scratch_ptr[dev] = ptr;
    }
    return g_scratch_ptr[dev];
}

int check_dims(int hin, int hout)
{
    if (hin <= 0 || hout <= 0) return fail(MLORA_EINVAL, "hin and hout must be positive (got %d, %d)", hin, hout);
    if ((hin & 7) || (hout & 7)) return fail(MLORA_EALIGN, "hin and hout must be multiples of 8 (got %d, %d)", hin, hout);
    return MLORA_OK;
}

}  // namespace

namespace mlora {

int device_compute_units()
{
    static std::mutex mu;
    static int cus[SCRATCH_MAX_DEVICES] = {};
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= SCRATCH_MAX_DEVICES) return 256;
    std::lock_guard<std::mutex> lock(mu);
    if (!cus[dev]) {
        int n = 0;
        if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0) n = 256;
        cus[dev] = n;
    }
    return cus[dev];
}

}  // namespace mlora

extern "C" {

const char *mlora_last_error(void) { return g_err; }
int mlora_version(void) { return 100; }

int mlora_pool_gather(const int32_t *tok_adapter, int T, const int32_t *page_tbl, const int32_t *rank,
                      const float *scaling, int n_adapters, int max_pages, int page_rows, int64_t n_pages,
                      int32_t *out_row_off, int32_t *out_rank, float *out_scale, int32_t *perm,
                      int32_t *seg_start, int32_t *seg_len, int32_t *seg_adapter, int32_t *chunk_start,
                      int32_t *chunk_len, int32_t *chunk_adapter, int group, int32_t *counters, int32_t *work,
                      void *stream)
{
    if (T < 0) return fail(MLORA_EINVAL, "T must be >= 0 (got %d)", T);
    if (T == 0) return MLORA_OK;
    if (!tok_adapter) return fail(MLORA_EINVAL, "tok_adapter must not be NULL");
    if (n_adapters <= 0 || n_adapters > (1 << 18)) return fail(MLORA_ERANGE, "n_adapters must be in 1..262144 (got %d)", n_adapters);
    const bool per_tok = out_row_off || out_rank || out_scale;
    if (per_tok) {
        if (!page_tbl || !rank || !scaling) return fail(MLORA_EINVAL, "page_tbl, rank and scaling are needed for the per-token view");
        if (max_pages <= 0 || page_rows <= 0) return fail(MLORA_EINVAL, "max_pages and page_rows must be positive");
    }
    const bool grouped = perm || seg_start || seg_len || seg_adapter || chunk_start || chunk_len || chunk_adapter || counters || work;
    if (grouped) {
        if (!(perm && seg_start && seg_len && seg_adapter && chunk_start && chunk_len && chunk_adapter && counters))
            return fail(MLORA_EINVAL, "the grouped view needs all of perm, seg_*, chunk_* and counters");
        if (T > MLORA_GATHER_MAX_T) return fail(MLORA_ERANGE, "T = %d exceeds MLORA_GATHER_MAX_T = %d", T, MLORA_GATHER_MAX_T);
        if (group != 1 && group != 2 && group != 4 && group != 8) return fail(MLORA_EINVAL, "group must be 1, 2, 4 or 8 (got %d)", group);
        if (work) {
            if (!page_tbl || !rank || !scaling) return fail(MLORA_EINVAL, "page_tbl, rank and scaling are needed for the work records");
            if (max_pages <= 0 || page_rows <= 0 || n_pages <= 0) return fail(MLORA_EINVAL, "max_pages, page_rows and n_pages must be positive");
            if (n_pages * (int64_t)page_rows > 0x7fffffffLL) return fail(MLORA_ERANGE, "a rows slab may hold at most 2^31-1 rows");
        }
    }
    if (!per_tok && !grouped) return MLORA_OK;
    mlora::GatherArgs a;
    memset(&a, 0, sizeof(a));
    a.tok_adapter = tok_adapter; a.page_tbl = page_tbl; a.rank = rank; a.scaling = scaling;
    a.T = T; a.n_adapters = n_adapters; a.max_pages = max_pages > 0 ? max_pages : 1;
    a.page_rows = page_rows > 0 ? page_rows : 1; a.group = grouped ? group : 1;
    a.out_row_off = out_row_off; a.out_rank = out_rank; a.out_scale = out_scale;
    a.perm = perm; a.seg_start = seg_start; a.seg_len = seg_len; a.seg_adapter = seg_adapter;
    a.chunk_start = chunk_start; a.chunk_len = chunk_len; a.chunk_adapter = chunk_adapter; a.counters = counters;
    a.n_pages = n_pages; a.work = work; a.work_cap = MLORA_WORK_CAP(T);
    const int rc = mlora::launch_gather(a, static_cast<hipStream_t>(stream));
    if (rc) return fail(MLORA_ELAUNCH, "gather launch failed: %s", hipGetErrorString((hipError_t)rc));
    return MLORA_OK;
}

int mlora_pool_scatter(int n_jobs, const void *const *src, void *const *dst_slab, const int32_t *row_elems,
                       const int32_t *pages, int n_slot_pages, int rank, int page_rows, int64_t n_pages,
                       int elt_bytes, void *stream)
{
    if (n_jobs < 0 || n_jobs > MLORA_SCATTER_MAX_JOBS) return fail(MLORA_ERANGE, "n_jobs must be in 0..%d (got %d)", MLORA_SCATTER_MAX_JOBS, n_jobs);
    if (n_jobs == 0) return MLORA_OK;
    if (!src || !dst_slab || !row_elems || !pages) return fail(MLORA_EINVAL, "NULL argument array");
    if (rank < 1 || rank > MLORA_MAX_RANK) return fail(MLORA_ERANGE, "rank must be in 1..%d (got %d)", MLORA_MAX_RANK, rank);
    if (page_rows < 1 || page_rows > 64 || (page_rows & (page_rows - 1))) return fail(MLORA_EINVAL, "page_rows must be a power of two in 1..64 (got %d)", page_rows);
    if (elt_bytes != 1 && elt_bytes != 2 && elt_bytes != 4) return fail(MLORA_EINVAL, "elt_bytes must be 1, 2 or 4 (got %d)", elt_bytes);
    if (n_pages <= 0 || n_pages * (int64_t)page_rows > 0x7fffffffLL) return fail(MLORA_ERANGE, "n_pages out of range");
    const int need = (rank + page_rows - 1) / page_rows;
    if (n_slot_pages < need) return fail(MLORA_ERANGE, "rank %d needs %d pages, %d given", rank, need, n_slot_pages);
    mlora::ScatterArgs a;
    memset(&a, 0, sizeof(a));
    for (int k = 0; k < 64; k++) a.pages[k] = -1;
    for (int k = 0; k < need; k++) {
        if (pages[k] < 0 || pages[k] >= n_pages) return fail(MLORA_ERANGE, "page id %d outside [0, %lld)", pages[k], (long long)n_pages);
        a.pages[k] = pages[k];
    }
    for (int j = 0; j < n_jobs; j++) {
        if (!src[j] || !dst_slab[j]) return fail(MLORA_EINVAL, "job %d: NULL device pointer", j);
        const int64_t rb = (int64_t)row_elems[j] * elt_bytes;
        if (row_elems[j] <= 0 || (rb & 15) || rb > 0x7fffffffLL) return fail(MLORA_EALIGN, "job %d: a row must be a positive multiple of 16 bytes", j);
        if (!aligned16(src[j]) || !aligned16(dst_slab[j])) return fail(MLORA_EALIGN, "job %d: device pointers must be 16-byte aligned", j);
        a.src[j] = src[j]; a.dst[j] = dst_slab[j]; a.row_bytes[j] = (int)rb;
    }
    a.n_jobs = n_jobs; a.rank = rank; a.n_pages = n_pages;
    a.page_shift = 0;
    while ((1 << a.page_shift) < page_rows) a.page_shift++;
    const int rc = mlora::launch_scatter(a, static_cast<hipStream_t>(stream));
    if (rc) return fail(MLORA_ELAUNCH, "scatter launch failed: %s", hipGetErrorString((hipError_t)rc));
    return MLORA_OK;
}

int mlora_host_alloc(int64_t bytes, void **host_ptr, void **dev_ptr)
{
    if (bytes <= 0 || !host_ptr || !dev_ptr) return fail(MLORA_EINVAL, "bytes must be positive and the out pointers non-NULL");
    void *h = nullptr, *d = nullptr;
    hipError_t e = hipHostMalloc(&h, (size_t)bytes, hipHostMallocMapped | hipHostMallocPortable);
    if (e != hipSuccess) return fail(MLORA_ELAUNCH, "hipHostMalloc of %lld bytes failed: %s", (long long)bytes, hipGetErrorString(e));
    e = hipHostGetDevicePointer(&d, h, 0);
    if (e != hipSuccess) { (void)hipHostFree(h); return fail(MLORA_ELAUNCH, "hipHostGetDevicePointer failed: %s", hipGetErrorString(e)); }
    memset(h, 0, (size_t)bytes);
    *host_ptr = h; *dev_ptr = d;
    return MLORA_OK;
}

int mlora_host_free(void *host_ptr)
{
    if (!host_ptr) return MLORA_OK;
    const hipError_t e = hipHostFree(host_ptr);
    if (e != hipSuccess) return fail(MLORA_ELAUNCH, "hipHostFree failed: %s", hipGetErrorString(e));
    return MLORA_OK;
}

static int assist_dims(int B, int tkn, int H, int n_slots, int slot_tokens)
{
    if (B < 0 || tkn < 0) return fail(MLORA_EINVAL, "B and tkn must be >= 0 (got %d, %d)", B, tkn);
    if (H <= 0 || (H & 7)) return fail(MLORA_EALIGN, "H must be a positive multiple of 8 (got %d)", H);
    if (n_slots <= 0 || slot_tokens <= 0) return fail(MLORA_EINVAL, "n_slots and slot_tokens must be positive");
    if (B > n_slots) return fail(MLORA_ERANGE, "%d requests do not fit %d request slots", B, n_slots);
    if (tkn > slot_tokens) return fail(MLORA_ERANGE, "%d tokens per request do not fit a slot of %d", tkn, slot_tokens);
    return MLORA_OK;
}

int mlora_assist_export(const void *hidden, int B, int tkn, int H, void *x_slots, int n_slots, int slot_tokens,
                        int16_t *signals, int n_proj, int n_workers, int cap, int sig_base, int sig_stride, void *stream)
{
    int rc = assist_dims(B, tkn, H, n_slots, slot_tokens);
    if (rc) return rc;
    if (B == 0 || tkn == 0) return MLORA_OK;
    if (!hidden || !x_slots || !signals) return fail(MLORA_EINVAL, "NULL pointer");
    if (!aligned16(hidden) || !aligned16(x_slots)) return fail(MLORA_EALIGN, "hidden and x_slots must be 16-byte aligned");
    if (n_proj < 1 || n_proj > mlora::ASSIST_MAX_PROJ) return fail(MLORA_ERANGE, "n_proj must be in 1..%d (got %d)", mlora::ASSIST_MAX_PROJ, n_proj);
    if (cap <= 0) return fail(MLORA_EINVAL, "cap (tokens per worker) must be positive");
    const int64_t active = (int64_t)B * ((tkn - 1) / cap + 1);      // one worker per (request, chunk of <= cap tokens)
    if (active > n_workers) return fail(MLORA_ERANGE, "%lld workers needed per projection, %d available", (long long)active, n_workers);
    if (sig_base < 2 || sig_stride < active || (int64_t)sig_base + (int64_t)sig_stride * n_proj > 32767)
        return fail(MLORA_ERANGE, "signal codes must be > 1, distinct per projection and fit 16 bits");
    mlora::AssistArgs a;
    memset(&a, 0, sizeof(a));
    a.dev = hidden; a.host_slots[0] = x_slots; a.signals = signals;
    a.B = B; a.tkn = tkn; a.H = H; a.n_slots = n_slots; a.slot_tokens = slot_tokens;
    a.n_proj = n_proj; a.n_workers = n_workers; a.n_active = (int)active; a.sig_base = sig_base; a.sig_stride = sig_stride;
    rc = mlora::launch_assist_export(a, static_cast<hipStream_t>(stream));
    if (rc) return fail(MLORA_ELAUNCH, "export launch failed: %s", hipGetErrorString((hipError_t)rc));
    return MLORA_OK;
}

int mlora_assist_import(int n_proj, void *const *res, const void *const *out_slots, int B, int tkn, int H, int out_size,
                        int col0, int n_slots, int slot_tokens, void *stream)
{
    int rc = assist_dims(B, tkn, H, n_slots, slot_tokens);
    if (rc) return rc;
    if (B == 0 || tkn == 0) return MLORA_OK;
    if (n_proj < 1 || n_proj > mlora::ASSIST_MAX_PROJ) return fail(MLORA_ERANGE, "n_proj must be in 1..%d (got %d)", mlora::ASSIST_MAX_PROJ, n_proj);
    if (!res || !out_slots) return fail(MLORA_EINVAL, "NULL argument array");
    if (out_size <= 0 || (out_size & 7) || col0 < 0 || (col0 & 7) || col0 + out_size > H)
        return fail(MLORA_EALIGN, "out_size and col0 must be multiples of 8 with col0 + out_size <= H");
    mlora::AssistArgs a;
    memset(&a, 0, sizeof(a));
    for (int q = 0; q < n_proj; q++) {
        if (!res[q] || !out_slots[q]) return fail(MLORA_EINVAL, "projection %d: NULL pointer", q);
        if (!aligned16(res[q]) || !aligned16(out_slots[q])) return fail(MLORA_EALIGN, "projection %d: pointers must be 16-byte aligned", q);
        a.dev_out[q] = res[q]; a.host_slots[q] = const_cast<void *>(out_slots[q]);
    }
    a.B = B; a.tkn = tkn; a.H = H; a.out = out_size; a.col0 = col0; a.n_slots = n_slots; a.slot_tokens = slot_tokens;
    a.n_proj = n_proj;
    rc = mlora::launch_assist_import(a, static_cast<hipStream_t>(stream));
    if (rc) return fail(MLORA_ELAUNCH, "import launch failed: %s", hipGetErrorString((hipError_t)rc));
    return MLORA_OK;
}

int64_t mlora_bgmv_workspace_bytes(int n_proj, int T, int max_hin, int max_rank)
{
    if (n_proj < 1 || T < 1 || max_hin < 1) return 0;
    int ksc, nte;
    mlora::bgmv_split_slices(max_rank, &ksc, &nte);
    const int64_t ks = (max_hin + ksc * 8 - 1) / (ksc * 8);
    return (int64_t)n_proj * T * ks * mlora::bgmv_split_rank_stride(max_rank) * (int64_t)sizeof(float);
}

// Work items in use <= T/group + segments + 1 (one short piece per adapter present, one for the adapter-less
// tokens), rounded up to the eight record residues; the gather packs them into the first records, so the rest
// needs no workgroup.
static int items_bound(int T, int n_adapters, int group)
{
    const int64_t segs = T < n_adapters ? T : n_adapters;
    const int64_t bound = ((int64_t)(T + group - 1) / group + segs + 1 + 7) / 8 * 8;
    const int64_t cap = MLORA_WORK_CAP(T);
    return (int)(bound < cap ? bound : cap);
}

static int64_t fine_workspace_bytes(int n_proj, int T, int max_hin, int max_rank)
{
    int ksc, nte;
    mlora::bgmv_split_slices(max_rank, &ksc, &nte, false, true);
    const int64_t ks = (max_hin + ksc * 8 - 1) / (ksc * 8);
    return (int64_t)n_proj * T * ks * mlora::bgmv_split_rank_stride(max_rank) * (int64_t)sizeof(float);
}

// 512-column workgroups a call makes in the larger of its two launches.
static int64_t fine_workgroups(int n_proj, const int32_t *hin, const int32_t *hout, int items)
{
    int ksc, nte;
    mlora::bgmv_split_slices(16, &ksc, &nte, false, true);
    int64_t sh = 0, ex = 0;
    for (int p = 0; p < n_proj; p++) {
        sh += (hin[p] + ksc * 8 - 1) / (ksc * 8);
        ex += (hout[p] + nte * 8 - 1) / (nte * 8);
    }
    return (sh > ex ? sh : ex) * items;
}

// Two-launch form: 512-column slices with the rank rows split over wavefronts (fine) while they make at most four
// workgroups per compute unit, the wider slices beyond.  Measured on Llama-7B widths, wide -> fine, us per call: 8
// tokens x 7 projections (560 workgroups) 26.6 -> 21.9 at rank 64, 12.5 -> 11.7 at rank 16; 32 tokens x 3 (768)
// 23.5 -> 20.8; 16 x 7 (1120) 34.6 -> 34.8; 32 x 7 (2240) 52.4 -> 59.6.
//
// Items of four tokens are far fewer than the host's bound where adapters have several tokens, so they also take the narrow
// slices while about T/4 and two pieces for every fifth adapter make at most three workgroups per unit above rank 32 (2.5 above
// 16).  One projection, 100 adapters, Zipf 0.8, wide -> fine, us: 160 tokens of ranks 8 to 64 26.2 -> 18.2, of rank 64 29.9 ->
// 24.6, of rank 32 18.0 -> 16.8, of rank 16 12.4 -> 12.4; 256 tokens (3.25 a unit) of ranks 8 to 64 26.5 -> 21.2, of rank 64 33.1
// -> 33.7, of rank 32 18.5 -> 19.0; 100 tokens x 3 of rank 64 43.7 -> 46.4.  The estimate of pieces is that popularity's; with
// others the line holds: 162 batches below it (64 to 700 adapters, uniform, Zipf 0.8 and 1.2; 144 to 256 tokens, four widths,
// ranks 24 to 64), fine / wide 0.63 to 1.006 times; of rank 64 and uniform 0.83 to 0.98, the last with 700 adapters and 144
// tokens (134 pieces, 4.2 workgroups a unit).
static bool prefer_sliced(int n_proj, const int32_t *hin, const int32_t *hout, int T, int n_adapters, int max_rank, int group)
{
    if (group > 4) return true;
    const int64_t cus = mlora::device_compute_units();
    if (fine_workgroups(n_proj, hin, hout, items_bound(T, n_adapters, group)) <= 4 * cus) return false;
    if (group < 4 || max_rank <= 16) return true;
    const int items = (T + 3) / 4 + 2 * (T < n_adapters ? T : n_adapters) / 5;
    return 4 * fine_workgroups(n_proj, hin, hout, (items + 7) / 8 * 8) > (max_rank > 32 ? 12 : 10) * cus;
}

// How a planned decode call runs best, and the workspace its two-launch form takes (mlora_bgmv_form).
//
// Fused, one launch: every item on one compute unit, whose chain of loads grows with the bytes of an item; it saves
// a launch, which is 1.6 us of a graph and 2.6 us of host time of an eager call.  Eight layers of Llama-7B attention
// projections in a graph, fused (several workgroups an item where they fit, column_part_shift) / two fine launches, us: rank 16
// (256 KiB an item), 32 tokens x 1 projection 53 / 60, 8 x 3 55 / 61, 64 x 1 55 / 65, 64 x 3 82 / 101; rank 32 (512 KiB), 8 x 1
// 74 / 64, 32 x 1 87 / 67; with one workgroup an item 32 x 3 126 / 109, 64 x 3 (more workgroups than the fine form likes)
// 136 / 152.  So: fused up to 320 KiB an item, up to 640 KiB where the slices have filled the chip, and never where one item
// is much longer than the others (MLP widths: rank 16, 16 tokens x 7 projections 17.4 us a call with one workgroup an
// item, 14.7 fine; rank 8 11.4 with two, 11.0 fine).
static int decode_form(int n_proj, const int32_t *hin, const int32_t *hout, int T, int n_adapters, int max_rank, int group)
{
    const int64_t cus = mlora::device_compute_units();
    int64_t item_bytes = 0;
    int widest = 0;
    for (int p = 0; p < n_proj; p++) {
        const int64_t b = 2LL * max_rank * ((int64_t)hin[p] + hout[p]);
        item_bytes = b > item_bytes ? b : item_bytes;
        widest = hin[p] > widest ? hin[p] : widest;
        widest = hout[p] > widest ? hout[p] : widest;
    }
    const int64_t segs = T < n_adapters ? T : n_adapters;
    // groups of two leave one odd item for about every other adapter
    const int64_t items = group == 1 ? T : (T + 1) / 2 + segs / 2;
    const bool one_round = group <= 2 && items * n_proj <= cus;
    const bool sliced = prefer_sliced(n_proj, hin, hout, T, n_adapters, max_rank, group);
    if (one_round && widest <= 8192 && item_bytes <= (sliced ? 640 << 10 : 320 << 10)) return MLORA_FORM_FUSED;
    return sliced ? MLORA_FORM_SLICED : MLORA_FORM_FINE;
}

int mlora_bgmv_form(int n_proj, const int32_t *hin, const int32_t *hout, int T, int n_adapters, int max_rank, int group,
                    int64_t *workspace_bytes)
{
    if (n_proj < 1 || n_proj > MLORA_MAX_PROJ) return fail(MLORA_ERANGE, "n_proj must be in 1..%d (got %d)", MLORA_MAX_PROJ, n_proj);
    if (!hin || !hout || !workspace_bytes) return fail(MLORA_EINVAL, "NULL pointer");
    if (T < 0 || n_adapters <= 0) return fail(MLORA_EINVAL, "T must be >= 0 and n_adapters positive (got %d, %d)", T, n_adapters);
    if (max_rank < 1 || max_rank > MLORA_MAX_RANK) return fail(MLORA_ERANGE, "max_rank must be in 1..%d (got %d)", MLORA_MAX_RANK, max_rank);
    if (group != 1 && group != 2 && group != 4 && group != 8) return fail(MLORA_EINVAL, "group must be 1, 2, 4 or 8 (got %d)", group);
    int max_hin = 0;
    for (int p = 0; p < n_proj; p++) {
        const int rc = check_dims(hin[p], hout[p]);
        if (rc) return rc;
        max_hin = hin[p] > max_hin ? hin[p] : max_hin;
    }
    *workspace_bytes = 0;
    if (T == 0) return MLORA_FORM_FUSED;
    // Narrow slices take more room a token than wide ones, so a shorter batch that takes them can need more than a longer one:
    // the size covers every batch up to T (prefer_sliced allows them at most four workgroups a unit).
    const int64_t coarse = mlora_bgmv_workspace_bytes(n_proj, T, max_hin, max_rank);
    const int64_t most = group > 4 ? 0 : 4LL * mlora::device_compute_units() * group / fine_workgroups(n_proj, hin, hout, 1);
    const int64_t fine = most > 0 ? fine_workspace_bytes(n_proj, most < T ? (int)most : T, max_hin, max_rank) : 0;
    *workspace_bytes = coarse > fine ? coarse : fine;
    return decode_form(n_proj, hin, hout, T, n_adapters, max_rank, group);
}

// form: MLORA_FORM_*; use_scratch: with the library's own per-device scratch array as its workspace
static int bgmv_multi_impl(int form, int n_proj, void *const *y, const void *const *x, const void *const *a_rows,
                     const void *const *b_rows, const int32_t *hin, const int32_t *hout,
                     const int32_t *tok_adapter, int T, const int32_t *page_tbl, const int32_t *rank,
                     const float *scaling, int n_adapters, int max_pages, int page_rows, int64_t n_pages,
                     int max_rank, const int32_t *work, int group, void *workspace, int64_t workspace_bytes,
                     bool use_scratch, int dtype, int accumulate, void *stream)
{
    if (dtype != MLORA_F16 && dtype != MLORA_BF16) return fail(MLORA_EDTYPE, "dtype must be MLORA_F16 or MLORA_BF16 (got %d)", dtype);
    if (n_proj < 1 || n_proj > MLORA_MAX_PROJ) return fail(MLORA_ERANGE, "n_proj must be in 1..%d (got %d)", MLORA_MAX_PROJ, n_proj);
    if (T < 0) return fail(MLORA_EINVAL, "T must be >= 0 (got %d)", T);
    if (T == 0) return MLORA_OK;
    if (!y || !x || !a_rows || !b_rows || !hin || !hout) return fail(MLORA_EINVAL, "per-projection arrays must not be NULL");
    if (!tok_adapter) return fail(MLORA_EINVAL, "tok_adapter must not be NULL");
    mlora::BgmvArgs a;
    memset(&a, 0, sizeof(a));
    int rc = check_pool(a.pool, page_tbl, rank, scaling, n_adapters, max_pages, page_rows, n_pages, max_rank);
    if (rc) return rc;
    if (work) {
        if (group != 1 && group != 2 && group != 4 && group != 8) return fail(MLORA_EINVAL, "group must be 1, 2, 4 or 8 (got %d)", group);
        if (group == 8 && max_rank > 32) return fail(MLORA_ERANGE, "group 8 supports max_rank <= 32 (got %d); use group 4", max_rank);
        if (!aligned16(work)) return fail(MLORA_EALIGN, "work records must be 16-byte aligned");
    } else if (group != 1) {
        return fail(MLORA_EINVAL, "group must be 1 when work is NULL (got %d)", group);
    }
    if (form != MLORA_FORM_FUSED && !work) return fail(MLORA_EINVAL, "the two-launch form needs the work records");
    if (form == MLORA_FORM_FINE && group > 4) return fail(MLORA_EINVAL, "MLORA_FORM_FINE takes groups of 1, 2 or 4 (got %d)", group);
    int max_hin = 0, max_hout = 0;
    for (int p = 0; p < n_proj; p++) {
        if (!y[p] || !x[p] || !a_rows[p] || !b_rows[p]) return fail(MLORA_EINVAL, "projection %d: NULL device pointer", p);
        if (!aligned16(y[p]) || !aligned16(x[p]) || !aligned16(a_rows[p]) || !aligned16(b_rows[p]))
            return fail(MLORA_EALIGN, "projection %d: device pointers must be 16-byte aligned", p);
        rc = check_dims(hin[p], hout[p]);
        if (rc) return rc;
        a.y[p] = y[p]; a.x[p] = x[p]; a.a_rows[p] = a_rows[p]; a.b_rows[p] = b_rows[p];
        a.hin[p] = hin[p]; a.hout[p] = hout[p];
        max_hin = hin[p] > max_hin ? hin[p] : max_hin;
        max_hout = hout[p] > max_hout ? hout[p] : max_hout;
    }
    a.tok_adapter = tok_adapter; a.tok_adapter64 = nullptr;
    a.work = work; a.work_cap = MLORA_WORK_CAP(T);
    a.items_cap = items_bound(T, n_adapters, group);
    a.T = T; a.n_proj = n_proj; a.accumulate = accumulate ? 1 : 0;
    if (use_scratch) {
        const int64_t need = mlora_bgmv_workspace_bytes(n_proj, T, max_hin, max_rank);
        if (need > (int64_t)SCRATCH_BYTES)
            return fail(MLORA_ENOSPACE, "this call needs %lld bytes of intermediate, the allocation-free entry point holds %lld "
                        "(n_proj x T x column slices x rank); use mlora_bgmv_multi with a workspace", (long long)need, (long long)SCRATCH_BYTES);
        workspace = scratch_of_current_device();
        if (!workspace) return MLORA_ELAUNCH;
        workspace_bytes = (int64_t)SCRATCH_BYTES;
    }
    if (form != MLORA_FORM_FUSED) {
        const int64_t need_fine = fine_workspace_bytes(n_proj, T, max_hin, max_rank);
        a.fine = form == MLORA_FORM_FINE || (form == MLORA_FORM_PAIR && workspace_bytes >= need_fine &&
                                             !prefer_sliced(n_proj, hin, hout, T, n_adapters, max_rank, group));
        const int64_t need = a.fine ? need_fine : mlora_bgmv_workspace_bytes(n_proj, T, max_hin, max_rank);
        if (!workspace) return fail(MLORA_EINVAL, "the two-launch form needs a workspace");
        if (workspace_bytes < need)
            return fail(MLORA_ENOSPACE, "workspace holds %lld bytes, %lld needed", (long long)workspace_bytes, (long long)need);
        if (!aligned16(workspace)) return fail(MLORA_EALIGN, "workspace must be 16-byte aligned");
        a.vws = static_cast<float *>(workspace);
        int ksc, nte;
        mlora::bgmv_split_slices(max_rank, &ksc, &nte, false, a.fine != 0);
        a.ks_max = (max_hin + ksc * 8 - 1) / (ksc * 8);
        a.cs_max = (max_hout + nte * 8 - 1) / (nte * 8);
        int sh = 0, ex = 0;
        for (int p = 0; p < n_proj; p++) {
            sh += (hin[p] + ksc * 8 - 1) / (ksc * 8);
            ex += (hout[p] + nte * 8 - 1) / (nte * 8);
            a.sh_end[p] = sh; a.ex_end[p] = ex;
        }
        for (int p = n_proj; p < mlora::MAX_PROJ; p++) a.sh_end[p] = a.ex_end[p] = 0x7fffffff;
        rc = mlora::launch_bgmv_split(a, dtype, group, max_rank, static_cast<hipStream_t>(stream));
    } else {
        rc = mlora::launch_bgmv(a, dtype, group, max_rank, false, static_cast<hipStream_t>(stream));
    }
    if (rc) return fail(MLORA_ELAUNCH, "bgmv launch failed: %s", hipGetErrorString((hipError_t)rc));
    return MLORA_OK;
}

int mlora_bgmv_multi(int n_proj, void *const *y, const void *const *x, const void *const *a_rows,
                     const void *const *b_rows, const int32_t *hin, const int32_t *hout,
                     const int32_t *tok_adapter, int T, const int32_t *page_tbl, const int32_t *rank,
                     const float *scaling, int n_adapters, int max_pages, int page_rows, int64_t n_pages,
                     int max_rank, const int32_t *work, int group, void *workspace, int64_t workspace_bytes,
                     int dtype, int accumulate, void *stream)
{
    return bgmv_multi_impl(workspace ? MLORA_FORM_SLICED : MLORA_FORM_FUSED, n_proj, y, x, a_rows, b_rows, hin, hout, tok_adapter, T,
                           page_tbl, rank, scaling, n_adapters, max_pages, page_rows, n_pages, max_rank, work, group, workspace,
                           workspace_bytes, false, dtype, accumulate, stream);
}

int mlora_bgmv_multi_form(int form, int n_proj, void *const *y, const void *const *x, const void *const *a_rows,
                          const void *const *b_rows, const int32_t *hin, const int32_t *hout,
                          const int32_t *tok_adapter, int T, const int32_t *page_tbl, const int32_t *rank,
                          const float *scaling, int n_adapters, int max_pages, int page_rows, int64_t n_pages,
                          int max_rank, const int32_t *work, int group, void *workspace, int64_t workspace_bytes,
                          int dtype, int accumulate, void *stream)
{
    if (form < MLORA_FORM_FUSED || form > MLORA_FORM_PAIR) return fail(MLORA_EINVAL, "form must be one of MLORA_FORM_* (got %d)", form);
    return bgmv_multi_impl(form, n_proj, y, x, a_rows, b_rows, hin, hout, tok_adapter, T, page_tbl, rank, scaling, n_adapters,
                           max_pages, page_rows, n_pages, max_rank, work, group, workspace, workspace_bytes, false, dtype,
                           accumulate, stream);
}

int mlora_bgmv_multi_noalloc(int n_proj, void *const *y, const void *const *x, const void *const *a_rows,
                             const void *const *b_rows, const int32_t *hin, const int32_t *hout,
                             const int32_t *tok_adapter, int T, const int32_t *page_tbl, const int32_t *rank,
                             const float *scaling, int n_adapters, int max_pages, int page_rows, int64_t n_pages,
                             int max_rank, const int32_t *work, int group, int dtype, int accumulate, void *stream)
{
    if (!work) return fail(MLORA_EINVAL, "mlora_bgmv_multi_noalloc needs the work records of mlora_pool_gather");
    return bgmv_multi_impl(MLORA_FORM_SLICED, n_proj, y, x, a_rows, b_rows, hin, hout, tok_adapter, T, page_tbl, rank, scaling,
                           n_adapters, max_pages, page_rows, n_pages, max_rank, work, group, nullptr, 0, true, dtype, accumulate,
                           stream);
}

int mlora_bgmv(void *y, const void *x, const void *a_rows, const void *b_rows, const int32_t *tok_adapter,
               const int32_t *page_tbl, const int32_t *rank, const float *scaling, int T, int hin, int hout,
               int n_adapters, int max_pages, int page_rows, int64_t n_pages, int max_rank, int dtype,
               int accumulate, void *stream)
{
    void *ys[1] = {y};
    const void *xs[1] = {x}, *as[1] = {a_rows}, *bs[1] = {b_rows};
    const int32_t hi[1] = {hin}, ho[1] = {hout};
    return mlora_bgmv_multi(1, ys, xs, as, bs, hi, ho, tok_adapter, T, page_tbl, rank, scaling, n_adapters,
                            max_pages, page_rows, n_pages, max_rank, nullptr, 1, nullptr, 0, dtype, accumulate, stream);
}

int mlora_bgmv_reflayout(void *y, const void *x, const void *wa_T_all, const void *wb_T_all,
                         const int64_t *indices, int T, int N, int L, int r, int hin, int hout, int layer_idx,
                         float scale, int dtype, void *stream)
{
    if (dtype != MLORA_F16 && dtype != MLORA_BF16) return fail(MLORA_EDTYPE, "dtype must be MLORA_F16 or MLORA_BF16 (got %d)", dtype);
    if (T < 0) return fail(MLORA_EINVAL, "T must be >= 0 (got %d)", T);
    if (T == 0) return MLORA_OK;
    if (!y || !x || !wa_T_all || !wb_T_all || !indices) return fail(MLORA_EINVAL, "NULL device pointer");
    if (N <= 0 || L <= 0) return fail(MLORA_EINVAL, "N and L must be positive (got %d, %d)", N, L);
    if (layer_idx < 0 || layer_idx >= L) return fail(MLORA_ERANGE, "layer_idx %d outside [0, %d)", layer_idx, L);
    if (r < 1 || r > MLORA_MAX_RANK) return fail(MLORA_ERANGE, "rank must be in 1..%d (got %d)", MLORA_MAX_RANK, r);
    int rc = check_dims(hin, hout);
    if (rc) return rc;
    if (!aligned16(y) || !aligned16(x) || !aligned16(wa_T_all) || !aligned16(wb_T_all))
        return fail(MLORA_EALIGN, "device pointers must be 16-byte aligned");
    if ((int64_t)N * L * r > 0x7fffffffLL) return fail(MLORA_ERANGE, "pool has more than 2^31-1 rank rows");
    mlora::BgmvArgs a;
    memset(&a, 0, sizeof(a));
    mlora::PoolView &pv = a.pool;
    pv.a_tbl = nullptr; pv.b_tbl = nullptr; pv.rank = nullptr; pv.scaling = nullptr;
    pv.n_adapters = N; pv.max_pages = 1; pv.page_shift = 0;
    pv.uniform_rank = r; pv.uniform_scale = scale;
    // A: rank rows of adapter i, layer l start at row (i*L + l)*r; the layer offset goes into the base pointer.
    pv.a_dense_stride = (long long)L * r;
    pv.n_rows_a = (long long)(N - 1) * L * r + r;
    // B^T: [hout, r] block of adapter i, layer l starts at element (i*L + l)*hout*r.
    pv.b_dense_stride = (long long)L * hout * r;
    pv.n_rows_b = 0;
    a.y[0] = y; a.x[0] = x;
    a.a_rows[0] = static_cast<const uint16_t *>(wa_T_all) + (size_t)layer_idx * r * hin;
    a.b_rows[0] = static_cast<const uint16_t *>(wb_T_all) + (size_t)layer_idx * hout * r;
    if (!aligned16(a.a_rows[0]) || !aligned16(a.b_rows[0]))
        return fail(MLORA_EALIGN, "layer slab of the pool is not 16-byte aligned (r * hin and hout * r must be multiples of 8)");
    a.hin[0] = hin; a.hout[0] = hout;
    a.tok_adapter = nullptr; a.tok_adapter64 = indices;
    a.T = T; a.n_proj = 1; a.accumulate = 1;
    rc = mlora::launch_bgmv(a, dtype, 1, r, true, static_cast<hipStream_t>(stream));
    if (rc) return fail(MLORA_ELAUNCH, "bgmv launch failed: %s", hipGetErrorString((hipError_t)rc));
    return MLORA_OK;
}

// Plan buffer of the reference-layout decode call: perm, seg_start, seg_len, seg_adapter, chunk_start, chunk_len,
// chunk_adapter (T int32 each, padded to 16 bytes), counters, then the work records.
static int64_t ref_plan_words(int T) { return ((int64_t)T + 3) / 4 * 4; }

int64_t mlora_reflayout_plan_bytes(int T)
{
    if (T <= 0) return 0;
    return (7 * ref_plan_words(T) + MLORA_CNT_WORDS + (int64_t)MLORA_WORK_CAP(T) * MLORA_WORK_WORDS) * (int64_t)sizeof(int32_t);
}

static int32_t *ref_plan_work(void *plan, int T) { return static_cast<int32_t *>(plan) + 7 * ref_plan_words(T) + MLORA_CNT_WORDS; }

static int ref_rank_ok(int r) { return r == 8 || r == 16 || r == 32 || r == 64; }

int mlora_reflayout_plan(const int64_t *indices, int T, int N, int L, int r, int group, void *plan, int64_t plan_bytes,
                         void *stream)
{
    if (T < 0) return fail(MLORA_EINVAL, "T must be >= 0 (got %d)", T);
    if (T == 0) return MLORA_OK;
    if (!indices || !plan) return fail(MLORA_EINVAL, "NULL pointer");
    if (T > MLORA_GATHER_MAX_T) return fail(MLORA_ERANGE, "T = %d exceeds MLORA_GATHER_MAX_T = %d", T, MLORA_GATHER_MAX_T);
    if (N <= 0 || N > (1 << 18) || L <= 0) return fail(MLORA_ERANGE, "N must be in 1..262144 and L positive (got %d, %d)", N, L);
    if (!ref_rank_ok(r)) return fail(MLORA_ERANGE, "the grouped reference-layout call needs rank 8, 16, 32 or 64 (got %d); mlora_bgmv_reflayout takes any rank", r);
    if (group != 1 && group != 2 && group != 4) return fail(MLORA_EINVAL, "group must be 1, 2 or 4 (got %d)", group);
    if ((int64_t)N * L * r > 0x7fffffffLL) return fail(MLORA_ERANGE, "pool has more than 2^31-1 rank rows");
    if (!aligned16(plan)) return fail(MLORA_EALIGN, "plan buffer must be 16-byte aligned");
    if (plan_bytes < mlora_reflayout_plan_bytes(T))
        return fail(MLORA_ENOSPACE, "plan buffer holds %lld bytes, %lld needed", (long long)plan_bytes, (long long)mlora_reflayout_plan_bytes(T));
    mlora::GatherArgs a;
    memset(&a, 0, sizeof(a));
    int32_t *ip = static_cast<int32_t *>(plan);
    const int64_t w = ref_plan_words(T);
    a.tok_adapter64 = indices;
    a.T = T; a.n_adapters = N; a.max_pages = 1; a.page_rows = 1; a.group = group;
    // rank row j of adapter a, relative to a layer's first row: a * L * r + j (wa_T_all is [N, L, r, hin])
    a.dense_stride = (long long)L * r; a.n_rows_dense = (long long)(N - 1) * L * r + r;
    a.uniform_rank = r; a.uniform_scale = 1.0f;
    a.perm = ip; a.seg_start = ip + w; a.seg_len = ip + 2 * w; a.seg_adapter = ip + 3 * w;
    a.chunk_start = ip + 4 * w; a.chunk_len = ip + 5 * w; a.chunk_adapter = ip + 6 * w; a.counters = ip + 7 * w;
    a.n_pages = 1; a.work = ref_plan_work(plan, T); a.work_cap = MLORA_WORK_CAP(T);
    const int rc = mlora::launch_gather(a, static_cast<hipStream_t>(stream));
    if (rc) return fail(MLORA_ELAUNCH, "gather launch failed: %s", hipGetErrorString((hipError_t)rc));
    return MLORA_OK;
}

int mlora_bgmv_reflayout_multi(int n_proj, void *const *y, const void *const *x, const void *const *wa_T_all,
                               const void *const *wb_T_all, const int32_t *hin, const int32_t *hout, const void *plan,
                               int T, int N, int L, int r, int layer_idx, float scale, int group, int dtype,
                               int accumulate, void *workspace, int64_t workspace_bytes, void *stream)
{
    if (dtype != MLORA_F16 && dtype != MLORA_BF16) return fail(MLORA_EDTYPE, "dtype must be MLORA_F16 or MLORA_BF16 (got %d)", dtype);
    if (n_proj < 1 || n_proj > MLORA_MAX_PROJ) return fail(MLORA_ERANGE, "n_proj must be in 1..%d (got %d)", MLORA_MAX_PROJ, n_proj);
    if (T < 0) return fail(MLORA_EINVAL, "T must be >= 0 (got %d)", T);
    if (T == 0) return MLORA_OK;
    if (!y || !x || !wa_T_all || !wb_T_all || !hin || !hout || !plan) return fail(MLORA_EINVAL, "NULL pointer");
    if (N <= 0 || L <= 0) return fail(MLORA_EINVAL, "N and L must be positive (got %d, %d)", N, L);
    if (layer_idx < 0 || layer_idx >= L) return fail(MLORA_ERANGE, "layer_idx %d outside [0, %d)", layer_idx, L);
    if (!ref_rank_ok(r)) return fail(MLORA_ERANGE, "the grouped reference-layout call needs rank 8, 16, 32 or 64 (got %d); mlora_bgmv_reflayout takes any rank", r);
    if (group != 1 && group != 2 && group != 4) return fail(MLORA_EINVAL, "group must be 1, 2 or 4 (got %d)", group);
    if ((int64_t)N * L * r > 0x7fffffffLL) return fail(MLORA_ERANGE, "pool has more than 2^31-1 rank rows");
    if (!aligned16(plan)) return fail(MLORA_EALIGN, "plan buffer must be 16-byte aligned");
    mlora::BgmvArgs a;
    memset(&a, 0, sizeof(a));
    mlora::PoolView &pv = a.pool;
    pv.n_adapters = N; pv.max_pages = 1; pv.page_shift = 0;
    pv.uniform_rank = r; pv.uniform_scale = scale;
    pv.a_dense_stride = (long long)L * r;
    pv.n_rows_a = (long long)(N - 1) * L * r + r;
    int max_hin = 0, max_hout = 0;
    for (int p = 0; p < n_proj; p++) {
        if (!y[p] || !x[p] || !wa_T_all[p] || !wb_T_all[p]) return fail(MLORA_EINVAL, "projection %d: NULL device pointer", p);
        int rc = check_dims(hin[p], hout[p]);
        if (rc) return rc;
        a.y[p] = y[p]; a.x[p] = x[p];
        a.a_rows[p] = static_cast<const uint16_t *>(wa_T_all[p]) + (size_t)layer_idx * r * hin[p];
        a.b_rows[p] = static_cast<const uint16_t *>(wb_T_all[p]) + (size_t)layer_idx * hout[p] * r;
        if (!aligned16(a.y[p]) || !aligned16(a.x[p]) || !aligned16(a.a_rows[p]) || !aligned16(a.b_rows[p]))
            return fail(MLORA_EALIGN, "projection %d: device pointers must be 16-byte aligned", p);
        a.hin[p] = hin[p]; a.hout[p] = hout[p];
        max_hin = hin[p] > max_hin ? hin[p] : max_hin;
        max_hout = hout[p] > max_hout ? hout[p] : max_hout;
    }
    a.b_transposed = 1; a.ref_layers = L;
    a.tok_adapter = nullptr; a.tok_adapter64 = nullptr;
    a.work = ref_plan_work(const_cast<void *>(plan), T); a.work_cap = MLORA_WORK_CAP(T);
    a.items_cap = items_bound(T, N, group);
    a.T = T; a.n_proj = n_proj; a.accumulate = accumulate ? 1 : 0;
    const int64_t need = mlora_bgmv_workspace_bytes(n_proj, T, max_hin, r);
    if (!workspace || !aligned16(workspace)) return fail(MLORA_EALIGN, "workspace must be a 16-byte aligned device pointer");
    if (workspace_bytes < need) return fail(MLORA_ENOSPACE, "workspace holds %lld bytes, %lld needed", (long long)workspace_bytes, (long long)need);
    a.vws = static_cast<float *>(workspace);
    int ksc, nte;
    mlora::bgmv_split_slices(r, &ksc, &nte, true);
    a.ks_max = (max_hin + ksc * 8 - 1) / (ksc * 8);
    a.cs_max = (max_hout + nte * 8 - 1) / (nte * 8);
    int sh = 0, ex = 0;
    for (int p = 0; p < n_proj; p++) {
        sh += (hin[p] + ksc * 8 - 1) / (ksc * 8);
        ex += (hout[p] + nte * 8 - 1) / (nte * 8);
        a.sh_end[p] = sh; a.ex_end[p] = ex;
    }
    for (int p = n_proj; p < mlora::MAX_PROJ; p++) a.sh_end[p] = a.ex_end[p] = 0x7fffffff;
    const int rc = mlora::launch_bgmv_split(a, dtype, group, r, static_cast<hipStream_t>(stream));
    if (rc) return fail(MLORA_ELAUNCH, "bgmv launch failed: %s", hipGetErrorString((hipError_t)rc));
    return MLORA_OK;
}

}  // extern "C"

namespace {

constexpr int SG_TM = 64;   // tokens per tile, as in sgmv_prefill.hip

struct SgmvWs { int max_tiles; int ks_cap; size_t off_cover, off_rec, off_proj, per_proj, off_hi, off_lo, total; };

// Workspace: the plan (tile list, tile records: depends on T and n_seg only), then per projection the
// K-split partial sums and the hi / lo halves of their sum.  `cap`: splits that there is room for at most.
SgmvWs sgmv_layout_splits(int T, int n_seg, int n_proj, int cap)
{
    SgmvWs w;
    w.max_tiles = T / SG_TM + 2 * n_seg + 1;       // aligned cuts can add one partial tile at either end of a segment
    // Room for the splits that a call of this size has a use for (shrink_shape chooses among those): all eight for a short
    // batch; for longer ones as many as make about 1024 workgroups of a tile, projection and split each (768 for a single
    // projection), and up to three times as many for a projection with a longer K than the others of its call.
    const long long per_split = (long long)w.max_tiles * n_proj;
    const long long target = n_proj > 1 ? 1024 : 768;
    long long ks = (target + per_split - 1) / per_split;
    ks = n_proj > 1 ? 3 * ks : ks;
    w.ks_cap = ks < cap ? (int)ks : cap;
    size_t off = ((size_t)w.max_tiles * 3 + 4) * sizeof(int32_t);
    off = (off + 255) & ~(size_t)255;
    w.off_cover = off;                              // int32 [T]: 1 where a token belongs to some segment
    off += (size_t)T * sizeof(int32_t);
    off = (off + 255) & ~(size_t)255;
    w.off_rec = off;
    off += (size_t)w.max_tiles * 80 * sizeof(int32_t);
    off = (off + 255) & ~(size_t)255;
    w.off_proj = off;
    w.off_hi = (size_t)w.ks_cap * T * MLORA_MAX_RANK * sizeof(float);
    w.off_lo = w.off_hi + (size_t)T * MLORA_MAX_RANK * sizeof(uint16_t);
    w.per_proj = (w.off_lo + (size_t)T * MLORA_MAX_RANK * sizeof(uint16_t) + 255) & ~(size_t)255;
    w.total = off + w.per_proj * n_proj;
    return w;
}

// The layout for a workspace of `have` bytes (negative: as large as the call can use).
// The number of splits steps up as a batch gets shorter, so a shorter batch can have a use for more workspace than a longer
// one, and fewer projections for more than many; where `have` does not hold the room for all of them, it holds as
// many as fit, down to one: with one split the size only grows with tokens, segments and
// projections, so a workspace sized for a larger call always serves a smaller one.
SgmvWs sgmv_layout(int T, int n_seg, int n_proj, int64_t have = -1)
{
    const SgmvWs w = sgmv_layout_splits(T, n_seg, n_proj, mlora::SGMV_SPLITS);
    if (have < 0 || (int64_t)w.total <= have) return w;
    const int64_t split = (int64_t)T * MLORA_MAX_RANK * (int64_t)sizeof(float);        // as large as the hi / lo halves together
    const int64_t fit = (have - (int64_t)w.off_proj) / n_proj / split - 1;
    return sgmv_layout_splits(T, n_seg, n_proj, fit < 1 ? 1 : (int)fit);
}

// Columns of y one expand workgroup covers, and the column blocks per tile that follow from it.
// 512 columns amortise the V operand; fewer when that leaves the chip idle (few tiles or projections), and a block
// count per tile that the tile-major order of the expand can use (a multiple of eight or just below one):
// otherwise the width that gives the nearest multiple of eight blocks, in whole cache lines.
int expand_block_cols(int n_proj, int max_tiles, int hout, int *ncb_out)
{
    int cols = 512;
    while (cols > 128 && (long long)max_tiles * n_proj * ((hout + cols - 1) / cols) < 1024) cols >>= 1;
    int ncb = (hout + cols - 1) / cols;
    if (!mlora::tile_major(ncb) && ncb >= 6) {
        const int n8 = ((ncb + 3) / 8) * 8 > 0 ? ((ncb + 3) / 8) * 8 : 8;
        const int c8 = ((hout + n8 - 1) / n8 + 63) / 64 * 64;
        if (c8 >= 256 && c8 <= 1024 && mlora::tile_major((hout + c8 - 1) / c8)) { cols = c8; ncb = (hout + c8 - 1) / c8; }
    }
    if (ncb_out) *ncb_out = ncb;
    return cols;
}

// K splits of a projection of `hin` columns where the narrowest of its call gets k: in proportion to the width, at least eight
// stages of 64 columns a split, and what the workspace holds.
int splits_of(int hin, int hin_min, int k, const SgmvWs &w)
{
    const int most = (hin + 511) / 512 < mlora::SGMV_SPLITS ? (hin + 511) / 512 : mlora::SGMV_SPLITS;
    int ks = (int)(((long long)k * hin + hin_min / 2) / hin_min);
    ks = ks < 1 ? 1 : (ks > most ? most : ks);
    return ks < w.ks_cap ? ks : w.ks_cap;
}

// Shape of a prefill call's shrink launch: whether a workgroup serves up to three projections of one x (share_x), the groups, and
// the K splits.  More splits and single projections make more and shorter workgroups; fewer splits mean fewer partial
// sums, shared x fewer lines from L2.  The rule estimates the launch for both kinds and four numbers of splits, and takes
// the least: workgroups of known length (4 ns a 128-byte line and compute unit) dealt, longest first, to the slots of the
// device; what all lines take together (2 us and 6.4 TB/s); the longer of the two and 0.3 of the other; 0.2 ns a split, token
// and projection (written, and read by the reduce launch or the expand).  Fitted to those eight shapes over 52 batches of 16
// to 9216 tokens (ranks 16 to 64; one, three, four and seven projections): the shape it names is 0.9 % off the best on
// average and 9 % at worst.  Llama-7B widths, rank 64, q/k/v, two layers and the plan in a graph, single / shared
// projections at 1, 2, 4 splits, us: 64 tokens 53, 41, 35 / 110, 67, 50; 1280 tokens 86, 81, 87 / 137, 101, 85; 6000 tokens 211,
// 211, 229 / 232, 202, 213.  The rule takes the host 0.2 us (q, k, v) to 1.0 us (seven projections) a call.
void shrink_shape(mlora::SgmvArgs &a, int tiles, int max_rank, const SgmvWs &w)
{
    static const int tried[] = {1, 2, 4, mlora::SGMV_SPLITS};
    const int cus = mlora::device_compute_units(), rows = max_rank <= 16 ? 16 : (max_rank <= 32 ? 32 : 64);
    int hin_min = a.pr[0].hin;
    for (int p = 1; p < a.n_proj; p++) hin_min = a.pr[p].hin < hin_min ? a.pr[p].hin : hin_min;
    // up to three consecutive projections that read the same activations form a group
    a.n_grp = 0;
    for (int p = 0; p < a.n_proj; p++) {
        if (p > 0 && a.pr[p].x == a.pr[p - 1].x && a.pr[p].hin == a.pr[p - 1].hin && a.grp_n[a.n_grp - 1] < 3) a.grp_n[a.n_grp - 1]++;
        else { a.grp_first[a.n_grp] = p; a.grp_n[a.n_grp] = 1; a.n_grp++; }
    }
    double best = 0.0;
    int best_k = 1;
    for (int share = 0; share <= (a.seg_uniform_len == 0 ? 1 : 0); share++) {
        // workgroups a unit holds, by their LDS (sh_group_bytes in sgmv_prefill.hip)
        const long long slots = (long long)cus * (rows == 16 || (share && rows == 32) ? 2 : 1);
        for (int t = 0; t < 4; t++) {
            const int k = tried[t];
            long long count[MLORA_MAX_PROJ];
            double len[MLORA_MAX_PROJ], lines = 0.0, parts = 0.0;
            for (int g = 0; g < a.n_grp; g++) {
                const int hin = a.pr[a.grp_first[g]].hin, nm = a.grp_n[g], stages = (hin + 63) / 64, ks = splits_of(hin, hin_min, k, w);
                count[g] = (long long)tiles * ks * (share ? 1 : nm);
                len[g] = (double)((stages + ks - 1) / ks) * (64 + (share ? nm : 1) * rows);
                lines += (double)tiles * stages * (share ? 64 + nm * rows : nm * (64 + rows));
                if (ks > 1) parts += (double)ks * nm * a.T;
            }
            for (int g = 1; g < a.n_grp; g++)                                   // longest first
                for (int r = g; r > 0 && len[r] > len[r - 1]; r--) {
                    const double l = len[r]; len[r] = len[r - 1]; len[r - 1] = l;
                    const long long c = count[r]; count[r] = count[r - 1]; count[r - 1] = c;
                }
            // dealing: slots that are free at the same time are kept together
            double at[2 * MLORA_MAX_PROJ + 2];
            long long n[2 * MLORA_MAX_PROJ + 2];
            int nb = 1;
            at[0] = 0.0; n[0] = slots;
            double end = 0.0;
            for (int g = 0; g < a.n_grp; g++) {
                long long c = count[g];
                const long long full = c / slots;                               // whole rounds over all slots
                if (full > 0) { for (int i = 0; i < nb; i++) at[i] += full * len[g]; c -= full * slots; }
                while (c > 0) {
                    int first = 0;
                    for (int i = 1; i < nb; i++) if (at[i] < at[first]) first = i;
                    const long long m = n[first] < c ? n[first] : c;
                    const double till = at[first] + len[g];
                    n[first] -= m;
                    c -= m;
                    int same = -1;
                    for (int i = 0; i < nb; i++) if (at[i] == till) same = i;
                    if (same >= 0) n[same] += m;
                    else if (n[first] == 0) { at[first] = till; n[first] = m; }
                    else { at[nb] = till; n[nb] = m; nb++; }
                    if (n[first] == 0 && first < nb) { nb--; at[first] = at[nb]; n[first] = n[nb]; }
                }
            }
            for (int i = 0; i < nb; i++) if (n[i] > 0 && at[i] > end) end = at[i];
            const double chain = 0.004 * end, all = 2.0 + 2e-5 * lines;
            const double us = (chain > all ? chain + 0.3 * all : all + 0.3 * chain) + 2e-4 * parts;
            if ((share == 0 && t == 0) || us < best) { best = us; best_k = k; a.share_x = share; }
        }
    }
    for (int p = 0; p < a.n_proj; p++) a.pr[p].ksplit = splits_of(a.pr[p].hin, hin_min, best_k, w);
    // longest workgroups first
    auto length = [&](int g) {
        const mlora::SgmvProj &pj = a.pr[a.grp_first[g]];
        return ((pj.hin + 63) / 64 + pj.ksplit - 1) / pj.ksplit * (64 + (a.share_x ? a.grp_n[g] : 1) * rows);
    };
    for (int g = 1; g < a.n_grp; g++)
        for (int r = g; r > 0 && length(r) > length(r - 1); r--) {
            const int f = a.grp_first[r], n = a.grp_n[r];
            a.grp_first[r] = a.grp_first[r - 1]; a.grp_n[r] = a.grp_n[r - 1];
            a.grp_first[r - 1] = f; a.grp_n[r - 1] = n;
        }
}

void carve(mlora::SgmvArgs &a, void *workspace, const SgmvWs &w)
{
    char *base = static_cast<char *>(workspace);
    int32_t *ip = reinterpret_cast<int32_t *>(base);
    a.tile_seg = ip; a.tile_tok0 = ip + w.max_tiles; a.tile_ntok = ip + 2 * (size_t)w.max_tiles;
    a.n_tiles = ip + 3 * (size_t)w.max_tiles;
    a.tok_cover = reinterpret_cast<int32_t *>(base + w.off_cover);
    a.tile_rec = reinterpret_cast<int32_t *>(base + w.off_rec);
    a.max_tiles = w.max_tiles;
    for (int p = 0; p < a.n_proj; p++) {
        char *pb = base + w.off_proj + w.per_proj * p;
        a.pr[p].v = reinterpret_cast<float *>(pb);
        a.pr[p].vhi = reinterpret_cast<uint16_t *>(pb + w.off_hi);
        a.pr[p].vlo = reinterpret_cast<uint16_t *>(pb + w.off_lo);
    }
}

// The shape of a call's launches, but for what sgmv_launch_shape adds.
void apply_shape(mlora::SgmvArgs &a, int max_rank, const SgmvWs &w, int phases)
{
    const int tiles = a.seg_uniform_len > 0 ? a.n_seg * ((a.seg_uniform_len + SG_TM - 1) / SG_TM) : (a.T + SG_TM / 2 * (a.n_seg - 1) + SG_TM - 1) / SG_TM;
    a.tiles = tiles;
    a.max_tiles = a.seg_uniform_len > 0 ? tiles : w.max_tiles;
    for (int p = 0; p < a.n_proj; p++) {
        int ncb = 0;
        const int cols = expand_block_cols(a.n_proj, w.max_tiles, a.pr[p].hout, &ncb);
        a.pr[p].cols = cols;
        a.pr[p].ncb = ncb;
    }
    shrink_shape(a, tiles, max_rank, w);
    // Whether x is read with the streaming hint: what a small call leaves in the last-level cache the next call on it finds there
    // (calls of one projection each on one x, the base GEMM behind its shrink), what a large call leaves there only
    // pushes other things out.  States of three batches in turn, ordinary / streaming, us.  Rank 64, by x and y of a call: the
    // reference's three calls (y written only) 92 MB 106 / 108, 109 MB 126 / 122, 134 MB 141 / 126; one paged projection,
    // 4096 to 4096, alone 109 MB 50 / 51, 170 MB 65 / 66, 230 MB 85 / 82, and three of them on one x 109 MB 149 / 154, 170 MB
    // 185 / 198, 230 MB 240 / 247 (11008 to 4096 alone 134 MB 62 / 60, 230 MB 78 / 74; 4096 to 11008 230 MB 89 / 91); q, k, v, o
    // 197 MB 79 / 86, 295 MB 117 / 115; seven projections 210 MB 109 / 105, 525 MB 221 / 210.  Base + LoRA in one pass, seven
    // projections: 700 tokens 354 / 355, 2000 tokens (263 MB) 733 / 740, 9216 tokens (1.2 GB) 3064 / 3066; rank 16, 2000 tokens 691 / 700.
    long long bytes = 0;
    for (int g = 0; g < a.n_grp; g++) bytes += (long long)a.T * a.pr[a.grp_first[g]].hin * 2;
    for (int p = 0; p < a.n_proj; p++) bytes += (long long)a.T * a.pr[p].hout * 2;
    a.stream_x = (phases & mlora::SGMV_APPLY) && bytes > (a.seg_uniform_len > 0 ? 100000000LL : 200000000LL);
}

}  // namespace

extern "C" {

int64_t mlora_sgmv_workspace_bytes(int T, int n_seg)
{
    if (T <= 0 || n_seg <= 0) return 256;
    return (int64_t)sgmv_layout(T, n_seg, 1).total;
}

int mlora_sgmv_expand_cols(int T, int n_seg, int n_proj, int hout)
{
    if (T <= 0 || n_seg <= 0 || n_proj < 1 || n_proj > MLORA_MAX_PROJ || hout <= 0) return 0;
    return expand_block_cols(n_proj, sgmv_layout(T, n_seg, n_proj).max_tiles, hout, nullptr);
}

int mlora_sgmv_splits(int T, int n_seg, int n_proj, int64_t workspace_bytes)
{
    if (T <= 0 || n_seg <= 0 || n_proj < 1 || n_proj > MLORA_MAX_PROJ || workspace_bytes < 0) return 0;
    const SgmvWs w = sgmv_layout(T, n_seg, n_proj, workspace_bytes);
    return (int64_t)w.total <= workspace_bytes ? w.ks_cap : 0;
}

int mlora_sgmv_shape(int n_proj, const void *const *x, const int32_t *hin, const int32_t *hout, int T, int n_seg, int seg_len,
                     int max_rank, int accumulate, int64_t workspace_bytes, int32_t *shape)
{
    if (n_proj < 1 || n_proj > MLORA_MAX_PROJ) return fail(MLORA_ERANGE, "n_proj must be in 1..%d (got %d)", MLORA_MAX_PROJ, n_proj);
    if (!x || !hin || !hout || !shape) return fail(MLORA_EINVAL, "NULL pointer");
    if (T <= 0 || n_seg <= 0 || seg_len < 0) return fail(MLORA_EINVAL, "T and n_seg must be positive (got %d, %d), seg_len >= 0", T, n_seg);
    if (seg_len > 0 && ((int64_t)n_seg * seg_len != T || n_proj != 1 || accumulate))
        return fail(MLORA_EINVAL, "equally long segments: T = n_seg * seg_len, one projection, y = delta");
    if (max_rank < 1 || max_rank > MLORA_MAX_RANK) return fail(MLORA_ERANGE, "max_rank must be in 1..%d (got %d)", MLORA_MAX_RANK, max_rank);
    mlora::SgmvArgs a;
    memset(&a, 0, sizeof(a));
    a.n_proj = n_proj; a.T = T; a.n_seg = n_seg; a.seg_uniform_len = seg_len; a.accumulate = accumulate ? 1 : 0;
    for (int p = 0; p < n_proj; p++) {
        const int rc = check_dims(hin[p], hout[p]);
        if (rc) return rc;
        a.pr[p].x = x[p]; a.pr[p].hin = hin[p]; a.pr[p].hout = hout[p];
    }
    const SgmvWs w = sgmv_layout(T, n_seg, n_proj, workspace_bytes < 0 ? 0 : workspace_bytes);
    if (workspace_bytes < (int64_t)w.total)
        return fail(MLORA_ENOSPACE, "workspace has %lld bytes, %lld needed", (long long)workspace_bytes, (long long)w.total);
    apply_shape(a, max_rank, w, mlora::SGMV_APPLY);
    mlora::sgmv_launch_shape(a, max_rank, mlora::SGMV_APPLY);
    shape[0] = a.share_x; shape[1] = a.stream_x; shape[2] = a.reduce; shape[3] = a.few;
    for (int p = 0; p < n_proj; p++) shape[4 + p] = a.pr[p].ksplit;
    return MLORA_OK;
}

int64_t mlora_sgmv_multi_workspace_bytes(int T, int n_seg, int n_proj)
{
    if (T <= 0 || n_seg <= 0 || n_proj < 1 || n_proj > MLORA_MAX_PROJ) return 256;
    return (int64_t)sgmv_layout(T, n_seg, n_proj).total;
}

static int sgmv_common(int n_proj, void *const *y, const void *const *x, const void *const *a_rows,
                       const void *const *b_rows, const int32_t *hin, const int32_t *hout, const int32_t *seg_start,
                       const int32_t *seg_len, const int32_t *seg_adapter, int n_seg, const int32_t *page_tbl,
                       const int32_t *rank, const float *scaling, int T, int n_adapters,
                       int max_pages, int page_rows, int64_t n_pages, int max_rank, int dtype, int accumulate,
                       void *workspace, int64_t workspace_bytes, int phases, void *stream, int tile_aligned = 0)
{
    if (dtype != MLORA_F16 && dtype != MLORA_BF16) return fail(MLORA_EDTYPE, "dtype must be MLORA_F16 or MLORA_BF16 (got %d)", dtype);
    if (T < 0 || n_seg < 0) return fail(MLORA_EINVAL, "T and n_seg must be >= 0 (got %d, %d)", T, n_seg);
    if (n_proj < 1 || n_proj > MLORA_MAX_PROJ) return fail(MLORA_ERANGE, "n_proj must be in 1..%d (got %d)", MLORA_MAX_PROJ, n_proj);
    if (T == 0 || n_seg == 0) return MLORA_OK;
    if (!seg_start || !seg_len || !seg_adapter) return fail(MLORA_EINVAL, "NULL device pointer");
    mlora::SgmvArgs a;
    memset(&a, 0, sizeof(a));
    int rc = check_pool(a.pool, page_tbl, rank, scaling, n_adapters, max_pages, page_rows, n_pages, max_rank);
    if (rc) return rc;
    a.n_proj = n_proj;
    if (phases & mlora::SGMV_APPLY) {
        if (!y || !x || !a_rows || !b_rows || !hin || !hout) return fail(MLORA_EINVAL, "per-projection arrays must not be NULL");
        for (int p = 0; p < n_proj; p++) {
            if (!y[p] || !x[p] || !a_rows[p] || !b_rows[p]) return fail(MLORA_EINVAL, "projection %d: NULL device pointer", p);
            rc = check_dims(hin[p], hout[p]);
            if (rc) return rc;
            if (!aligned16(y[p]) || !aligned16(x[p]) || !aligned16(a_rows[p]) || !aligned16(b_rows[p]))
                return fail(MLORA_EALIGN, "projection %d: device pointers must be 16-byte aligned", p);
            a.pr[p].y = y[p]; a.pr[p].x = x[p]; a.pr[p].a_rows = a_rows[p]; a.pr[p].b_rows = b_rows[p];
            a.pr[p].hin = hin[p]; a.pr[p].hout = hout[p];
        }
    }
    const SgmvWs w = sgmv_layout(T, n_seg, n_proj, workspace_bytes < 0 ? 0 : workspace_bytes);
    if (!workspace || !aligned16(workspace)) return fail(MLORA_EALIGN, "workspace must be a 16-byte aligned device pointer");
    if (workspace_bytes < (int64_t)w.total)
        return fail(MLORA_ENOSPACE, "workspace has %lld bytes, %lld needed", (long long)workspace_bytes, (long long)w.total);
    a.seg_start = seg_start; a.seg_len = seg_len; a.seg_adapter = seg_adapter; a.n_seg = n_seg;
    a.T = T; a.accumulate = accumulate ? 1 : 0; a.b_transposed = 0; a.seg_uniform_len = 0; a.tile_aligned = tile_aligned;
    carve(a, workspace, w);
    if (phases & mlora::SGMV_APPLY) apply_shape(a, max_rank, w, phases);                 // the plan itself has no use for one
    rc = mlora::launch_sgmv(a, dtype, max_rank, phases, static_cast<hipStream_t>(stream));
    if (rc) return fail(MLORA_ELAUNCH, "sgmv launch failed: %s", hipGetErrorString((hipError_t)rc));
    return MLORA_OK;
}

int mlora_sgmv(void *y, const void *x, const void *a_rows, const void *b_rows, const int32_t *seg_start,
               const int32_t *seg_len, const int32_t *seg_adapter, int n_seg, const int32_t *page_tbl,
               const int32_t *rank, const float *scaling, int T, int hin, int hout,
               int n_adapters, int max_pages, int page_rows, int64_t n_pages, int max_rank,
               int dtype, int accumulate, void *workspace, int64_t workspace_bytes, void *stream)
{
    void *ys[1] = {y};
    const void *xs[1] = {x}, *as[1] = {a_rows}, *bs[1] = {b_rows};
    const int32_t hi[1] = {hin}, ho[1] = {hout};
    return sgmv_common(1, ys, xs, as, bs, hi, ho, seg_start, seg_len, seg_adapter, n_seg, page_tbl, rank, scaling, T,
                       n_adapters, max_pages, page_rows, n_pages, max_rank, dtype, accumulate, workspace,
                       workspace_bytes, mlora::SGMV_PLAN | mlora::SGMV_APPLY, stream);
}

int mlora_sgmv_plan(const int32_t *seg_start, const int32_t *seg_len, const int32_t *seg_adapter, int n_seg,
                    const int32_t *page_tbl, const int32_t *rank, const float *scaling, int T, int n_adapters,
                    int max_pages, int page_rows, int64_t n_pages, int max_rank, void *workspace,
                    int64_t workspace_bytes, void *stream)
{
    return sgmv_common(1, nullptr, nullptr, nullptr, nullptr, nullptr, nullptr, seg_start, seg_len, seg_adapter, n_seg,
                       page_tbl, rank, scaling, T, n_adapters, max_pages, page_rows, n_pages, max_rank, MLORA_F16, 0,
                       workspace, workspace_bytes, mlora::SGMV_PLAN, stream);
}

int mlora_sgmv_plan_aligned(const int32_t *seg_start, const int32_t *seg_len, const int32_t *seg_adapter, int n_seg,
                            const int32_t *page_tbl, const int32_t *rank, const float *scaling, int T, int n_adapters,
                            int max_pages, int page_rows, int64_t n_pages, int max_rank, void *workspace,
                            int64_t workspace_bytes, void *stream)
{
    return sgmv_common(1, nullptr, nullptr, nullptr, nullptr, nullptr, nullptr, seg_start, seg_len, seg_adapter, n_seg,
                       page_tbl, rank, scaling, T, n_adapters, max_pages, page_rows, n_pages, max_rank, MLORA_F16, 0,
                       workspace, workspace_bytes, mlora::SGMV_PLAN, stream, 1);
}

int mlora_sgmv_planned(void *y, const void *x, const void *a_rows, const void *b_rows, const int32_t *seg_start,
                       const int32_t *seg_len, const int32_t *seg_adapter, int n_seg, const int32_t *page_tbl,
                       const int32_t *rank, const float *scaling, int T, int hin, int hout,
                       int n_adapters, int max_pages, int page_rows, int64_t n_pages, int max_rank,
                       int dtype, int accumulate, void *workspace, int64_t workspace_bytes, void *stream)
{
    void *ys[1] = {y};
    const void *xs[1] = {x}, *as[1] = {a_rows}, *bs[1] = {b_rows};
    const int32_t hi[1] = {hin}, ho[1] = {hout};
    return sgmv_common(1, ys, xs, as, bs, hi, ho, seg_start, seg_len, seg_adapter, n_seg, page_tbl, rank, scaling, T,
                       n_adapters, max_pages, page_rows, n_pages, max_rank, dtype, accumulate, workspace,
                       workspace_bytes, mlora::SGMV_APPLY, stream);
}

int mlora_sgmv_multi_planned(int n_proj, void *const *y, const void *const *x, const void *const *a_rows,
                             const void *const *b_rows, const int32_t *hin, const int32_t *hout,
                             const int32_t *seg_start, const int32_t *seg_len, const int32_t *seg_adapter, int n_seg,
                             const int32_t *page_tbl, const int32_t *rank, const float *scaling, int T,
                             int n_adapters, int max_pages, int page_rows, int64_t n_pages, int max_rank,
                             int dtype, int accumulate, void *workspace, int64_t workspace_bytes, void *stream)
{
    return sgmv_common(n_proj, y, x, a_rows, b_rows, hin, hout, seg_start, seg_len, seg_adapter, n_seg, page_tbl, rank,
                       scaling, T, n_adapters, max_pages, page_rows, n_pages, max_rank, dtype, accumulate, workspace,
                       workspace_bytes, mlora::SGMV_APPLY, stream);
}

int64_t mlora_gemm_lora_partial_bytes(int n_proj, const int32_t *hin, const int32_t *hout, int T)
{
    if (n_proj < 1 || n_proj > MLORA_MAX_PROJ || !hin || !hout || T <= 0) return 0;
    mlora::GemmLoraArgs g;
    mlora::GemmShape sh;
    memset(&g, 0, sizeof(g));
    g.n_proj = n_proj; g.T = T;
    for (int p = 0; p < n_proj; p++) {
        if (hin[p] <= 0 || hout[p] <= 0) return 0;
        g.pr[p].hin = hin[p]; g.pr[p].hout = hout[p];
    }
    return mlora::gemm_lora_shape(g, true, &sh);
}

int mlora_gemm_lora_planned(int n_proj, void *const *y, const void *const *x, const void *const *w,
                            const void *const *a_rows, const void *const *b_rows, const int32_t *hin,
                            const int32_t *hout, const int32_t *seg_start, const int32_t *seg_len,
                            const int32_t *seg_adapter, int n_seg, const int32_t *page_tbl, const int32_t *rank,
                            const float *scaling, int T, int n_adapters, int max_pages, int page_rows,
                            int64_t n_pages, int max_rank, int dtype, void *workspace, int64_t workspace_bytes,
                            void *stream)
{
    return mlora_gemm_lora_split(n_proj, y, x, w, a_rows, b_rows, hin, hout, seg_start, seg_len, seg_adapter, n_seg, page_tbl,
                                 rank, scaling, T, n_adapters, max_pages, page_rows, n_pages, max_rank, dtype, workspace,
                                 workspace_bytes, nullptr, 0, stream);
}

int mlora_gemm_lora_split(int n_proj, void *const *y, const void *const *x, const void *const *w,
                          const void *const *a_rows, const void *const *b_rows, const int32_t *hin,
                          const int32_t *hout, const int32_t *seg_start, const int32_t *seg_len,
                          const int32_t *seg_adapter, int n_seg, const int32_t *page_tbl, const int32_t *rank,
                          const float *scaling, int T, int n_adapters, int max_pages, int page_rows,
                          int64_t n_pages, int max_rank, int dtype, void *workspace, int64_t workspace_bytes,
                          void *partials, int64_t partial_bytes, void *stream)
{
    if (dtype != MLORA_F16 && dtype != MLORA_BF16) return fail(MLORA_EDTYPE, "dtype must be MLORA_F16 or MLORA_BF16 (got %d)", dtype);
    if (T < 0 || n_seg < 0) return fail(MLORA_EINVAL, "T and n_seg must be >= 0 (got %d, %d)", T, n_seg);
    if (n_proj < 1 || n_proj > MLORA_MAX_PROJ) return fail(MLORA_ERANGE, "n_proj must be in 1..%d (got %d)", MLORA_MAX_PROJ, n_proj);
    if (T == 0) return MLORA_OK;
    if (!y || !x || !w || !hin || !hout) return fail(MLORA_EINVAL, "per-projection arrays must not be NULL");
    const bool lora = n_seg > 0;
    if (lora && (!a_rows || !b_rows || !seg_start || !seg_len || !seg_adapter)) return fail(MLORA_EINVAL, "NULL pointer for a call with segments");
    mlora::SgmvArgs a;
    memset(&a, 0, sizeof(a));
    mlora::GemmLoraArgs g;
    memset(&g, 0, sizeof(g));
    int rc;
    if (lora) {
        rc = check_pool(a.pool, page_tbl, rank, scaling, n_adapters, max_pages, page_rows, n_pages, max_rank);
        if (rc) return rc;
    }
    a.n_proj = n_proj;
    for (int p = 0; p < n_proj; p++) {
        if (!y[p] || !x[p] || !w[p] || (lora && (!a_rows[p] || !b_rows[p]))) return fail(MLORA_EINVAL, "projection %d: NULL device pointer", p);
        rc = check_dims(hin[p], hout[p]);
        if (rc) return rc;
        if (!aligned16(y[p]) || !aligned16(x[p]) || !aligned16(w[p]) || (lora && (!aligned16(a_rows[p]) || !aligned16(b_rows[p]))))
            return fail(MLORA_EALIGN, "projection %d: device pointers must be 16-byte aligned", p);
        // the kernel addresses a weight through one buffer descriptor with 32-bit offsets
        if ((int64_t)hin[p] * hout[p] * 2 >= (1LL << 32)) return fail(MLORA_ERANGE, "projection %d: base weight of 4 GiB or more", p);
        if ((int64_t)256 * hin[p] * 2 >= (1LL << 32)) return fail(MLORA_ERANGE, "projection %d: hin too large", p);
        a.pr[p].y = y[p]; a.pr[p].x = x[p]; a.pr[p].hin = hin[p]; a.pr[p].hout = hout[p];
        g.pr[p].y = y[p]; g.pr[p].x = x[p]; g.pr[p].w = w[p]; g.pr[p].hin = hin[p]; g.pr[p].hout = hout[p];
        if (lora) {
            a.pr[p].a_rows = a_rows[p]; a.pr[p].b_rows = b_rows[p]; g.pr[p].b_rows = b_rows[p];
            // the B rows slab is addressed through one descriptor as well
            if ((int64_t)a.pool.n_rows_b * hout[p] * 2 >= 0xfff00000LL) return fail(MLORA_ERANGE, "projection %d: B rows slab of 4 GiB or more", p);
        }
    }
    g.n_proj = n_proj; g.T = T; g.lora = lora ? 1 : 0;
    if (partials) {
        const int64_t need = mlora_gemm_lora_partial_bytes(n_proj, hin, hout, T);
        if (partial_bytes < need) return fail(MLORA_ENOSPACE, "partials hold %lld bytes, %lld needed", (long long)partial_bytes, (long long)need);
        if (!aligned16(partials)) return fail(MLORA_EALIGN, "partials must be 16-byte aligned");
        if (need > 0) { g.partials = static_cast<float *>(partials); g.partial_bytes = need; }
    }
    if (lora) {
        const SgmvWs ws = sgmv_layout(T, n_seg, n_proj, workspace_bytes < 0 ? 0 : workspace_bytes);
        if (!workspace || !aligned16(workspace)) return fail(MLORA_EALIGN, "workspace must be a 16-byte aligned device pointer");
        if (workspace_bytes < (int64_t)ws.total)
            return fail(MLORA_ENOSPACE, "workspace has %lld bytes, %lld needed", (long long)workspace_bytes, (long long)ws.total);
        a.seg_start = seg_start; a.seg_len = seg_len; a.seg_adapter = seg_adapter; a.n_seg = n_seg;
        a.T = T; a.accumulate = 0; a.b_transposed = 0; a.seg_uniform_len = 0;
        carve(a, workspace, ws);
        apply_shape(a, max_rank, ws, mlora::SGMV_SHRINK);
        rc = mlora::launch_sgmv(a, dtype, max_rank, mlora::SGMV_SHRINK, static_cast<hipStream_t>(stream));
        if (rc) return fail(MLORA_ELAUNCH, "shrink launch failed: %s", hipGetErrorString((hipError_t)rc));
        for (int p = 0; p < n_proj; p++) {
            g.pr[p].v = a.pr[p].v; g.pr[p].vhi = a.pr[p].vhi; g.pr[p].vlo = a.pr[p].vlo; g.pr[p].ksplit = a.pr[p].ksplit;
        }
        g.tile_rec = a.tile_rec; g.n_tiles = a.n_tiles; g.max_tiles = a.max_tiles; g.n_rows_b = a.pool.n_rows_b;
    }
    rc = mlora::launch_gemm_lora(g, dtype, lora ? max_rank : 16, static_cast<hipStream_t>(stream));
    if (rc) return fail(MLORA_ELAUNCH, "gemm launch failed: %s", hipGetErrorString((hipError_t)rc));
    return MLORA_OK;
}

int mlora_prefill_reflayout(void *y, const void *x, const void *A_T, const void *B_T, int B, int Lpad, int L,
                            int r, int hin, int hout, int layer_idx, int dtype, void *workspace,
                            int64_t workspace_bytes, void *stream)
{
    if (dtype != MLORA_F16 && dtype != MLORA_BF16) return fail(MLORA_EDTYPE, "dtype must be MLORA_F16 or MLORA_BF16 (got %d)", dtype);
    if (B < 0 || Lpad < 0) return fail(MLORA_EINVAL, "B and Lpad must be >= 0 (got %d, %d)", B, Lpad);
    if (B == 0 || Lpad == 0) return MLORA_OK;
    if ((int64_t)B * Lpad > 0x7fffffffLL) return fail(MLORA_ERANGE, "B * Lpad exceeds 2^31-1 tokens");
    if (!y || !x || !A_T || !B_T) return fail(MLORA_EINVAL, "NULL device pointer");
    if (L <= 0 || layer_idx < 0 || layer_idx >= L) return fail(MLORA_ERANGE, "layer_idx %d outside [0, %d)", layer_idx, L);
    if (r < 8 || r > MLORA_MAX_RANK || (r & 7)) return fail(MLORA_ERANGE, "prefill on the reference layout needs a rank that is a multiple of 8 in 8..%d (got %d)", MLORA_MAX_RANK, r);
    int rc = check_dims(hin, hout);
    if (rc) return rc;
    if (!aligned16(y) || !aligned16(x) || !aligned16(A_T) || !aligned16(B_T))
        return fail(MLORA_EALIGN, "device pointers must be 16-byte aligned");
    if ((int64_t)B * L * r > 0x7fffffffLL) return fail(MLORA_ERANGE, "pool has more than 2^31-1 rank rows");
    const int T = B * Lpad;
    const SgmvWs w = sgmv_layout(T, B, 1, workspace_bytes < 0 ? 0 : workspace_bytes);
    if (!workspace || !aligned16(workspace)) return fail(MLORA_EALIGN, "workspace must be a 16-byte aligned device pointer");
    if (workspace_bytes < (int64_t)w.total)
        return fail(MLORA_ENOSPACE, "workspace has %lld bytes, %lld needed", (long long)workspace_bytes, (long long)w.total);
    mlora::SgmvArgs a;
    memset(&a, 0, sizeof(a));
    mlora::PoolView &pv = a.pool;
    pv.n_adapters = B; pv.max_pages = 1; pv.page_shift = 0;
    pv.uniform_rank = r; pv.uniform_scale = 1.0f;
    pv.a_dense_stride = (long long)L * r;
    pv.n_rows_a = (long long)(B - 1) * L * r + r;
    pv.b_dense_stride = (long long)L * hout * r;
    pv.n_rows_b = 0;
    a.n_proj = 1;
    a.pr[0].y = y; a.pr[0].x = x;
    a.pr[0].a_rows = static_cast<const uint16_t *>(A_T) + (size_t)layer_idx * r * hin;
    a.pr[0].b_rows = static_cast<const uint16_t *>(B_T) + (size_t)layer_idx * hout * r;
    a.pr[0].hin = hin; a.pr[0].hout = hout;
    a.n_seg = B; a.T = T; a.accumulate = 0; a.b_transposed = 1; a.seg_uniform_len = Lpad;
    carve(a, workspace, w);
    apply_shape(a, r, w, mlora::SGMV_APPLY);
    rc = mlora::launch_sgmv(a, dtype, r, mlora::SGMV_PLAN | mlora::SGMV_APPLY, static_cast<hipStream_t>(stream));
    if (rc) return fail(MLORA_ELAUNCH, "prefill launch failed: %s", hipGetErrorString((hipError_t)rc));
    return MLORA_OK;
}

}  // extern "C"
