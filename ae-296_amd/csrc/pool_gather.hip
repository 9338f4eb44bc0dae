// Adapter-pool index/offset gather for gfx950.
//
// Groups the tokens of a batch by adapter (stable: ordered by adapter id, then by token id) and derives
// segments, the decode work list (chunks of at most `group` tokens of one adapter) and the work records.
// Three forms: counting with one LDS counter per adapter, for up to 512 tokens of fewer than 2048 adapters
// (gather_few_kernel) and for more of either (gather_count_kernel, pools of fewer than 8192 slots), and a bitonic sort
// of 32-bit keys (gather_kernel, larger pools, whose counters do not fit LDS).
// Further blocks write the per-token view: page base rows, rank and scaling of each token's
// adapter.  All outputs are integers or copied floats, so they are bit-exact by construction.
//
// Stands where the reference draws / selects its per-token index vector
// (lightllm/models/lora_gpu.py:120,124,143,155) and drops the real per-request ids
// (lightllm/server/router/model_infer/pre_process.py:50,100).
#include "mlora_args.hpp"
#include "mlora_dev.hpp"
#include <type_traits>

namespace mlora {

constexpr int GATHER_NT_MAX = 1024;
constexpr int GATHER_MAX_T = 8192;
constexpr int TOK_BITS = 13;                 // token id field of the sort key
constexpr int COUNT_MAX_N_SMALL = 2048;      // adapters (and one) the instances of the counting form hold counters for
constexpr int COUNT_MAX_N_LARGE = 8192;

// Adapter id of token i as the kernels see it: negative = none, >= n_adapters = out of range (counted, then none).
// An int64 id (the reference's index vector) outside [0, n_adapters) is "none" on either side.
__device__ __forceinline__ int gather_adapter(const GatherArgs &g, int i)
{
    if (g.tok_adapter) return g.tok_adapter[i];
    const long long a = g.tok_adapter64[i];
    return a < 0 ? -1 : (a >= g.n_adapters ? g.n_adapters : (int)a);
}
__device__ __forceinline__ int gather_rank(const GatherArgs &g, int a) { return g.rank ? g.rank[a] : g.uniform_rank; }
__device__ __forceinline__ float gather_scale(const GatherArgs &g, int a) { return g.scaling ? g.scaling[a] : g.uniform_scale; }
// Row (in a rows slab) of rank row j of adapter a, -1 if it does not exist.
__device__ __forceinline__ int gather_row(const GatherArgs &g, int a, int j)
{
    if (!g.page_tbl) {
        const long long row = (long long)a * g.dense_stride + j;
        return row < g.n_rows_dense ? (int)row : -1;
    }
    if (j / g.page_rows >= g.max_pages) return -1;
    const int pg = g.page_tbl[(long long)a * g.max_pages + j / g.page_rows];
    return (pg >= 0 && pg < g.n_pages) ? pg * g.page_rows + j % g.page_rows : -1;
}

// ---- per-token view: page base rows, rank and scaling of each token's adapter (block of NT threads)
__device__ __forceinline__ void per_token_view(const GatherArgs &g, int block, int nt)
{
    const long long idx = (long long)block * nt + threadIdx.x;
    const long long total = (long long)g.T * g.max_pages;
    if (idx >= total) return;
    const int t = (int)(idx / g.max_pages), pg = (int)(idx - (long long)t * g.max_pages);
    int a = gather_adapter(g, t);
    if (a >= g.n_adapters) a = -1;
    int r = 0;
    float s = 0.f;
    int off = -1;
    if (a >= 0) {
        r = g.rank[a];
        s = g.scaling[a];
        const int np = (r + g.page_rows - 1) / g.page_rows;
        if (pg < np) off = g.page_tbl[(long long)a * g.max_pages + pg] * g.page_rows;
    }
    if (g.out_row_off) g.out_row_off[idx] = off;
    if (pg == 0) {
        if (g.out_rank) g.out_rank[t] = r;
        if (g.out_scale) g.out_scale[t] = s;
    }
}

// Inclusive scan over the block's per-thread values; op = 0 sum, 1 max, 2 min.
template <int OP>
__device__ __forceinline__ int scan_op(int a, int b)
{
    if constexpr (OP == 0) return a + b;
    else if constexpr (OP == 1) return a > b ? a : b;
    else return a < b ? a : b;
}

template <int OP>
__device__ int block_scan_inclusive(int v, int identity, int *s_wave /* [16] */)
{
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        const int o = __shfl_up(v, d);
        if (lane >= d) v = scan_op<OP>(v, o);
    }
    __syncthreads();                 // s_wave may still be read by a previous scan
    if (lane == 63) s_wave[wave] = v;
    __syncthreads();
    int base = identity;
    for (int w = 0; w < wave; w++) base = scan_op<OP>(base, s_wave[w]);
    return scan_op<OP>(base, v);
}

// ------------------------------------------------------------------ counting form
// Lanes of the wavefront that hold the same key (among the lanes of `active`), for keys below 2^nbits.
__device__ __forceinline__ unsigned long long same_key(unsigned key, int nbits, unsigned long long active)
{
    unsigned long long m = active;
    for (int b = 0; b < nbits; b++) {
        const bool bit = (key >> b) & 1u;
        const unsigned long long set = __ballot(bit);
        m &= bit ? set : ~set;
    }
    return m;
}

__device__ __forceinline__ unsigned long long block_scan_inclusive64(unsigned long long v, unsigned long long *s_wave /* [16] */)
{
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        const unsigned long long o = __shfl_up(v, d);
        if (lane >= d) v += o;
    }
    __syncthreads();                 // s_wave may still be read by a previous scan
    if (lane == 63) s_wave[wave] = v;
    __syncthreads();
    unsigned long long base = 0;
    for (int w = 0; w < wave; w++) base += s_wave[w];
    return base + v;
}

// Groups up to MAXT tokens over fewer than MAXN adapters by counting: one LDS counter per adapter.
//
// What bounds it is a chain of dependent steps and the records it writes, not bytes.  The sorting form below walks
// log2(T)^2 / 2 barriers and writes all records (320 bytes each) from one compute unit; here every workgroup repeats
// the counting, which is a few steps, and writes its own share of the records, so no workgroup waits for another:
//   1. a wavefront takes 64 tokens and finds the lanes that name the same adapter with one ballot per key bit; the
//      wavefronts add their counts to the adapters' counters in turn (token order, which keeps the grouping stable);
//   2. one scan over the adapters gives every segment's start, index and first chunk;
//   3. every token drops itself at its place, every head of a chunk its chunk header, in LDS;
//   4. records are written from those headers.
// Block 0 also writes the grouped view (perm, segments, chunks, counters).  Measured (graph replay of launch after
// launch, sorting form -> this one): 16.4 -> 7.2 us for 256 tokens of 64 adapters, 30.3 -> 9.0 us for 512 of 1000 with mixed
// ranks (both served by gather_few_kernel now), 358 -> 29 us for 8192 of 1000.
// T <= 2048 keeps the order by falling rank inside each eighth of the records, beyond that plain chunk order (as
// the sorting form does).
template <int MAXT, int MAXN>
__global__ __launch_bounds__(1024) void gather_count_kernel(const GatherArgs g, const int n_rec_blocks)
{
    constexpr int NT = 1024;
    constexpr int EPT = MAXT / NT;
    constexpr bool RANKED = MAXT <= 2048;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    if ((int)blockIdx.x >= n_rec_blocks) { per_token_view(g, (int)blockIdx.x - n_rec_blocks, NT); return; }
    const bool first_block = blockIdx.x == 0;

    __shared__ int s_cnt[MAXN];                // tokens per adapter; [n_adapters] = tokens without one
    __shared__ uint32_t s_base[MAXN];          // first position | first chunk << 14
    __shared__ uint16_t s_perm[MAXT];
    __shared__ uint32_t s_chunk[MAXT];         // start | len << 13 | adapter << 17
    __shared__ uint8_t s_crank[MAXT];
    __shared__ float s_cscale[MAXT];
    __shared__ unsigned long long s_wave[16];
    __shared__ int s_bad;
    const int T = g.T, n = g.n_adapters;
    for (int i = tid; i <= n; i += NT) s_cnt[i] = 0;
    if (tid == 0) s_bad = 0;
    int key[EPT], idx[EPT], rk[EPT];
    float sc[EPT];
    // adapter (n = none), and what its record will need, of this thread's tokens e * NT + tid
#pragma unroll
    for (int e = 0; e < EPT; e++) {
        const int i = e * NT + tid;
        key[e] = n; rk[e] = 0; sc[e] = 0.f;
        if (e * NT < T) {
            bool bad = false;
            if (i < T) {
                const int a = gather_adapter(g, i);
                bad = a >= n;
                if (a >= 0 && !bad) key[e] = a;
            }
            const unsigned long long mb = __ballot(bad);
            if (e == 0) __syncthreads();       // the counters are cleared
            if (lane == 0 && mb && first_block) atomicAdd(&s_bad, __popcll(mb));
        }
    }
    if (g.work) {
#pragma unroll
        for (int e = 0; e < EPT; e++)
            if (key[e] < n) {                  // requested now, used after the counting
                const int r = gather_rank(g, key[e]);
                rk[e] = r < 0 ? 0 : (r > MAX_RANK ? MAX_RANK : r);
                sc[e] = gather_scale(g, key[e]);
            }
    }
    int nbits = 1;
    while ((n >> nbits) != 0) nbits++;
#pragma unroll
    for (int e = 0; e < EPT; e++) {
        idx[e] = 0;
        if (e * NT < T) {
            const bool act = e * NT + tid < T;
            const unsigned long long active = __ballot(act);
            const unsigned long long same = same_key((unsigned)key[e], nbits, active);
            const int in_wave = __popcll(same & ((1ull << lane) - 1ull));
            const int waves = (T - e * NT + 63) / 64 < NT / 64 ? (T - e * NT + 63) / 64 : NT / 64;
            int before = 0;
            for (int w = 0; w < waves; w++) {  // in token order
                if (wave == w && act && in_wave == 0) {
                    before = s_cnt[key[e]];
                    s_cnt[key[e]] = before + __popcll(same);
                }
                __syncthreads();
            }
            const int leader = act ? __builtin_ctzll(same) : lane;
            idx[e] = __shfl(before, leader) + in_wave;
        }
    }
    // start, segment index and first chunk of every adapter, in adapter order (tokens without one come last)
    const int gmask = g.group - 1, gshift = __builtin_ctz((unsigned)g.group);
    unsigned long long carry = 0;              // tokens | segments << 20 | chunks << 40
    for (int a0 = 0; a0 <= n; a0 += NT) {
        const int a = a0 + tid;
        const int c = a <= n ? s_cnt[a] : 0;
        const unsigned long long own = (unsigned long long)c | ((unsigned long long)(c > 0 && a < n) << 20) |
                                       ((unsigned long long)((c + gmask) >> gshift) << 40);
        const unsigned long long incl = carry + block_scan_inclusive64(own, s_wave);
        const unsigned long long excl = incl - own;
        const int start = (int)(excl & 0xfffffu), seg = (int)((excl >> 20) & 0xfffffu), ch = (int)(excl >> 40);
        if (a <= n) s_base[a] = (uint32_t)(start & 0x3fff) | ((uint32_t)(ch & 0x3fff) << 14);
        if (first_block && c > 0 && a < n) { g.seg_start[seg] = start; g.seg_len[seg] = c; g.seg_adapter[seg] = a; }
        __syncthreads();
        unsigned long long all = 0;
#pragma unroll
        for (int w = 0; w < NT / 64; w++) all += s_wave[w];
        carry += all;
    }
    const int n_chunks = (int)(carry >> 40);
#pragma unroll
    for (int e = 0; e < EPT; e++) {
        const int i = e * NT + tid;
        if (i < T) {
            const uint32_t b = s_base[key[e]];
            const int start = (int)(b & 0x3fffu), at = start + idx[e];
            s_perm[at] = (uint16_t)i;
            if ((idx[e] & gmask) == 0) {
                const int c = (int)(b >> 14) + (idx[e] >> gshift), left = s_cnt[key[e]] - idx[e];
                const int len = left < g.group ? left : g.group;
                s_chunk[c] = (uint32_t)at | ((uint32_t)len << TOK_BITS) | ((uint32_t)key[e] << (TOK_BITS + 4));
                s_crank[c] = (uint8_t)rk[e];
                s_cscale[c] = sc[e];
            }
        }
    }
    __syncthreads();
    const uint32_t tmask = (1u << TOK_BITS) - 1u;
    if (first_block) {
        for (int i = tid; i < T; i += NT) g.perm[i] = s_perm[i];
        for (int c = tid; c < n_chunks; c += NT) {
            const uint32_t h = s_chunk[c];
            const int a = (int)(h >> (TOK_BITS + 4));
            g.chunk_start[c] = (int)(h & tmask);
            g.chunk_len[c] = (int)((h >> TOK_BITS) & 15u);
            g.chunk_adapter[c] = a < n ? a : -1;
        }
        if (tid < 8)
            g.counters[tid] = tid == 0 ? (int)((carry >> 20) & 0xfffffu) : tid == 1 ? T - s_cnt[n] : tid == 2 ? n_chunks : tid == 3 ? s_bad : 0;
    }
    if (!g.work) return;

    // Launch order of the records: records b, b + 8, ... hold one eighth of the chunks, by falling rank inside it
    // when the batch mixes ranks (ties keep chunk order: the chunks of one adapter stay next to each other).
    const int per_xcd = (n_chunks + 7) >> 3;
    bool mixed = false;
    __shared__ uint16_t s_ord[RANKED ? MAXT : 1];
    __shared__ int s_at[RANKED ? 8 : 1][MAX_RANK + 1];
    if constexpr (RANKED) {
        int differs = 0;
        for (int c = tid; c < n_chunks; c += NT) differs |= s_crank[c] != s_crank[0];
        for (int i = tid; i < 8 * (MAX_RANK + 1); i += NT) (&s_at[0][0])[i] = 0;
        mixed = __syncthreads_or(differs) != 0;
        if (mixed) {
            // a counting sort per eighth, one wavefront each
            const int lo = wave * per_xcd, hi = lo + per_xcd < n_chunks ? lo + per_xcd : n_chunks;
            if (wave < 8)
                for (int c = lo + lane; c < hi; c += 64) atomicAdd(&s_at[wave][s_crank[c]], 1);
            __syncthreads();
            if (wave < 8) {
                const int cnt = s_at[wave][MAX_RANK - lane];           // lane l: rank 64 - l
                int incl = cnt;
#pragma unroll
                for (int d = 1; d < 64; d <<= 1) {
                    const int o = __shfl_up(incl, d);
                    if (lane >= d) incl += o;
                }
                s_at[wave][MAX_RANK - lane] = lo + incl - cnt;
                if (lane == 63) s_at[wave][0] = lo + incl;
            }
            __syncthreads();
            if (wave < 8)
                for (int c0 = lo; c0 < hi; c0 += 64) {
                    const int c = c0 + lane;
                    const bool act = c < hi;
                    const unsigned r = act ? s_crank[c] : 0u;
                    const unsigned long long same = same_key(r, 7, __ballot(act));
                    const int in_wave = __popcll(same & ((1ull << lane) - 1ull));
                    int at = 0;
                    if (act && in_wave == 0) { at = s_at[wave][r]; s_at[wave][r] = at + __popcll(same); }
                    // the next 64 chunks' leaders are other lanes of this wavefront: they read what was written here
                    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
                    __builtin_amdgcn_wave_barrier();
                    at = __shfl(at, act ? __builtin_ctzll(same) : lane) + in_wave;
                    if (act) s_ord[at] = (uint16_t)c;
                }
            __syncthreads();
        }
    }
    // 16 bytes per step: header quad, two token quads, a zero quad, then 16 quads of row indices.
    constexpr int QPR = WORK_WORDS / 4;
    int4 *out = reinterpret_cast<int4 *>(g.work);
    const int quads = g.work_cap * QPR;
    for (int q = (int)blockIdx.x * NT + tid; q < quads; q += n_rec_blocks * NT) {
        const int b = q / QPR, w4 = q - b * QPR;
        const int pos = (b & 7) * per_xcd + (b >> 3);
        int4 v = make_int4(0, w4 == 0 ? -1 : 0, 0, 0);
        if ((b >> 3) < per_xcd && pos < n_chunks) {
            const int c = mixed ? s_ord[RANKED ? pos : 0] : pos;
            const uint32_t h = s_chunk[c];
            const int start = (int)(h & tmask), len = (int)((h >> TOK_BITS) & 15u), r = s_crank[c];
            int a = (int)(h >> (TOK_BITS + 4));
            a = a < n ? a : -1;
            if (w4 == 0) v = make_int4(len, a, r, __builtin_bit_cast(int, s_cscale[c]));
            else if (w4 <= 2) {
                const int k0 = (w4 - 1) * 4;
                v.x = k0 + 0 < len ? (int)s_perm[start + k0 + 0] : -1;
                v.y = k0 + 1 < len ? (int)s_perm[start + k0 + 1] : -1;
                v.z = k0 + 2 < len ? (int)s_perm[start + k0 + 2] : -1;
                v.w = k0 + 3 < len ? (int)s_perm[start + k0 + 3] : -1;
            } else if (w4 >= WORK_ROWS_AT / 4) {
                const int j0 = (w4 - WORK_ROWS_AT / 4) * 4;
                int rr[4];
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    const int j = j0 + e;
                    rr[e] = (a >= 0 && j < r) ? gather_row(g, a, j) : -1;
                }
                v = make_int4(rr[0], rr[1], rr[2], rr[3]);
            }
        }
        out[q] = v;
    }
}

// The counting form of an ordinary decode batch: up to 512 tokens over fewer than 2048 adapters.
//
// What bounds it is the chain of steps between barriers, so it has fewer and shorter ones than the kernel above: a token's
// 64-token run (the lanes of one wavefront) adds its count to one byte of the adapter's eight, all runs at once, instead of in
// turn; the bytes below a run's own give its place and all eight the adapter's tokens (v_sad_u8 adds four).  The scan over
// the adapters moves between lanes by DPP and takes one barrier, the order by rank is one comparison with each other chunk of
// the same eighth, and four wavefronts have shorter barriers than sixteen (the records are written by four times as many
// workgroups).  Time stamps of the kernel above: of 5 to 7 us 1.8 were the scan, 0.6 to 1.0 the counting, 0.5 to 1.6 the order
// by rank and 1.2 the records.  Whole steps, that kernel -> this one: 32 tokens of 8 adapters and one projection 12.7 -> 11.2 us, a
// graph of 7 tokens of mixed ranks, four layers 62.0 -> 59.4, 256 tokens of 64 adapters, four layers 93.6 -> 91.8.
constexpr int FEW_NT = 256;
constexpr int FEW_MAX_T = 512;               // eight runs of 64
constexpr int FEW_MAX_N = 2048;              // adapters and one for "none"
__global__ __launch_bounds__(FEW_NT) void gather_few_kernel(const GatherArgs g, const int n_rec_blocks)
{
    constexpr int NT = FEW_NT, EPT = FEW_MAX_T / NT, NW = NT / 64;
    constexpr int PER_EIGHTH = FEW_MAX_T / 8;                          // chunks of an eighth at most
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    if ((int)blockIdx.x >= n_rec_blocks) { per_token_view(g, (int)blockIdx.x - n_rec_blocks, NT); return; }
    const bool first_block = blockIdx.x == 0;

    __shared__ __attribute__((aligned(8))) uint32_t s_cnt[FEW_MAX_N][2];        // byte w: tokens of run w; [n_adapters] = without one
    __shared__ uint32_t s_base[FEW_MAX_N];                                      // first position | first chunk << 14
    __shared__ uint16_t s_perm[FEW_MAX_T];
    __shared__ int4 s_chunk[FEW_MAX_T];                                         // start | len << 13, adapter (n = none), rank, scaling
    __shared__ int4 s_rec[FEW_MAX_T];                                           // the same in the order of the records
    __shared__ __attribute__((aligned(16))) uint16_t s_key[8][PER_EIGHTH];      // rank << 6 | 63 - place, of the chunks of an eighth
    __shared__ uint32_t s_tot[NW][2];
    __shared__ int s_bad;
    const int T = g.T, n = g.n_adapters;
    for (int i = tid; i <= n; i += NT) *reinterpret_cast<uint2 *>(s_cnt[i]) = make_uint2(0u, 0u);
    if (tid < 8 * PER_EIGHTH * 2 / 16) reinterpret_cast<int4 *>(s_key)[tid] = make_int4(0, 0, 0, 0);
    if (tid == 0) s_bad = 0;
    // adapter (n = none), and what its record will need, of this thread's tokens e * NT + tid
    int key[EPT], rk[EPT], pg[EPT];
    float sc[EPT];
    bool bad[EPT];
#pragma unroll
    for (int e = 0; e < EPT; e++) {
        const int i = e * NT + tid;
        key[e] = n; rk[e] = 0; sc[e] = 0.f; pg[e] = 0; bad[e] = false;
        if (i < T) {
            const int a = gather_adapter(g, i);
            bad[e] = a >= n;
            if (a >= 0 && !bad[e]) key[e] = a;
        }
    }
    if (g.work) {
#pragma unroll
        for (int e = 0; e < EPT; e++)
            if (key[e] < n) {                  // requested now, used after the counting; the page table's line for the records
                const int r = gather_rank(g, key[e]);
                rk[e] = r < 0 ? 0 : (r > MAX_RANK ? MAX_RANK : r);
                sc[e] = gather_scale(g, key[e]);
                if (g.page_tbl) pg[e] = g.page_tbl[(long long)key[e] * g.max_pages];
            }
    }
    int nbits = 1;
    while ((n >> nbits) != 0) nbits++;
    __syncthreads();
    int in_wave[EPT];
#pragma unroll
    for (int e = 0; e < EPT; e++) {
        in_wave[e] = 0;
        if (e * NT < T) {
            const bool act = e * NT + tid < T;
            const unsigned long long same = same_key((unsigned)key[e], nbits, __ballot(act));
            in_wave[e] = __popcll(same & ((1ull << lane) - 1ull));
            const int w = e * NW + wave;
            if (act && in_wave[e] == 0) atomicAdd(&s_cnt[key[e]][w >> 2], (uint32_t)__popcll(same) << (8 * (w & 3)));
            if (first_block) {
                const unsigned long long mb = __ballot(bad[e]);
                if (lane == 0 && mb) atomicAdd(&s_bad, __popcll(mb));
            }
        }
    }
    __syncthreads();
    // start, segment index and first chunk of every adapter, in adapter order (tokens without one come last)
    const int gmask = g.group - 1, gshift = __builtin_ctz((unsigned)g.group);
    const int per = (n + NT) / NT, a0 = tid * per;                     // adapters a0 .. a0 + per of 0 .. n
    auto tokens_of = [&](int a) {
        const uint2 v = *reinterpret_cast<const uint2 *>(s_cnt[a]);
        return __builtin_amdgcn_sad_u8(v.x, 0u, __builtin_amdgcn_sad_u8(v.y, 0u, 0u));
    };
    uint32_t own_ts = 0, own_ch = 0;                                   // tokens | segments << 16, chunks
    for (int q = 0; q < per; q++) {
        const int a = a0 + q;
        const uint32_t c = a <= n ? tokens_of(a) : 0u;
        own_ts += c | (uint32_t)(c > 0 && a < n) << 16;
        own_ch += (c + gmask) >> gshift;
    }
    const uint32_t in_ts = wave_scan(own_ts), in_ch = wave_scan(own_ch);
    if (lane == 63) { s_tot[wave][0] = in_ts; s_tot[wave][1] = in_ch; }
    __syncthreads();
    uint32_t ts = in_ts - own_ts, ch = in_ch - own_ch, all_ts = 0, all_ch = 0;
#pragma unroll
    for (int w = 0; w < NW; w++) {
        const uint32_t t = s_tot[w][0], c = s_tot[w][1];
        ts += w < wave ? t : 0u; ch += w < wave ? c : 0u;
        all_ts += t; all_ch += c;
    }
    for (int q = 0; q < per; q++) {
        const int a = a0 + q;
        if (a > n) break;
        const uint32_t c = tokens_of(a), start = ts & 0xffffu, seg = ts >> 16;
        s_base[a] = start | ch << 14;
        if (first_block && c > 0 && a < n) { g.seg_start[seg] = (int)start; g.seg_len[seg] = (int)c; g.seg_adapter[seg] = a; }
        ts += c | (uint32_t)(c > 0 && a < n) << 16;
        ch += (c + gmask) >> gshift;
    }
    const int n_chunks = (int)all_ch, per_xcd = (n_chunks + 7) >> 3;
    __syncthreads();
    // Records b, b + 8, ... hold one eighth of the chunks, by falling rank inside it (ties keep chunk order: the chunks of one
    // adapter stay next to each other).  Where all ranks are equal that is the order of the chunks.
    const bool by_rank = g.rank != nullptr;
#pragma unroll
    for (int e = 0; e < EPT; e++) {
        const int i = e * NT + tid;
        if (i < T) {
            const uint32_t b = s_base[key[e]];
            const uint2 v = *reinterpret_cast<const uint2 *>(s_cnt[key[e]]);
            const int w = e * NW + wave;
            const uint32_t below = (1u << (8 * (w & 3))) - 1u;
            const int idx = (int)__builtin_amdgcn_sad_u8(v.x & (w < 4 ? below : ~0u), 0u,
                                                         __builtin_amdgcn_sad_u8(v.y & (w < 4 ? 0u : below), 0u, (uint32_t)in_wave[e]));
            const int total = (int)__builtin_amdgcn_sad_u8(v.x, 0u, __builtin_amdgcn_sad_u8(v.y, 0u, 0u));
            const int at = (int)(b & 0x3fffu) + idx;
            s_perm[at] = (uint16_t)i;
            if ((idx & gmask) == 0) {
                const int c = (int)(b >> 14) + (idx >> gshift), left = total - idx;
                int eighth = 0;
#pragma unroll
                for (int k = 1; k < 8; k++) eighth += c >= k * per_xcd;
                const int4 h = make_int4(at | (left < g.group ? left : g.group) << TOK_BITS, key[e], rk[e],
                                         __builtin_bit_cast(int, sc[e]));
                s_chunk[c] = h;
                if (by_rank) s_key[eighth][c - eighth * per_xcd] = (uint16_t)(rk[e] << 6 | (63 - (c - eighth * per_xcd)));
                else s_rec[c] = h;
            }
        }
        asm volatile("" :: "v"(pg[e]));        // the page table's line has arrived
    }
    __syncthreads();
    if (by_rank && g.work) {
        for (int c = tid; c < n_chunks; c += NT) {
            int eighth = 0;
#pragma unroll
            for (int k = 1; k < 8; k++) eighth += c >= k * per_xcd;
            const int first = eighth * per_xcd;
            const uint32_t own = s_key[eighth][c - first];
            int at = first;
            for (int j = 0; j < per_xcd; j += 8) {                      // keys past the chunks are 0: never greater
                const uint4 k8 = *reinterpret_cast<const uint4 *>(&s_key[eighth][j]);
                at += ((k8.x & 0xffffu) > own) + ((k8.x >> 16) > own) + ((k8.y & 0xffffu) > own) + ((k8.y >> 16) > own) +
                      ((k8.z & 0xffffu) > own) + ((k8.z >> 16) > own) + ((k8.w & 0xffffu) > own) + ((k8.w >> 16) > own);
            }
            s_rec[at] = s_chunk[c];
        }
        __syncthreads();
    }
    const int tmask = (1 << TOK_BITS) - 1;
    if (g.work) {
        // 16 bytes per step: header quad, two token quads, a zero quad, then 16 quads of row indices.
        constexpr int QPR = WORK_WORDS / 4;
        int4 *out = reinterpret_cast<int4 *>(g.work);
        const int quads = g.work_cap * QPR;
        for (int q = (int)blockIdx.x * NT + tid; q < quads; q += n_rec_blocks * NT) {
            const int b = q / QPR, w4 = q - b * QPR;
            const int pos = (b & 7) * per_xcd + (b >> 3);
            int4 v = make_int4(0, w4 == 0 ? -1 : 0, 0, 0);
            if ((b >> 3) < per_xcd && pos < n_chunks) {
                const int4 h = s_rec[pos];
                const int start = h.x & tmask, len = h.x >> TOK_BITS, a = h.y < n ? h.y : -1, r = h.z;
                if (w4 == 0) v = make_int4(len, a, r, h.w);
                else if (w4 <= 2) {
                    const int k0 = (w4 - 1) * 4;
                    v.x = k0 + 0 < len ? (int)s_perm[start + k0 + 0] : -1;
                    v.y = k0 + 1 < len ? (int)s_perm[start + k0 + 1] : -1;
                    v.z = k0 + 2 < len ? (int)s_perm[start + k0 + 2] : -1;
                    v.w = k0 + 3 < len ? (int)s_perm[start + k0 + 3] : -1;
                } else if (w4 >= WORK_ROWS_AT / 4) {
                    const int j0 = (w4 - WORK_ROWS_AT / 4) * 4;
                    int rr[4];
#pragma unroll
                    for (int e = 0; e < 4; e++) {
                        const int j = j0 + e;
                        rr[e] = (a >= 0 && j < r) ? gather_row(g, a, j) : -1;
                    }
                    v = make_int4(rr[0], rr[1], rr[2], rr[3]);
                }
            }
            out[q] = v;
        }
    }
    if (first_block) {
        for (int i = tid; i < T; i += NT) g.perm[i] = s_perm[i];
        for (int c = tid; c < n_chunks; c += NT) {
            const int4 h = s_chunk[c];
            g.chunk_start[c] = h.x & tmask;
            g.chunk_len[c] = h.x >> TOK_BITS;
            g.chunk_adapter[c] = h.y < n ? h.y : -1;
        }
        if (tid < 8)
            g.counters[tid] = tid == 0 ? (int)(all_ts >> 16) : tid == 1 ? T - (int)tokens_of(n)
                              : tid == 2 ? n_chunks : tid == 3 ? s_bad : 0;
    }
}

// One workgroup of GATHER_NT threads groups up to MAXT tokens (EPT sorted positions per thread in the
// scans).  The MAXT = 2048 instance also keeps the chunk headers in LDS, which makes writing the work
// records cheap; decode batches are normally that small.
template <int GATHER_NT, int MAXT>
__global__ __launch_bounds__(GATHER_NT) void gather_kernel(const GatherArgs g)
{
    constexpr int EPT = MAXT / GATHER_NT;
    const int tid = threadIdx.x;
    if (blockIdx.x > 0) { per_token_view(g, (int)blockIdx.x - 1, GATHER_NT); return; }
    if (!g.perm) return;

    // ---- grouped view (one workgroup)
    constexpr bool LDS_HDR = MAXT <= 2048;                 // chunk headers fit in LDS next to the keys
    __shared__ uint32_t s_key[MAXT];
    __shared__ int s_chdr[LDS_HDR ? MAXT : 1];             // start | len << 13 | rank << 17 per chunk
    __shared__ float s_cscale[LDS_HDR ? MAXT : 1];
    __shared__ int s_wave[16];
    __shared__ int s_cnt[2];
    const int T = g.T;
    int n2 = 2;
    while (n2 < T) n2 <<= 1;
    if (tid < 2) s_cnt[tid] = 0;
    __syncthreads();
    const uint32_t sentinel = (uint32_t)g.n_adapters;   // "no adapter" sorts after every real adapter
    for (int i = tid; i < n2; i += GATHER_NT) {
        uint32_t key = 0xffffffffu;
        bool valid = false, bad = false;
        if (i < T) {
            const int a = gather_adapter(g, i);
            bad = a >= g.n_adapters;
            valid = a >= 0 && !bad;
            key = ((valid ? (uint32_t)a : sentinel) << TOK_BITS) | (uint32_t)i;
        }
        s_key[i] = key;
        const unsigned long long mv = __ballot(valid), mb = __ballot(bad);
        if ((tid & 63) == 0) {
            if (mv) atomicAdd(&s_cnt[0], __popcll(mv));
            if (mb) atomicAdd(&s_cnt[1], __popcll(mb));
        }
    }
    __syncthreads();
    for (int k = 2; k <= n2; k <<= 1) {
        for (int j = k >> 1; j > 0; j >>= 1) {
            for (int i = tid; i < (n2 >> 1); i += GATHER_NT) {
                const int lo = 2 * i - (i & (j - 1));
                const int hi = lo + j;
                const uint32_t a = s_key[lo], b = s_key[hi];
                const bool up = (lo & k) == 0;
                if ((a > b) == up) { s_key[lo] = b; s_key[hi] = a; }
            }
            __syncthreads();
        }
    }
    const int n_valid = s_cnt[0];
    const int gmask = g.group - 1;

    // Each thread owns EPT consecutive sorted positions.
    int ad[EPT], head[EPT];
    const int base = tid * EPT;
#pragma unroll
    for (int e = 0; e < EPT; e++) {
        const int i = base + e;
        ad[e] = -1; head[e] = 0;
        if (i < T) {
            const uint32_t key = s_key[i];
            ad[e] = (int)(key >> TOK_BITS);
            g.perm[i] = (int)(key & ((1u << TOK_BITS) - 1u));
            head[e] = (i == 0) || ((int)(s_key[i - 1] >> TOK_BITS) != ad[e]);
        }
    }
    // segment start of every position: running max of head positions
    int run = 0, segstart[EPT];
#pragma unroll
    for (int e = 0; e < EPT; e++) { if (head[e]) run = base + e; segstart[e] = run; }
    {
        const int incl = block_scan_inclusive<1>(run, 0, s_wave);
        const int prev = __shfl_up(incl, 1);          // exclusive value for this thread
        __syncthreads();
        if ((tid & 63) == 63) s_wave[tid >> 6] = incl;
        __syncthreads();
        int excl = (tid & 63) ? prev : ((tid >> 6) ? s_wave[(tid >> 6) - 1] : 0);
        bool seen = false;
#pragma unroll
        for (int e = 0; e < EPT; e++) { seen = seen || head[e]; if (!seen) segstart[e] = excl; }
    }
    // segment end of every position: next head position after it (T if none): reverse running min
    int segend[EPT];
    {
        int nxt = T;
        int own_first = T;                       // first head position inside this thread's range
#pragma unroll
        for (int e = EPT - 1; e >= 0; e--) { segend[e] = nxt; if (head[e]) nxt = base + e; }
        own_first = nxt;
        // suffix min over threads = prefix min over reversed thread order
        const int rt = GATHER_NT - 1 - tid;
        __syncthreads();
        __shared__ int s_first[GATHER_NT];
        s_first[rt] = own_first;
        __syncthreads();
        const int mine = s_first[tid];            // value of thread (NT-1-tid)
        const int incl = block_scan_inclusive<2>(mine, T, s_wave);
        __syncthreads();
        s_first[tid] = incl;                      // min over reversed index <= tid
        __syncthreads();
        const int after = rt > 0 ? s_first[rt - 1] : T;   // min over threads with larger tid
#pragma unroll
        for (int e = 0; e < EPT; e++) if (segend[e] == T) segend[e] = after < T ? after : T;
    }
    // running counts of real segment heads and of chunk heads
    int nseg_local = 0, nch_local = 0, chead[EPT];
#pragma unroll
    for (int e = 0; e < EPT; e++) {
        const int i = base + e;
        chead[e] = (i < T) && (((i - segstart[e]) & gmask) == 0);
        nseg_local += (head[e] && ad[e] < g.n_adapters) ? 1 : 0;
        nch_local += chead[e];
    }
    const int seg_incl = block_scan_inclusive<0>(nseg_local, 0, s_wave);
    const int ch_incl = block_scan_inclusive<0>(nch_local, 0, s_wave);
    int seg_idx = seg_incl - nseg_local, ch_idx = ch_incl - nch_local;
#pragma unroll
    for (int e = 0; e < EPT; e++) {
        const int i = base + e;
        const bool real = ad[e] >= 0 && ad[e] < g.n_adapters;
        if (head[e] && real) {
            g.seg_start[seg_idx] = i;
            g.seg_len[seg_idx] = segend[e] - i;
            g.seg_adapter[seg_idx] = ad[e];
            seg_idx++;
        }
        if (chead[e]) {
            const int left = segend[e] - i;
            const int len = left < g.group ? left : g.group;
            g.chunk_start[ch_idx] = i;
            g.chunk_len[ch_idx] = len;
            g.chunk_adapter[ch_idx] = real ? ad[e] : -1;
            if constexpr (LDS_HDR) {
                if (g.work) {
                    int rk = 0;
                    float sc = 0.f;
                    if (real) { rk = gather_rank(g, ad[e]); rk = rk < 0 ? 0 : (rk > MAX_RANK ? MAX_RANK : rk); sc = gather_scale(g, ad[e]); }
                    s_chdr[ch_idx] = i | (len << TOK_BITS) | (rk << (TOK_BITS + 4));
                    s_cscale[ch_idx] = sc;
                }
            }
            ch_idx++;
        }
    }
    // ---- decode work records, in launch order: the records in use first; records b, b + 8, ... hold consecutive
    // chunks (the one-launch decode form, whose workgroup b of a projection reads record b, runs them on one XCD:
    // workgroups are dealt to the 8 XCDs round-robin; the two-launch form takes the records in order).  Batches
    // beyond 2048 tokens (chunk headers not in LDS) keep plain chunk order inside each range.
    if (g.work) {
        __shared__ int s_nchunks;
        if (tid == GATHER_NT - 1) s_nchunks = ch_incl;
        __syncthreads();                         // chunk_* arrays written above are visible to the whole block
        const int n_chunks = s_nchunks;
        const int per_xcd = (n_chunks + 7) >> 3;
        if constexpr (LDS_HDR) {
            // Within each of the eight ranges of chunks the records are written in order of falling rank
            // (ties keep chunk order, so the chunks of one adapter stay next to each other): the workgroups of
            // the wide items are then dispatched first and the narrow ones fill in behind them.  A counting sort:
            // chunks per (XCD, rank), then one thread per (XCD, rank) places its chunks.
            __shared__ int s_ord[MAXT];
            __shared__ int s_cntx[8][MAX_RANK + 1];
            int differs = 0;                     // a pool of one rank keeps chunk order and skips the sort
            for (int c = tid; c < n_chunks; c += GATHER_NT) differs |= (s_chdr[c] >> (TOK_BITS + 4)) != (s_chdr[0] >> (TOK_BITS + 4));
            for (int i = tid; i < 8 * (MAX_RANK + 1); i += GATHER_NT) (&s_cntx[0][0])[i] = 0;
            const bool mixed = __syncthreads_or(differs) != 0;
            if (mixed)
                for (int c = tid; c < n_chunks; c += GATHER_NT) atomicAdd(&s_cntx[c / per_xcd][s_chdr[c] >> (TOK_BITS + 4)], 1);
            __syncthreads();
            if (mixed && tid < 8 * (MAX_RANK + 1)) {
                const int xcd = tid / (MAX_RANK + 1), rk = tid - xcd * (MAX_RANK + 1);
                if (s_cntx[xcd][rk] > 0) {
                    int at = xcd * per_xcd;
                    for (int r2 = rk + 1; r2 <= MAX_RANK; r2++) at += s_cntx[xcd][r2];
                    const int lo = xcd * per_xcd, hi = lo + per_xcd < n_chunks ? lo + per_xcd : n_chunks;
                    for (int c = lo; c < hi; c++)
                        if ((s_chdr[c] >> (TOK_BITS + 4)) == rk) s_ord[at++] = c;
                }
            }
            __syncthreads();
            // 16 bytes per step: header quad, two token quads, a zero quad, then 16 quads of row indices.
            constexpr int QPR = WORK_WORDS / 4;
            int4 *out = reinterpret_cast<int4 *>(g.work);
            const int quads = g.work_cap * QPR;
            const uint32_t tmask = (1u << TOK_BITS) - 1u;
#pragma unroll 4
            for (int q = tid; q < quads; q += GATHER_NT) {
                const int b = q / QPR, w4 = q - b * QPR;
                const int pos = (b & 7) * per_xcd + (b >> 3);
                int4 v = make_int4(0, w4 == 0 ? -1 : 0, 0, 0);
                if ((b >> 3) < per_xcd && pos < n_chunks) {
                    const int c = mixed ? s_ord[pos] : pos;
                    const int hdr = s_chdr[c];
                    const int start = hdr & (int)tmask, len = (hdr >> TOK_BITS) & 15, rk = hdr >> (TOK_BITS + 4);
                    int a = (int)(s_key[start] >> TOK_BITS);
                    a = a < g.n_adapters ? a : -1;
                    if (w4 == 0) v = make_int4(len, a, rk, __builtin_bit_cast(int, s_cscale[c]));
                    else if (w4 <= 2) {
                        const int k0 = (w4 - 1) * 4;
                        v.x = k0 + 0 < len ? (int)(s_key[start + k0 + 0] & tmask) : -1;
                        v.y = k0 + 1 < len ? (int)(s_key[start + k0 + 1] & tmask) : -1;
                        v.z = k0 + 2 < len ? (int)(s_key[start + k0 + 2] & tmask) : -1;
                        v.w = k0 + 3 < len ? (int)(s_key[start + k0 + 3] & tmask) : -1;
                    } else if (w4 >= WORK_ROWS_AT / 4) {
                        const int j0 = (w4 - WORK_ROWS_AT / 4) * 4;
                        int rr[4];
#pragma unroll
                        for (int e = 0; e < 4; e++) {
                            const int j = j0 + e;
                            rr[e] = (a >= 0 && j < rk) ? gather_row(g, a, j) : -1;
                        }
                        v = make_int4(rr[0], rr[1], rr[2], rr[3]);
                    }
                }
                out[q] = v;
            }
        } else {
        const long long words = (long long)g.work_cap * WORK_WORDS;
        for (long long idx = tid; idx < words; idx += GATHER_NT) {
            const int b = (int)(idx / WORK_WORDS), w = (int)(idx - (long long)b * WORK_WORDS);
            const int c = (b & 7) * per_xcd + (b >> 3);
            int val = w == 1 ? -1 : 0;
            if ((b >> 3) < per_xcd && c < n_chunks) {
                const int start = g.chunk_start[c], len = g.chunk_len[c], a = g.chunk_adapter[c];
                int rk = 0;
                if (a >= 0) { rk = gather_rank(g, a); rk = rk < 0 ? 0 : (rk > MAX_RANK ? MAX_RANK : rk); }
                if (w == 0) val = len;
                else if (w == 1) val = a;
                else if (w == 2) val = rk;
                else if (w == 3) val = a >= 0 ? __builtin_bit_cast(int, gather_scale(g, a)) : 0;
                else if (w < 12) val = (w - 4) < len ? (int)(s_key[start + (w - 4)] & ((1u << TOK_BITS) - 1u)) : -1;
                else if (w < WORK_ROWS_AT) val = 0;
                else {
                    const int j = w - WORK_ROWS_AT;
                    val = (a >= 0 && j < rk) ? gather_row(g, a, j) : -1;
                }
            }
            g.work[idx] = val;
        }
        }
    }
    if (tid == GATHER_NT - 1) {
        g.counters[0] = seg_incl;
        g.counters[1] = n_valid;
        g.counters[2] = ch_incl;
        g.counters[3] = s_cnt[1];
        g.counters[4] = 0; g.counters[5] = 0; g.counters[6] = 0; g.counters[7] = 0;
    }
}

int launch_gather(const GatherArgs &a, hipStream_t s)
{
    const long long per_tok = (a.out_row_off || a.out_rank || a.out_scale) ? (long long)a.T * a.max_pages : 0;
    // Beyond 512 tokens the runs no longer fit the eight bytes of a counter, beyond 2047 adapters a thread scans more than eight.
    if (a.perm && a.T <= FEW_MAX_T && a.n_adapters < FEW_MAX_N) {
        // a workgroup per 256 16-byte pieces of the records, up to a quarter of the chip
        const long long quads = a.work ? (long long)a.work_cap * (WORK_WORDS / 4) : 0;
        int nb = (int)((quads + FEW_NT - 1) / FEW_NT);
        nb = nb < 1 ? 1 : (nb > 64 ? 64 : nb);
        hipLaunchKernelGGL(gather_few_kernel, dim3((unsigned)(nb + (per_tok + FEW_NT - 1) / FEW_NT)), dim3(FEW_NT), 0, s, a, nb);
        return (int)hipGetLastError();
    }
    const unsigned view = (unsigned)((per_tok + GATHER_NT_MAX - 1) / GATHER_NT_MAX);
    // The counting form needs one LDS counter per adapter (and one for "none"); larger pools sort.  512 tokens of 6000
    // adapters, where the counters are cleared and scanned in six rounds: 17 us counting, 31 sorting.
    if (a.perm && a.n_adapters < COUNT_MAX_N_LARGE) {
        // a workgroup per 1024 16-byte pieces of the records, up to a quarter of the chip
        const long long quads = a.work ? (long long)a.work_cap * (WORK_WORDS / 4) : 0;
        int nb = (int)((quads + GATHER_NT_MAX - 1) / GATHER_NT_MAX);
        nb = nb < 1 ? 1 : (nb > 64 ? 64 : nb);
        if (a.T <= 2048 && a.n_adapters < COUNT_MAX_N_SMALL)
            hipLaunchKernelGGL((gather_count_kernel<2048, COUNT_MAX_N_SMALL>), dim3((unsigned)nb + view), dim3(GATHER_NT_MAX), 0, s, a, nb);
        else if (a.T <= 2048)
            hipLaunchKernelGGL((gather_count_kernel<2048, COUNT_MAX_N_LARGE>), dim3((unsigned)nb + view), dim3(GATHER_NT_MAX), 0, s, a, nb);
        else
            hipLaunchKernelGGL((gather_count_kernel<GATHER_MAX_T, COUNT_MAX_N_LARGE>), dim3((unsigned)nb + view), dim3(GATHER_NT_MAX), 0, s, a, nb);
        return (int)hipGetLastError();
    }
    const unsigned grid = 1u + view;
    if (a.T <= 2048) hipLaunchKernelGGL((gather_kernel<GATHER_NT_MAX, 2048>), dim3(grid), dim3(GATHER_NT_MAX), 0, s, a);
    else hipLaunchKernelGGL((gather_kernel<GATHER_NT_MAX, GATHER_MAX_T>), dim3(grid), dim3(GATHER_NT_MAX), 0, s, a);
    return (int)hipGetLastError();
}

}  // namespace mlora
