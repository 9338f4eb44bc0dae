// SGMV prefill kernels for gfx950: tokens are packed per segment (one adapter per segment)
//     y[t] (+)= s_a * (x[t] . A_a) . B_a
// computed on v_mfma_f32_16x16x32_{f16,bf16} tiles in two to four launches on one stream (the first can be shared by all projections
// and layers of a batch):
//   plan   : cuts every segment into tiles of at most 64 tokens (work list in the workspace);
//   shrink : V[split][t][0..R) = x[t, Kslice] . A_a[:, Kslice]^T   (split-K, fp32 partials), or with one
//            split the result itself as a hi + lo pair of 16-bit values, so that the intermediate keeps
//            fp32 accuracy through the second MFMA;
//   reduce : sums the K splits into such pairs and, where y = delta, zeroes the rows outside every segment (up to
//            rank 32, and in launches of few tiles, the expand sums the splits itself; where y accumulates the
//            launch is then left out, as it is with one split);
//   expand : y[t, cols] (+)= s_a * (Vhi + Vlo) . B_a[:, cols].
// Both MFMA operands of the shrink pass through a ring of LDS stages that global memory fills directly.
// The expand parks the B tile in LDS (rank must be the
// in-lane K dimension, the pool stores rank rows), reads it back with the transposing LDS read,
// and passes the output through a wavefront-private LDS tile so that every y access is a
// 16-byte, row-contiguous one (8-byte accesses straight from the accumulators were measured slower).
//
// Replaces torch.bmm(torch.bmm(x, A), B) at lightllm/models/lora_gpu.py:127-128,145-146,157-158.
#include "mlora_args.hpp"
#include "mlora_dev.hpp"
#include <type_traits>

namespace mlora {

// Activations and outputs pass through once: streaming (nontemporal) accesses.  A and B rows are
// re-read by every token tile of a segment and stay ordinary cached loads (measured: streaming them
// too loses what the other three gain).


constexpr int TM = 64;       // tokens per tile
constexpr int TN = 128;      // output columns per expand step
constexpr int SG_NT = 256;   // 4 wavefronts, 16 tokens each
constexpr int VSTRIDE = MAX_RANK;
typedef short short4_t __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) short4_t lds_short4;

__device__ __forceinline__ void seg_of(const SgmvArgs &p, int s, int &start, int &len, int &adapter)
{
    start = p.seg_start[s]; len = p.seg_len[s]; adapter = p.seg_adapter[s];
    if (start < 0 || len < 0 || start > p.T) { start = 0; len = 0; }
    if (len > p.T - start) len = p.T - start;
}

// v / d by the inverse of d that the host has put into the arguments: the product is the quotient or one less, for every v and d.
// A division by an argument is some forty instructions through the float reciprocal, and a workgroup had up to five of them
// between its id and its first load: four layers of one prompt of 64 tokens, rank 64, q/k/v, 46.8 -> 46.3 us, the reference's
// call of 16 x 512 tokens, three projections, 118.7 -> 117.6.
static unsigned inverse_of(int d) { return 0xffffffffu / (unsigned)(d > 0 ? d : 1); }
__device__ __forceinline__ int divided(int v, int d, unsigned inv)
{
    const unsigned q = __umulhi((unsigned)v, inv);
    return (int)(q + ((unsigned)v - q * (unsigned)d >= (unsigned)d ? 1u : 0u));
}

// Workgroup id -> (tile, second index) for the shrink (second = K split) and the expand (second = column
// block).  Workgroups are dealt to the 8 XCDs round-robin by id and every XCD has its own L2; tiles are
// ordered by segment, so runs of XRUN consecutive tiles mostly share one adapter.  All workgroups of a
// run that have the same second index read the same slice of A (or B): they are given ids with the same
// residue mod 8, i.e. one XCD, and the residue rotates with the second index so the XCDs stay balanced.
constexpr int XRUN = 8;
// So does `rot`, from one group of projections to the next: tiles are rarely a multiple of 64, and the XCDs with a run more
// than the others would be the same ones every time.
__device__ __forceinline__ void xcd_remap(int w, int n_second, unsigned inv, int rot, int &tile, int &second)
{
    const int r = w & 7, slot = w >> 3;
    const int i = slot % XRUN;
    const int j = divided(slot / XRUN, n_second, inv);
    second = slot / XRUN - j * n_second;
    const int run = ((r - second - rot) & 7) + 8 * j;
    tile = run * XRUN + i;
}
__host__ __device__ inline long long xcd_grid(int max_tiles, int n_second)
{
    const long long runs = (max_tiles + XRUN - 1) / XRUN;
    return 8LL * ((runs + 7) / 8) * n_second * XRUN;
}

// Launches of few tiles number the second index fastest, without padding: the runs above would leave most ids of a
// batch of a tile or two without work (512 workgroups for 8 at one tile and eight splits), and what runs together
// is everything anyway.
__host__ __device__ inline bool few_tiles(int max_tiles) { return max_tiles < XRUN * 8; }
__device__ __forceinline__ void place(int w, int n_second, unsigned inv, int max_tiles, int rot, int &tile, int &second)
{
    if (few_tiles(max_tiles)) { tile = divided(w, n_second, inv); second = w - tile * n_second; }
    else xcd_remap(w, n_second, inv, rot, tile, second);
}
__host__ __device__ inline long long place_grid(int max_tiles, int n_second)
{
    return few_tiles(max_tiles) ? (long long)max_tiles * n_second : xcd_grid(max_tiles, n_second);
}

// Shrink launches of a few tiles have them as the grid's second dimension, one tile's groups behind each other: nothing to divide
// by. With more, the longest groups of all tiles go first.  Whole calls of 1 to 24 prompts of 1 to 1000 tokens, two layers of
// Llama-7B, one, three, four and seven projections, ranks 16 to 64, second dimension against longest first: up to 16 tiles (of
// the host's bound) 1 % faster on average (0.92 to 1.06 times, one tile 47.9 -> 47.0 us), 17 to 32 0.99 to 1.005 times on average
// and up to 1.08, 33 to 56 1.01 to 1.02 times at rank 64 and up to 1.11 (seven projections, 4 x 400 tokens 211 -> 234 us).
__host__ __device__ inline bool tile_rows(int max_tiles) { return max_tiles <= 2 * XRUN; }

// Expand launches use a second order where it fits: tile-major, the column blocks of a tile next to each other, so
// that the eight workgroups running side by side (one per XCD) update one contiguous stretch of 64 y rows instead
// of the same 1 KiB column block of 64 different tiles (DRAM pages stay open: a bare read-modify-write walk over
// config 5's y is 11 % faster this way).  The blocks of a tile are numbered up to the next multiple of eight and
// rotated by the tile's run of eight, so a column block of a run stays on one XCD (its B tile is fetched into one
// L2) and the unused numbers fall on every XCD in turn.  Only where few numbers stay unused (at most an eighth):
// with 10 blocks in 16 numbers two XCDs get twice the work of the others for eight tiles at a time, the dispatcher
// hands out workgroups in order, and the launch was 9 % slower than in the order above (config 4 with 512-column
// blocks; the host therefore picks the block width so that the count fits, see tile_major in mlora_args.hpp).
__host__ __device__ inline long long expand_grid(int max_tiles, int ncb)
{
    return tile_major(ncb) && !few_tiles(max_tiles) ? (long long)max_tiles * ((ncb + 7) & ~7) : place_grid(max_tiles, ncb);
}

// Group (or projection) of workgroup w, and its number there, from the groups' first numbers behind them.  All ends are read at once:
// looking them up in turn is a chain of scalar loads in front of everything else.
struct GroupId { int group, rest; };
__device__ __forceinline__ GroupId group_at(const unsigned (&end)[MAX_PROJ], unsigned w)
{
    GroupId r = {0, (int)w};
#pragma unroll
    for (int i = 0; i + 1 < MAX_PROJ; i++)
        if (w >= end[i]) { r.group = i + 1; r.rest = (int)(w - end[i]); }
    return r;
}

// What a workgroup needs to know about its tile: from the plan's record, or, for equally long segments on a dense
// pool (the reference's prefill, segment s = adapter s), computed, which needs no plan at all.
// (A compile-time choice: a branch on it around the row lookups made the shrink wait for each of its twelve in turn,
// which doubled the whole call.)
template <bool UNIFORM>
struct Tile {
    int ntok, adapter, rank, tok0;
    float scale;
    const int32_t *__restrict__ rows;   // record: row of every rank row, -1 = absent
    long long row0;                     // uniform: row of rank row 0
    __device__ __forceinline__ int row(int j, long long n_rows) const
    {
        if constexpr (!UNIFORM) return rows[j];
        const long long r = row0 + j;
        return j < rank && r < n_rows ? (int)r : -1;
    }
};

template <bool UNIFORM>
__device__ __forceinline__ Tile<UNIFORM> tile_of(const SgmvArgs &p, int tile)
{
    Tile<UNIFORM> t;
    if constexpr (UNIFORM) {
        const int len = p.seg_uniform_len;
        const int seg = divided(tile, p.seg_tiles, p.seg_tiles_inv), i = tile - seg * p.seg_tiles;
        t.ntok = len - i * TM < TM ? len - i * TM : TM;
        t.adapter = seg;
        t.rank = p.pool.uniform_rank < MAX_RANK ? p.pool.uniform_rank : MAX_RANK;
        t.scale = p.pool.uniform_scale;
        t.tok0 = seg * len + i * TM;
        t.rows = nullptr;
        t.row0 = (long long)seg * p.pool.a_dense_stride;
    } else {
        const int32_t *__restrict__ rec = p.tile_rec + (size_t)tile * TILE_WORDS;
        t.ntok = rec[0]; t.adapter = rec[1]; t.rank = rec[2]; t.scale = __builtin_bit_cast(float, rec[3]); t.tok0 = rec[4];
        t.rows = rec + TILE_ROWS_AT;
        t.row0 = 0;
    }
    return t;
}

// ------------------------------------------------------------------ plan
// (segments on a paged pool; equally long ones on a dense pool need none, see Tile)
//
// A workgroup writes the list entries and records of PLAN_TILES tiles and the cover flags of PLAN_TOKENS tokens; every one
// counts the tiles of all segments itself, a few steps, so that none waits for another.  What bounds it is the start of a
// launch and the chain segments -> adapter -> rank, scaling, page table -> record, most of it on lines that no cache holds any
// more; the counting runs beside it.  One prompt of 64 tokens 4.0 -> 3.7 us, sixteen of 9216 12.0 -> 11.2 (before, the rank and the
// page table were asked for behind the headers).
constexpr int PLAN_NT = 256;
constexpr int PLAN_TILES = 16;
constexpr int PLAN_TOKENS = 4 * PLAN_NT;
__global__ __launch_bounds__(PLAN_NT) void sgmv_plan_kernel(const SgmvArgs p)
{
    __shared__ int s_start[PLAN_NT], s_end[PLAN_NT], s_first[PLAN_NT];  // segments of a batch: tokens, and the first tile
    __shared__ int s_wave[PLAN_NT / 64];
    __shared__ int s_hdr[PLAN_TILES][6];                                // tokens, adapter, rank, scaling, first token, segment
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int t0 = (int)blockIdx.x * PLAN_TILES, k0 = (int)blockIdx.x * PLAN_TOKENS;
    const PoolView &pv = p.pool;
    if (tid < PLAN_TILES) s_hdr[tid][0] = 0;
    int carry = 0;
    bool cover[PLAN_TOKENS / PLAN_NT] = {};
    for (int s0 = 0; s0 < p.n_seg; s0 += PLAN_NT) {
        const int s = s0 + tid;
        int start = 0, len = 0, adapter = -1;
        if (s < p.n_seg) seg_of(p, s, start, len, adapter);
        // what the records of the segment's tiles will need, requested with nothing else to wait for; the page table's line
        // for the rows
        const bool real = adapter >= 0 && adapter < pv.n_adapters;
        int rk = 0, sc = 0, pg = 0;
        if (real) {
            rk = pv.rank[adapter];
            sc = __builtin_bit_cast(int, pv.scaling[adapter]);
            pg = pv.a_tbl[(long long)adapter * pv.max_pages];
        }
        // tiles of a segment: every TM tokens from its start, or (aligned) the pieces between multiples of TM
        const int lead = p.tile_aligned ? start % TM : 0;
        const int nt = len > 0 ? (lead + len + TM - 1) / TM : 0;
        const int v = (int)wave_scan((uint32_t)nt);
        if (s0 > 0) __syncthreads();                   // the previous batch of segments has been looked at
        if (lane == 63) s_wave[wave] = v;
        __syncthreads();
        int first = carry + v - nt, all = carry;
#pragma unroll
        for (int w = 0; w < PLAN_NT / 64; w++) { first += w < wave ? s_wave[w] : 0; all += s_wave[w]; }
        s_start[tid] = start; s_end[tid] = start + len; s_first[tid] = first;
        // this workgroup's tiles of the segment
        const int i0 = t0 - first > 0 ? t0 - first : 0, i1 = t0 + PLAN_TILES - first < nt ? t0 + PLAN_TILES - first : nt;
        const int cap = pv.max_pages << pv.page_shift < MAX_RANK ? pv.max_pages << pv.page_shift : MAX_RANK;
        rk = rk < 0 ? 0 : (rk > cap ? cap : rk);
        for (int i = i0; i < i1; i++) {
            if (first + i >= p.max_tiles) break;
            const int b = i == 0 ? start : start - lead + i * TM;
            const int e = start - lead + (i + 1) * TM < start + len ? start - lead + (i + 1) * TM : start + len;
            int *h = s_hdr[first + i - t0];
            h[0] = e - b; h[1] = real ? adapter : -1; h[2] = rk; h[3] = sc; h[4] = b; h[5] = s;
        }
        asm volatile("" :: "v"(pg));                   // the page table's line has arrived
        __syncthreads();
        // Which tokens belong to a tile at all: y = delta mode must define the rows of the others (zeros).
        const int ns = p.n_seg - s0 < PLAN_NT ? p.n_seg - s0 : PLAN_NT;
        if (k0 < p.T)
            for (int q = 0; q < ns; q++) {
                const int b = s_start[q], e = s_end[q], at = p.tile_aligned ? b - b % TM : b;
#pragma unroll
                for (int u = 0; u < PLAN_TOKENS / PLAN_NT; u++) {
                    const int t = k0 + u * PLAN_NT + tid;
                    cover[u] = cover[u] || (t >= b && t < e && s_first[q] + (t - at) / TM < p.max_tiles);
                }
            }
        carry = all;
    }
    // Per-tile records: everything a shrink / expand workgroup needs, so that it starts from one load.  Records beyond the
    // tiles in use are marked empty, so that a workgroup starts from its record alone and does not wait for the count first.
    constexpr int WPT = PLAN_TILES * TILE_WORDS / PLAN_NT;
    static_assert(WPT * PLAN_NT == PLAN_TILES * TILE_WORDS, "every thread writes as many words");
    int page[WPT];
#pragma unroll
    for (int u = 0; u < WPT; u++) {                    // all table lookups leave together: each is made, at entry 0 where there is none
        const int idx = u * PLAN_NT + tid, lt = idx / TILE_WORDS, j = idx - lt * TILE_WORDS - TILE_ROWS_AT;
        const int *h = s_hdr[lt];
        const bool has = j >= 0 && h[0] > 0 && h[1] >= 0 && j < h[2];
        page[u] = pv.a_tbl[has ? (long long)h[1] * pv.max_pages + (j >> pv.page_shift) : 0];
        page[u] = has ? page[u] : -1;
    }
#pragma unroll
    for (int u = 0; u < WPT; u++) {
        const int idx = u * PLAN_NT + tid, lt = idx / TILE_WORDS, w = idx - lt * TILE_WORDS, j = w - TILE_ROWS_AT;
        const int *h = s_hdr[lt];
        int val = h[0] <= 0 ? -w : (w < 6 ? h[w] : 0); // an empty record: no tokens, no adapter
        if (j >= 0) {
            const long long row = ((long long)page[u] << pv.page_shift) + (j & ((1 << pv.page_shift) - 1));
            val = page[u] < 0 || row >= pv.n_rows_a ? -1 : (int)row;
        }
        if (t0 + lt < p.max_tiles && (h[0] > 0 || w < 2)) p.tile_rec[(size_t)(t0 + lt) * TILE_WORDS + w] = val;
    }
    if (tid < PLAN_TILES && s_hdr[tid][0] > 0) {
        p.tile_seg[t0 + tid] = s_hdr[tid][5]; p.tile_tok0[t0 + tid] = s_hdr[tid][4]; p.tile_ntok[t0 + tid] = s_hdr[tid][0];
    }
    if (blockIdx.x == 0 && tid == 0) p.n_tiles[0] = carry < p.max_tiles ? carry : p.max_tiles;
#pragma unroll
    for (int u = 0; u < PLAN_TOKENS / PLAN_NT; u++) {
        const int t = k0 + u * PLAN_NT + tid;
        if (t < p.T) p.tok_cover[t] = cover[u] ? 1 : 0;
    }
}

// ------------------------------------------------------------------ shrink
template <int DT>
__device__ __forceinline__ float4_t mfma16(const uint4 &a, const uint4 &b, float4_t c)
{
    if constexpr (DT == DT_F16)
        return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(half8_t, a), __builtin_bit_cast(half8_t, b), c, 0, 0, 0);
    else
        return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf168_t, a), __builtin_bit_cast(bf168_t, b), c, 0, 0, 0);
}

constexpr int SG_NM = 3;                    // projections of one x that a shrink workgroup serves at most (a larger group is cut by the host)
constexpr int SH_CH = 8;                    // 16-byte chunks of a stage row: one 128-byte line
constexpr int SH_ROWB = SH_CH * 16;
// How a workgroup is built: SHARE: four wavefronts, up to SG_NM projections; otherwise KG groups of four, one projection,
// each group with its own half of the K range and its own ring.
template <bool SHARE> constexpr int SH_KG = SHARE ? 1 : 2;
// LDS of a group's ring: four stages of the most rows (more of fewer rows)
template <int RMAX, bool SHARE> constexpr int sh_group_bytes() { return 4 * (TM + (SHARE ? SG_NM : 1) * RMAX) * SH_ROWB; }

// hi + lo 16-bit halves of N values (hi = round16(v), lo = round16(v - hi)), packed in pairs.
template <int DT, int N>
__device__ __forceinline__ void split_hi_lo(const float (&v)[N], uint32_t (&hi)[N / 2], uint32_t (&lo)[N / 2])
{
    uint32_t h[N], l[N];
#pragma unroll
    for (int e = 0; e < N; e++) {
        h[e] = cvt16<DT>(v[e]);
        const float back = lo_f32<DT>(h[e]);
        l[e] = cvt16<DT>(v[e] - back);
    }
#pragma unroll
    for (int e = 0; e < N / 2; e++) { hi[e] = h[2 * e] | (h[2 * e + 1] << 16); lo[e] = l[2 * e] | (l[2 * e + 1] << 16); }
}

// One workgroup: 64 tokens x RMAX ranks over one K range, for one projection, or (SHARE) for up to SG_NM projections that
// read the same x.  A stage is 64 columns of the x rows and of every projection's A rows; global memory fills a ring of stages
// in LDS directly (global_load_lds, whole lines), so that three or more stages are in flight while one is multiplied.  A
// wavefront takes half of the tokens and half of the ranks (at rank 16 a quarter of the tokens).
// What bounds it is the lines a compute unit can have on their way (some hundred, whatever the kernel asks for) times how
// long they take: 11 million lines of 735 cycles for sixteen ragged prompts of Llama-13B, 9216 tokens, of which the A rows of
// every tile are more than half.  Staging a stage in registers, with the next one requested only when it had been parked in LDS,
// and every wavefront reading all of A back (4 KiB of LDS reads a column for three projections; now 2): that batch 189 us
// (now 176), 16 x 512 tokens of one projection at rank 64 19.5 us (15.3), one prompt of 64 tokens, three projections, 7.0 us
// (6.0).  Reading operands straight from global memory, 64 bytes a row and load, took 328 and 21 us.
template <int DT, int RMAX, bool UNIFORM, bool SHARE>
__global__ __launch_bounds__(SG_NT *SH_KG<SHARE>) void sgmv_shrink_kernel(const SgmvArgs p)
{
    constexpr int KG = SH_KG<SHARE>;
    constexpr int NB = RMAX / 16;                               // rank blocks of 16
    constexpr int WT = NB >= 2 ? 2 : 4;                         // wavefronts along the tokens, the others along the ranks
    constexpr int TBW = TM / 16 / WT, NBW = NB * WT / 4;        // 16 x 16 blocks per wavefront and projection
    constexpr int GROUP_BYTES = sh_group_bytes<RMAX, SHARE>();
    constexpr int CH = SH_CH, ROWB = SH_ROWB;
    constexpr int RPL = 1024 / ROWB;                            // rows one load of a wavefront fills
    __shared__ __attribute__((aligned(16))) unsigned char s_ring[KG * GROUP_BYTES];
    // SHARE: a workgroup per (tile, split) of a group; otherwise one per projection, the projections of a group being the
    // fastest index, so that they run side by side on one XCD and find x in its L2.
    const GroupId at = group_at(p.grp_end, blockIdx.x);
    const int grp = at.group, w = at.rest, ng = SHARE ? 1 : p.grp_n[grp];
    auto by_group = [&](int v) {                                // v / ng
        return ng == 1 ? v : (ng == 2 ? v >> 1 : (int)(__umulhi((unsigned)v, 0xaaaaaaabu) >> 1));
    };
    int tile = (int)blockIdx.y, split, p0 = p.grp_first[grp];
    if (tile_rows(p.max_tiles)) {
        split = by_group(w);
        p0 += w - split * ng;
    } else if (few_tiles(p.max_tiles)) {
        const int q = by_group(w);
        p0 += w - q * ng;
        place(q, p.pr[p0].ksplit, p.pr[p0].ksplit_inv, p.max_tiles, grp * 3, tile, split);
    } else {
        const int q = by_group(w >> 3);
        p0 += (w >> 3) - q * ng;
        place(q * 8 + (w & 7), p.pr[p0].ksplit, p.pr[p0].ksplit_inv, p.max_tiles, grp * 3, tile, split);
        if (tile >= p.max_tiles) return;                        // records beyond the tiles in use hold no tokens
    }
    const int nm = SHARE ? p.grp_n[grp] : 1;
    const SgmvProj &pj = p.pr[p0];
    const Tile<UNIFORM> tl = tile_of<UNIFORM>(p, tile);
    // Row of rank row `lane`, requested with the record's header; the loads get theirs from the other lanes, and the end of the
    // kernel asks the mask which of them exist.
    int mine = tl.row((int)threadIdx.x & 63, p.pool.n_rows_a);
    const int ntok = tl.ntok, tok0 = tl.tok0;
    if (tl.adapter < 0 || ntok <= 0 || tok0 < 0 || tok0 + ntok > p.T) return;
    asm volatile("" : "+v"(mine));                              // loaded by all lanes
    const unsigned long long have = __ballot(mine >= 0);

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave_all = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int kg = wave_all >> 2, wave = wave_all & 3;
    const int m = lane & 15, g = lane >> 4;
    const int hin = pj.hin;
    const int ncc = hin >> 3;                                   // 16-byte chunks per row
    const int whole = ncc / CH, nstage = (ncc + CH - 1) / CH;   // full stages, stages
    const int per = pj.kper;
    const int st0 = split * per < whole ? split * per : whole, st1 = st0 + per < whole ? st0 + per : whole;
    const int half = (st1 - st0 + KG - 1) / KG;                 // every group walks this many steps, the last one may have fewer stages
    const int g0 = st0 + kg * half < st1 ? st0 + kg * half : st1;
    const int n = st1 - g0 < half ? st1 - g0 : half;
    // whether this range ends with a stage of fewer columns
    const bool tail = whole < nstage && split * per <= whole && whole < split * per + per;
    unsigned char *ring = s_ring + kg * GROUP_BYTES;
    typedef __attribute__((address_space(3))) unsigned char lds_byte;
    const unsigned ring_at = (unsigned)(__UINTPTR_TYPE__)(lds_byte *)ring;

    auto run = [&](auto nm_tag) {
        constexpr int NM = decltype(nm_tag)::value;
        constexpr int ROWS = TM + NM * RMAX, STAGE = ROWS * ROWB;
        constexpr int D = GROUP_BYTES / STAGE < 8 ? GROUP_BYTES / STAGE : 8;            // stages of the ring
        constexpr int XU = TM / RPL / 4, AI = NM * RMAX / RPL, AU = (AI + 3) / 4, NL = XU + AU;
        static_assert(D >= 3 && NL * (D - 2) < 64, "the ring and the load counter");
        // One load of a wavefront fills RPL rows of a stage (1 KiB): lane i row i / CH, slot i % CH.  Chunk c of row r is stored
        // in slot c ^ key(r): 16 operand rows of one chunk column then lie in 16 different bank groups.
        // Rows past the tile's tokens repeat the last one, absent rank rows read row 0; neither is stored.
        auto key = [](int r) { return (r >> 1) & 7; };
        const char *src[NL];
        unsigned dst[NL];
#pragma unroll
        for (int u = 0; u < NL; u++) {
            const int i = u < XU ? wave + 4 * u : (wave + 4 * (u - XU) < AI ? wave + 4 * (u - XU) : wave + 4 * (u - XU) - AI);
            const int r = i * RPL + lane / CH;                  // row of the x tile, or of the A tiles one after the other
            const int c = lane % CH ^ key(r);
            const char *row;
            if (u < XU) {
                row = reinterpret_cast<const char *>(static_cast<const uint16_t *>(pj.x) + (size_t)(tok0 + (r < ntok ? r : ntok - 1)) * hin);
            } else {
                const int mm = i * RPL / RMAX, at = __shfl(mine, r - mm * RMAX);
                row = reinterpret_cast<const char *>(static_cast<const uint16_t *>(p.pr[p0 + mm].a_rows) + (size_t)(at >= 0 ? at : 0) * hin);
            }
            src[u] = row + (size_t)g0 * ROWB + c * 16;
            dst[u] = (unsigned)(i * RPL + (u < XU ? 0 : TM)) * ROWB;
        }
        auto request = [&](int slot) {                          // the next stage, into a slot of the ring
            const unsigned at = ring_at + (unsigned)slot * STAGE;
            if (p.stream_x) {
#pragma unroll
                for (int u = 0; u < XU; u++)
                    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off nt" :: "s"(at + dst[u]), "v"(src[u]) : "memory");
            } else {
#pragma unroll
                for (int u = 0; u < XU; u++)
                    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off" :: "s"(at + dst[u]), "v"(src[u]) : "memory");
            }
#pragma unroll
            for (int u = XU; u < NL; u++)
                asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off" :: "s"(at + dst[u]), "v"(src[u]) : "memory");
#pragma unroll
            for (int u = 0; u < NL; u++) src[u] += ROWB;
        };
        // operands: x rows of this wavefront's token blocks, A rows of its rank blocks; slice k of 32 columns is chunk 4 k + g
        const int tw = WT == 4 ? wave : wave >> 1, rw = WT == 4 ? 0 : wave & 1;
        unsigned xat[CH / 4], aat[CH / 4];
#pragma unroll
        for (int k = 0; k < CH / 4; k++) {
            const unsigned slot = (unsigned)(((4 * k + g) ^ key(m)) * 16);
            xat[k] = (unsigned)(tw * TBW * 16 + m) * ROWB + slot;
            aat[k] = (unsigned)(TM + rw * NBW * 16 + m) * ROWB + slot;
        }
        float4_t acc[NM][TBW][NBW];
#pragma unroll
        for (int mm = 0; mm < NM; mm++)
#pragma unroll
            for (int tb = 0; tb < TBW; tb++)
#pragma unroll
                for (int nb = 0; nb < NBW; nb++) acc[mm][tb][nb] = float4_t{0.f, 0.f, 0.f, 0.f};
        auto multiply = [&](const unsigned char *st) {
#pragma unroll
            for (int k = 0; k < CH / 4; k++) {
                uint4 xf[TBW];
#pragma unroll
                for (int tb = 0; tb < TBW; tb++) xf[tb] = *reinterpret_cast<const uint4 *>(st + xat[k] + tb * 16 * ROWB);
#pragma unroll
                for (int mm = 0; mm < NM; mm++)
#pragma unroll
                    for (int nb = 0; nb < NBW; nb++) {
                        const uint4 af = *reinterpret_cast<const uint4 *>(st + aat[k] + (mm * RMAX + nb * 16) * ROWB);
#pragma unroll
                        for (int tb = 0; tb < TBW; tb++) acc[mm][tb][nb] = mfma16<DT>(af, xf[tb], acc[mm][tb][nb]);
                    }
            }
        };
        // At the barrier of step i every wavefront's loads of stage i have landed and all reads of stage i - 1 are done,
        // so its slot takes stage i + D - 1.
#pragma unroll
        for (int d = 0; d < D - 1; d++)
            if (d < n) request(d);
        int slot = 0;
#pragma unroll 1
        for (int i = 0; i < half; i++) {
            if (i + D - 2 < n) __builtin_amdgcn_s_waitcnt(0x0f70 | ((NL * (D - 2)) & 15) | (((NL * (D - 2)) >> 4) << 14));
            else __builtin_amdgcn_s_waitcnt(0x0f70);
            __syncthreads();
            if (i + D - 1 < n) request(slot == 0 ? D - 1 : slot - 1);
            if (i < n) multiply(ring + slot * STAGE);
            slot = slot + 1 < D ? slot + 1 : 0;
        }
        if (tail) {
            // chunks past the rows' end are zeros on both sides; the last group of wavefronts does this stage
            __syncthreads();
            if (kg == KG - 1) {
#pragma unroll
                for (int u = 0; u < NL; u++) {
                    const int r = (int)(dst[u] / ROWB) + lane / CH, c = lane % CH ^ key(r);
                    const bool ok = whole * CH + c < ncc;
                    const uint4 v = ok ? ldg16(src[u] + (size_t)(whole - g0 - n) * ROWB) : zero16();
                    *reinterpret_cast<uint4 *>(ring + dst[u] + lane * 16) = v;
                }
            }
            __syncthreads();
            if (kg == KG - 1) multiply(ring);
        }
        if constexpr (KG > 1) {                                 // the groups' sums, in K order
            __syncthreads();
            float4_t *s_acc = reinterpret_cast<float4_t *>(s_ring);
#pragma unroll
            for (int q = 1; q < KG; q++)
                if (kg == q)
#pragma unroll
                    for (int tb = 0; tb < TBW; tb++)
#pragma unroll
                        for (int nb = 0; nb < NBW; nb++) s_acc[(((q - 1) * 4 + wave) * TBW * NBW + tb * NBW + nb) * 64 + lane] = acc[0][tb][nb];
            __syncthreads();
            if (kg > 0) return;
#pragma unroll
            for (int q = 1; q < KG; q++)
#pragma unroll
                for (int tb = 0; tb < TBW; tb++)
#pragma unroll
                    for (int nb = 0; nb < NBW; nb++) acc[0][tb][nb] += s_acc[(((q - 1) * 4 + wave) * TBW * NBW + tb * NBW + nb) * 64 + lane];
        }
        // D[rank 4g+i][token m] per 16x16 block: a lane holds four neighbouring ranks of a token; ranks that do not exist
        // are stored as zero.
#pragma unroll
        for (int nb = 0; nb < NBW; nb++) {
            const int c0 = (rw * NBW + nb) * 16 + 4 * g;
            bool real[4];
#pragma unroll
            for (int e = 0; e < 4; e++) real[e] = (have >> (c0 + e) & 1ull) != 0;
#pragma unroll
            for (int mm = 0; mm < NM; mm++) {
                const SgmvProj &pm = p.pr[p0 + mm];
#pragma unroll
                for (int tb = 0; tb < TBW; tb++) {
                    const int t = (tw * TBW + tb) * 16 + m;
                    if (t >= ntok) continue;
                    float o[4];
#pragma unroll
                    for (int e = 0; e < 4; e++) o[e] = real[e] ? acc[mm][tb][nb][e] : 0.f;
                    if (pm.ksplit > 1) {
                        *reinterpret_cast<float4_t *>(pm.v + ((size_t)split * p.T + tok0 + t) * VSTRIDE + c0) = float4_t{o[0], o[1], o[2], o[3]};
                        continue;
                    }
                    if (p.scaled) {
#pragma unroll
                        for (int e = 0; e < 4; e++) o[e] = tl.scale * o[e];
                    }
                    uint32_t hi[2], lo[2];
                    split_hi_lo<DT>(o, hi, lo);
                    *reinterpret_cast<uint2 *>(pm.vhi + (size_t)(tok0 + t) * VSTRIDE + c0) = make_uint2(hi[0], hi[1]);
                    *reinterpret_cast<uint2 *>(pm.vlo + (size_t)(tok0 + t) * VSTRIDE + c0) = make_uint2(lo[0], lo[1]);
                }
            }
        }
    };
    if constexpr (SHARE) {
        if (nm == 3) { run(std::integral_constant<int, 3>{}); return; }
        if (nm == 2) { run(std::integral_constant<int, 2>{}); return; }
    }
    run(std::integral_constant<int, 1>{});
}

// ------------------------------------------------------------------ reduce
// vsum[t][c] = sum over K splits of the shrink partials, stored as hi + lo 16-bit halves so that the expand MFMAs see the
// fp32 value to about 2^-16 relative.  One thread per (token, 8 rank columns).  With one split the shrink has stored
// the halves itself; what is left then is to define the rows outside every segment.
template <int DT, int RMAX>
__global__ __launch_bounds__(256) void sgmv_reduce_kernel(const SgmvArgs p)
{
    constexpr int CPT = RMAX / 8;     // 8-column groups per token
    const SgmvProj &pj = p.pr[blockIdx.y];
    const long long idx = (long long)blockIdx.x * 256 + threadIdx.x;
    if (idx >= (long long)p.T * CPT) return;
    const int t = (int)(idx / CPT), c0 = (int)(idx - (long long)t * CPT) * 8;
    if (p.seg_uniform_len == 0 && p.tok_cover[t] == 0) {
        // token outside every segment: no tile touches its row.  y = delta mode defines it as zeros
        // (the CPT threads of the token share the row); accumulate mode keeps it.
        if (!p.accumulate) {
            uint16_t *__restrict__ yrow = static_cast<uint16_t *>(pj.y) + (size_t)t * pj.hout;
            for (int cc = c0 >> 3; cc < (pj.hout >> 3); cc += CPT) stg16(yrow + (size_t)cc * 8, zero16());
        }
        return;
    }
    if (pj.ksplit == 1) return;
    float v[8];
    sum_splits_any(pj.v + (size_t)t * VSTRIDE + c0, (size_t)p.T * VSTRIDE, pj.ksplit, v);
    uint32_t hi[4], lo[4];
    split_hi_lo<DT>(v, hi, lo);
    stg16(pj.vhi + (size_t)t * VSTRIDE + c0, make_uint4(hi[0], hi[1], hi[2], hi[3]));
    stg16(pj.vlo + (size_t)t * VSTRIDE + c0, make_uint4(lo[0], lo[1], lo[2], lo[3]));
}

// ------------------------------------------------------------------ expand
// Up to rank 32 the K splits are summed by the expand itself and the reduce launch falls away.  At rank 64 the sums are
// four times as long as at 16 and every column block of a tile repeats them, so the reduce launch stays there but for the
// launches of few tiles below (sgmv_launch_shape): 1280 tokens, seven projections, rank 64, two splits 62.6 us of expand summing,
// 55.4 and a reduce of 5.2 not; at rank 16 the whole call of 8 x 512 tokens 185 -> 179.

// The reference's call (BT) only writes y, and its whole batch is about one round of workgroups: no registers for y, and a staging
// tile of half a step, so that four workgroups fit a unit instead of three (16 x 512 tokens, rank 64, 1024 workgroups: q, k and v
// 124.5 us with three, 118.9 with four).
template <int DT, int RMAX, bool BT>
__global__ __launch_bounds__(SG_NT, BT ? 4 : 1) void sgmv_expand_kernel(const SgmvArgs p)
{
    // One workgroup: 64 tokens (16 per wavefront) x cols_per_block output columns, 128 columns per step.
    // The B tile of a step is parked in LDS row-major and read back column-wise with the transposing LDS
    // read (the MFMA needs rank as the in-lane K dimension, the pool stores rank rows).  The 16 x 128
    // result of a wavefront goes through a wavefront-private LDS tile so that y is read and written with
    // 16-byte accesses in which a 16-lane row covers 256 contiguous bytes of one token.  Loads of y and B
    // run one step ahead of the arithmetic.
    constexpr int KP = RMAX <= 32 ? 32 : 64;   // K of the expand MFMAs (rank padded with zeros)
    constexpr int KS = KP / 32;
    constexpr int NBC = TN / 16;               // 16-column blocks per step
    constexpr int BPITCH = TN * 2 + 16;        // bytes per rank row of the LDS B tile (16-byte aligned rows)
    constexpr int ON = BT ? TN / 2 : TN;       // columns staged at a time
    constexpr int OPITCH = ON + 4;             // floats per token row of the staging tile
    constexpr int TPITCH = KP * 2 + 16;        // reference layout: bytes per output column of the LDS tile (K contiguous)
    constexpr int BQ = KP * (TN / 8) / SG_NT;  // B-tile loads per thread and step (either layout: KP x TN values)
    __shared__ __attribute__((aligned(16))) unsigned char s_b[BT ? TN * TPITCH : KP * BPITCH];
    __shared__ __attribute__((aligned(16))) float s_out[SG_NT / 64][16][OPITCH];
    __shared__ int s_brow[BT ? 1 : KP];
    constexpr int VPITCH = KP + 8;             // 16-bit values per token row of the folded intermediate, which lies in s_out (BT: s_b)
    uint16_t *const s_v = BT ? reinterpret_cast<uint16_t *>(s_b) : reinterpret_cast<uint16_t *>(&s_out[0][0][0]);
    static_assert(2 * TM * VPITCH * 2 <= (int)(BT ? sizeof(s_b) : sizeof(s_out)), "the folded intermediate fits there");
    typedef __attribute__((address_space(3))) volatile float lds_vfloat;
    typedef __attribute__((address_space(3))) volatile float4_t lds_vfloat4;

    const GroupId at = group_at(p.ex_end, blockIdx.x);
    const SgmvProj &pj = p.pr[at.group];
    const int cols_per_block = pj.cols;
    int tile, colblk;
    {
        const int w = at.rest;
        if (tile_major(pj.ncb) && !few_tiles(p.max_tiles)) {
            const int ncb8 = (pj.ncb + 7) & ~7;
            tile = divided(w, ncb8, pj.ncb_inv);
            colblk = w - tile * ncb8 - ((tile >> 3) & 7);
            colblk += colblk < 0 ? ncb8 : 0;
            if (colblk >= pj.ncb) return;
        } else {
            place(w, pj.ncb, pj.ncb_inv, p.max_tiles, 0, tile, colblk);
        }
    }
    if (tile >= p.max_tiles) return;
    const Tile<BT> tl = tile_of<BT>(p, tile);        // the reference layout and equal segments go together
    const int ntok = tl.ntok, adapter = tl.adapter, r = tl.rank, tok0 = tl.tok0;
    const float scale = tl.scale;
    const PoolView &pv = p.pool;
    if (ntok <= 0 || tok0 < 0 || tok0 + ntok > p.T) return;
    const int hout = pj.hout;
    uint16_t *__restrict__ y = static_cast<uint16_t *>(pj.y);
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int m = lane & 15, g = lane >> 4;
    const int col_begin = colblk * cols_per_block;
    int col_end = col_begin + cols_per_block;
    col_end = col_end < hout ? col_end : hout;

    if (adapter < 0) {
        if (!p.accumulate) {
            // segment without adapter: y = delta means zeros
            const int cpr = (col_end - col_begin) >> 3;
            for (int e = tid; e < ntok * cpr; e += SG_NT) {
                const int t = e / cpr, c = e - t * cpr;
                stg16(y + (size_t)(tok0 + t) * hout + col_begin + c * 8, zero16());
            }
        }
        return;
    }
    if constexpr (!BT) {
        // B rows share the page table with the A rows
        for (int j = tid; j < KP; j += SG_NT) {
            const int row = j < MAX_RANK ? tl.row(j, pv.n_rows_a) : -1;
            s_brow[j] = (row >= 0 && row < pv.n_rows_b) ? row : -1;
        }
    }

    // ---- V operand: 16 tokens of this wavefront x KP ranks as a hi + lo pair of 16-bit values (written by the reduce
    // kernel, or made here out of a few splits' partial sums); rank columns beyond the adapter's rank are zero.
    int trow = wave * 16 + m;
    trow = trow < ntok ? trow : ntok - 1;
    uint4 vhi[KS], vlo[KS];
    const bool fold = p.fold && pj.ksplit > 1;
    if (fold) {
        // whole rows of the partial sums, four ranks a thread; the operands are read back from LDS behind the barrier
        constexpr int RQ = RMAX / 4;
#pragma unroll
        for (int i = 0; i < TM * RQ / SG_NT; i++) {
            const int e = i * SG_NT + tid, t = e / RQ, c0 = (e - t * RQ) * 4;
            float v[4];
            sum_splits4(pj.v + (size_t)(tok0 + (t < ntok ? t : ntok - 1)) * VSTRIDE + c0, (size_t)p.T * VSTRIDE, pj.ksplit, v);
            uint32_t hi[2], lo[2];
            split_hi_lo<DT>(v, hi, lo);
            *reinterpret_cast<uint2 *>(s_v + t * VPITCH + c0) = make_uint2(hi[0], hi[1]);
            *reinterpret_cast<uint2 *>(s_v + (TM + t) * VPITCH + c0) = make_uint2(lo[0], lo[1]);
        }
    } else {
#pragma unroll
        for (int ks = 0; ks < KS; ks++) {
            const int c0 = ks * 32 + 8 * g;
            vhi[ks] = zero16(); vlo[ks] = zero16();
            if (c0 < RMAX) {
                vhi[ks] = ldg16(pj.vhi + ((size_t)(tok0 + trow) * VSTRIDE + c0));
                vlo[ks] = ldg16(pj.vlo + ((size_t)(tok0 + trow) * VSTRIDE + c0));
            }
        }
    }
    const uint16_t *__restrict__ brows = static_cast<const uint16_t *>(pj.b_rows);
    const uint16_t *__restrict__ bt = brows + (BT ? (size_t)adapter * (size_t)pv.b_dense_stride : 0);
    __syncthreads();
    if (fold) {
#pragma unroll
        for (int ks = 0; ks < KS; ks++) {
            const int c0 = ks * 32 + 8 * g;
            const bool real = c0 < RMAX;
            vhi[ks] = real ? *reinterpret_cast<const uint4 *>(s_v + trow * VPITCH + c0) : zero16();
            vlo[ks] = real ? *reinterpret_cast<const uint4 *>(s_v + (TM + trow) * VPITCH + c0) : zero16();
        }
    }

    // Loads of a step (this thread's share of the B tile and of the y rows) are issued one step ahead.
    // y rows of this wavefront: lane handles (token p / 16, 16-byte chunk p % 16), p = lane + 64 q.
    uint4 y_nx[4], b_nx[BQ];
    const bool accumulate = !BT && p.accumulate;
    auto prefetch = [&](int col0) {
        if (accumulate) {
#pragma unroll
            for (int q = 0; q < 4; q++) {
                const int pp = lane + 64 * q, t = pp >> 4, c = pp & 15;
                const int col = col0 + c * 8;
                const bool ok = wave * 16 + t < ntok && col < col_end;
                y_nx[q] = ok ? ldg16_stream(y + (size_t)(tok0 + wave * 16 + t) * hout + col) : zero16();
            }
        }
        if constexpr (!BT) {
#pragma unroll
            for (int q = 0; q < BQ; q++) {
                const int e = tid + q * SG_NT;
                const int j = e / (TN / 8), c = e - j * (TN / 8);
                const int row = s_brow[j];
                const int col = col0 + c * 8;
                b_nx[q] = (row >= 0 && col < col_end) ? ldg16(brows + (size_t)row * hout + col) : zero16();
            }
        } else {
            // reference layout: column c of the adapter's [hout, r] block holds its r values contiguously, so
            // the tile of TN columns is one contiguous run when r = KP; 16-byte chunk (column, 8 ranks) per load
#pragma unroll
            for (int q = 0; q < BQ; q++) {
                const int e = tid + q * SG_NT;
                const int cl = e / (KP / 8), k0 = (e - cl * (KP / 8)) * 8;
                const int col = col0 + cl;
                b_nx[q] = (col < col_end && k0 < r) ? ldg16(bt + (size_t)col * r + k0) : zero16();
            }
        }
    };
    prefetch(col_begin);
#pragma unroll 1
    for (int col0 = col_begin; col0 < col_end; col0 += TN) {
        uint4 y0[4];
#pragma unroll
        for (int q = 0; q < 4; q++) y0[q] = y_nx[q];
        if constexpr (!BT) {
            // park B[0..KP) x [col0, col0+TN) in LDS, rows beyond the rank as zeros
            __syncthreads();
#pragma unroll
            for (int q = 0; q < BQ; q++) {
                const int e = tid + q * SG_NT;
                const int j = e / (TN / 8), c = e - j * (TN / 8);
                *reinterpret_cast<uint4 *>(s_b + j * BPITCH + c * 16) = b_nx[q];
            }
            __syncthreads();
        } else {
            // park the tile column-major (K contiguous per column): exactly the in-lane order the MFMA wants
            __syncthreads();
#pragma unroll
            for (int q = 0; q < BQ; q++) {
                const int e = tid + q * SG_NT;
                const int cl = e / (KP / 8), kc = e - cl * (KP / 8);
                *reinterpret_cast<uint4 *>(s_b + cl * TPITCH + kc * 16) = b_nx[q];
            }
            __syncthreads();
        }
        if (col0 + TN < col_end) prefetch(col0 + TN);
        float4_t acc[NBC];
#pragma unroll
        for (int nb = 0; nb < NBC; nb++) acc[nb] = float4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int nb = 0; nb < NBC; nb++) {
#pragma unroll
            for (int ks = 0; ks < KS; ks++) {
                uint4 bop;
                if constexpr (!BT) {
                    // lane (n = m, k group g) needs B[ks*32 + 8g + e][nb*16 + m], e < 8: a column of the row-major
                    // tile.  ds_read_b64_tr_b16 does the transpose: the 16 lanes of a group read a 4 x 16 block
                    // (lane i: row i / 4, columns 4 (i % 4) ..+3) and lane n gets the 4 rows of column n.
                    const unsigned char *src = s_b + (ks * 32 + 8 * g + (m >> 2)) * BPITCH + (nb * 16 + (m & 3) * 4) * 2;
                    const short4_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_short4 *)src);
                    const short4_t hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_short4 *)(src + 4 * BPITCH));
                    bop = make_uint4(__builtin_bit_cast(uint2, lo).x, __builtin_bit_cast(uint2, lo).y,
                                     __builtin_bit_cast(uint2, hi).x, __builtin_bit_cast(uint2, hi).y);
                } else {
                    bop = *reinterpret_cast<const uint4 *>(s_b + (nb * 16 + m) * TPITCH + (ks * 4 + g) * 16);
                }
                // D[token 4g+i][column m of the block]: A operand = V, B operand = B
                acc[nb] = mfma16<DT>(vhi[ks], bop, acc[nb]);
                acc[nb] = mfma16<DT>(vlo[ks], bop, acc[nb]);
            }
        }
        // ---- transpose through this wavefront's own LDS tile, then 16-byte row-contiguous y update.
        // The tile is private to the wavefront and LDS operations of one wavefront complete in order, so no
        // barrier is needed; the accesses are volatile so that the compiler keeps them in program order and
        // emits one ds_write_b32 per element (left to itself it pairs these stores into ds_write2_b32 and,
        // in the variant without the B tile, gets two of the paired offsets wrong).
#pragma unroll
        for (int h = 0; h < TN / ON; h++) {
            lds_vfloat *so = (lds_vfloat *)&s_out[wave][4 * g][m];
#pragma unroll
            for (int nb = 0; nb < ON / 16; nb++)
#pragma unroll
                for (int i = 0; i < 4; i++) so[i * OPITCH + nb * 16] = acc[h * (ON / 16) + nb][i];
#pragma unroll
            for (int q = 0; q < ON / 32; q++) {
                const int pp = lane + 64 * q, t = pp / (ON / 8), c = pp % (ON / 8);
                const int col = col0 + h * ON + c * 8;
                const float4_t d0 = *(lds_vfloat4 *)&s_out[wave][t][c * 8];
                const float4_t d1 = *(lds_vfloat4 *)&s_out[wave][t][c * 8 + 4];
                if (wave * 16 + t < ntok && col < col_end) {
                    float o[8];
                    if (accumulate) unpack8<DT>(y0[q], o);
                    else {
#pragma unroll
                        for (int e = 0; e < 8; e++) o[e] = 0.f;
                    }
                    o[0] = fmaf(scale, d0[0], o[0]); o[1] = fmaf(scale, d0[1], o[1]);
                    o[2] = fmaf(scale, d0[2], o[2]); o[3] = fmaf(scale, d0[3], o[3]);
                    o[4] = fmaf(scale, d1[0], o[4]); o[5] = fmaf(scale, d1[1], o[5]);
                    o[6] = fmaf(scale, d1[2], o[6]); o[7] = fmaf(scale, d1[3], o[7]);
                    stg16_stream(y + (size_t)(tok0 + wave * 16 + t) * hout + col, pack8<DT>(o));
                }
            }
        }
    }
}

// The expand of a launch of few tiles.  The kernel above takes 64 tokens at a time, one 128-column step after the other, so a
// prompt of a tile or two is a chain of a few long steps on a part of the chip.  Here a workgroup takes 16 tokens and 256
// columns, 64 per wavefront, in one step, everything requested at once: the partial sums and the row table first, then B
// and y; B is read by four workgroups instead of one.  What bounds it is the chain record -> row table -> B -> y; with each B load
// waiting for its own row lookup 3.9 us of 8.8 went by before the last was requested.
// Two layers and the plan in a graph, Llama-7B widths, that kernel -> this one, us, by workgroups: rank 64, q/k/v, 64 tokens
// 37.2 -> 27.7 (192), 2 x 100 43.3 -> 36.6 (768), 8 x 64 60.7 -> 51.6 (2304), 2 x 512 69.1 -> 68.2 (3264), 8 x 128 73.1 -> 77.4 (3840);
// seven projections, 2 x 100 72.9 -> 66.7 (2656), 4 x 64 77.2 -> 79.7 (3984).  Rank 32, q/k/v, 64 tokens 31.0 -> 25.0, 8 x 128
// 63.3 -> 62.0 (3840); q/k/v/o 8 x 128 74.6 -> 71.6 (5120); seven projections 8 x 64 85.1 -> 95.9 (7968).  Rank 16, q/k/v/o 16 x 64
// 71.5 -> 70.9 (6144); seven 8 x 64 78.2 -> 83.0 (7968).
// The number is that of 64-token tiles the batch is likely to make (sgmv_launch_shape), four pieces each, and not that of the
// grid, which covers the host's bound on tiles: many short prompts leave most of a grid empty and are where this kernel gains
// most, one piece a prompt against a whole tile.  Seven projections, 16 x 4 tokens (5976 by the rule, 22576 dispatched, 2656 with
// tokens) 70.8 -> 59.4 at rank 16, 76.2 -> 65.2 at 32; 32 x 8, beyond the line, 119 -> 102 (rank 16); q/k/v/o 24 x 8 52.2 ->
// 45.8.  Over 1 to 32 prompts of 1 to 400 tokens, ranks 16 and 32, four sets of projections (whole, of the larger model, as one
// of two shards, ragged), each batch alone or sixteen in turn, the rule is 0.1 to 1.0 % off the better kernel on average, at rank
// 64 0.3 to 1.9 % (beyond its line prompts of up to 16 tokens would gain 6 to 20 %).  It is worst with all seven projections of
// the whole layer at 40 to 100 tokens a prompt: 8 x 40 62.1 -> 69.2 at rank 16, 71.7 -> 80.4 at 32, 3 x 100 58.2 -> 60.6 and
// 60.9 -> 65.4; any lower line would lose more on the narrower layers, where the same numbers gain up to 20 %.
// One number up to rank 32, as both kernels sum the splits there whatever their number.  Above, this one saves the reduce launch,
// but not with one K split: rank 64, q/k/v, 2 x 100 59.9 -> 58.3 (768), 8 x 64 71.9 -> 71.7 (2304); there the line lies where
// four projections of 128 tokens do (512).
// The reference's call, whose B is four times as many lines from L2, against the kernel above with four workgroups a unit; three
// calls on one x, several inputs in turn, hidden 4096: rank 16, 4 x 256 34.4 -> 32.1 (1024), 6 x 256 41.3 -> 40.8 (1536), 16 x 100
// 42.5 -> 46.9 (2048), 8 x 512 59.7 -> 63.3 (4096), 12 x 512 80.7 -> 86.6 (6144); rank 32, 6 x 256 45.4 -> 45.7 (1536), 8 x 256
// 48.4 -> 50.9 (2048); hidden 5120, rank 16, 6 x 256 45.0 -> 43.5 (1920), 8 x 256 49.1 -> 52.2 (2560).  Rank 64, 16 x 64 54.7 -> 52.9
// (1024) and 63.1 -> 59.6 (1280, hidden 5120), 4 x 512 59.8 -> 65.2 (2048).
constexpr int FEW_COLS = 256;
static int few_expand(int max_rank, bool bt, int splits)                // workgroups up to which it is taken
{
    if (max_rank <= 32) return bt ? 2047 : 6144;
    return splits == 1 ? 512 : (bt ? 1023 : 3200);
}
template <int DT, int RMAX, bool BT>
__global__ __launch_bounds__(SG_NT) void sgmv_expand_few_kernel(const SgmvArgs p)
{
    constexpr int KP = RMAX <= 32 ? 32 : 64, KS = KP / 32;      // K of the MFMAs (rank padded with zeros)
    constexpr int CW = FEW_COLS / 4, NBC = CW / 16;             // columns of a wavefront
    constexpr int BPITCH = CW * 2 + 16, TPITCH = KP * 2 + 16;   // bytes per LDS row of B: a rank row, or (reference layout) an output column
    constexpr int BQ = KP / 8;                                  // B loads per lane
    constexpr int VPITCH = KP + 8, OPITCH = CW + 4;
    constexpr int BBYTES = BT ? CW * TPITCH : KP * BPITCH, WBYTES = BBYTES > 16 * OPITCH * 4 ? BBYTES : 16 * OPITCH * 4;
    __shared__ __attribute__((aligned(16))) unsigned char s_b[4][WBYTES];       // private to a wavefront: B, then its result
    __shared__ __attribute__((aligned(16))) uint16_t s_v[2][16][VPITCH];
    static_assert(16 * OPITCH * 4 <= sizeof(s_b[0]), "a wavefront's result fits its B tile");

    // grid: column blocks of all projections x pieces
    const GroupId at = group_at(p.ex_end, blockIdx.x);
    const SgmvProj &pj = p.pr[at.group];
    const int colblk = at.rest, tile = (int)blockIdx.y >> 2, sub = (int)blockIdx.y & 3;
    const Tile<BT> tl = tile_of<BT>(p, tile);
    const int ntok = tl.ntok - sub * 16 < 16 ? tl.ntok - sub * 16 : 16, tok0 = tl.tok0 + sub * 16;
    if (ntok <= 0 || tok0 < 0 || tok0 + ntok > p.T) return;
    const int hout = pj.hout, r = tl.rank;
    uint16_t *__restrict__ y = static_cast<uint16_t *>(pj.y);
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int m = lane & 15, g = lane >> 4;
    const int col0 = colblk * FEW_COLS + wave * CW;
    // this lane's pieces of y: token q * 8 + lane / 8, 8 columns
    const int yc = col0 + (lane & 7) * 8;
    if (tl.adapter < 0) {
        if (!p.accumulate && yc < hout)
#pragma unroll
            for (int q = 0; q < 2; q++)
                if (q * 8 + (lane >> 3) < ntok) stg16(y + (size_t)(tok0 + q * 8 + (lane >> 3)) * hout + yc, zero16());
        return;
    }
    // Row of rank row `lane`, requested with the partial sums; a B load gets its row from another lane.
    int mine = -1;
    if constexpr (!BT) mine = tl.row(lane, p.pool.n_rows_a);
    const int nsplit = pj.ksplit;
    const bool fold = p.fold && nsplit > 1;
    // folding: 16 tokens x KP / 4 quads; the shrink has filled RMAX columns
    const int ft = tid / (KP / 4) & 15, fc = (tid % (KP / 4)) * 4, fs = fc < RMAX ? fc : 0;
    float4_t part[SGMV_SPLITS];                                         // (requested also where there is nothing to fold: no branch)
    {
        const float *src = pj.v + (size_t)(tok0 + (ft < ntok ? ft : ntok - 1)) * VSTRIDE + fs;
        const size_t stride = (size_t)p.T * VSTRIDE;
#pragma unroll
        for (int u = 0; u < SGMV_SPLITS; u++) part[u] = *reinterpret_cast<const float4_t *>(src + (u < nsplit ? u : 0) * stride);
    }
    // B and y: every load is made, at an address inside the operand, and what is not wanted becomes zero when it has arrived
    const uint16_t *__restrict__ brows = static_cast<const uint16_t *>(pj.b_rows);
    uint4 bv[BQ];
    bool bok[BQ];
    if constexpr (!BT) {
        int row[BQ];
#pragma unroll
        for (int q = 0; q < BQ; q++) row[q] = __shfl(mine, q * 8 + (lane >> 3));
#pragma unroll
        for (int q = 0; q < BQ; q++) {
            bok[q] = row[q] >= 0 && row[q] < p.pool.n_rows_b && yc < hout;
            bv[q] = ldg16(brows + (bok[q] ? (size_t)row[q] * hout + yc : 0));
        }
    } else {
        const uint16_t *__restrict__ bt = brows + (size_t)tl.adapter * (size_t)p.pool.b_dense_stride;
#pragma unroll
        for (int q = 0; q < BQ; q++) {
            const int e = q * 64 + lane, col = col0 + e / (KP / 8), k0 = (e % (KP / 8)) * 8;
            bok[q] = col < hout && k0 < r;
            bv[q] = ldg16(bt + (bok[q] ? (size_t)col * r + k0 : 0));
        }
    }
    uint4 yv[2] = {zero16(), zero16()};
    if (p.accumulate) {
#pragma unroll
        for (int q = 0; q < 2; q++) {
            const int t = q * 8 + (lane >> 3);
            yv[q] = ldg16_stream(y + (size_t)(tok0 + (t < ntok ? t : ntok - 1)) * hout + (yc < hout ? yc : 0));
        }
    }
    const int trow = m < ntok ? m : ntok - 1;
    uint4 vhi[KS], vlo[KS];
    if (fold) {
        float v[4];
#pragma unroll
        for (int e = 0; e < 4; e++) {
            v[e] = 0.f;
#pragma unroll
            for (int u = 0; u < SGMV_SPLITS; u++) v[e] += u < nsplit ? part[u][e] : 0.f;
            v[e] = fc < RMAX ? v[e] : 0.f;
        }
        uint32_t hi[2], lo[2];
        split_hi_lo<DT>(v, hi, lo);
        *reinterpret_cast<uint2 *>(&s_v[0][ft][fc]) = make_uint2(hi[0], hi[1]);
        *reinterpret_cast<uint2 *>(&s_v[1][ft][fc]) = make_uint2(lo[0], lo[1]);
        __syncthreads();
#pragma unroll
        for (int ks = 0; ks < KS; ks++) {
            vhi[ks] = *reinterpret_cast<const uint4 *>(&s_v[0][trow][ks * 32 + 8 * g]);
            vlo[ks] = *reinterpret_cast<const uint4 *>(&s_v[1][trow][ks * 32 + 8 * g]);
        }
    } else {
#pragma unroll
        for (int ks = 0; ks < KS; ks++) {
            const int c0 = ks * 32 + 8 * g;
            vhi[ks] = c0 < RMAX ? ldg16(pj.vhi + (size_t)(tok0 + trow) * VSTRIDE + c0) : zero16();
            vlo[ks] = c0 < RMAX ? ldg16(pj.vlo + (size_t)(tok0 + trow) * VSTRIDE + c0) : zero16();
        }
    }
    // the wavefront's B tile through its own LDS, then its result: operations of one wavefront on LDS complete in order
    unsigned char *sb = s_b[wave];
#pragma unroll
    for (int q = 0; q < BQ; q++) {
        const int e = q * 64 + lane;
        unsigned char *at = BT ? sb + e / (KP / 8) * TPITCH + e % (KP / 8) * 16 : sb + e / 8 * BPITCH + e % 8 * 16;
        const uint32_t keep = bok[q] ? ~0u : 0u;
        *reinterpret_cast<uint4 *>(at) = make_uint4(bv[q].x & keep, bv[q].y & keep, bv[q].z & keep, bv[q].w & keep);
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
    float4_t acc[NBC];
#pragma unroll
    for (int nb = 0; nb < NBC; nb++) {
        acc[nb] = float4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int ks = 0; ks < KS; ks++) {
            uint4 bop;
            if constexpr (!BT) {
                // lane (column m, ranks ks * 32 + 8 g ..) by the transposing read, see the kernel above
                const unsigned char *src = sb + (ks * 32 + 8 * g + (m >> 2)) * BPITCH + (nb * 16 + (m & 3) * 4) * 2;
                const uint2 lo = __builtin_bit_cast(uint2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_short4 *)src));
                const uint2 hi = __builtin_bit_cast(uint2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_short4 *)(src + 4 * BPITCH)));
                bop = make_uint4(lo.x, lo.y, hi.x, hi.y);
            } else {
                bop = *reinterpret_cast<const uint4 *>(sb + (nb * 16 + m) * TPITCH + (ks * 4 + g) * 16);
            }
            acc[nb] = mfma16<DT>(vhi[ks], bop, acc[nb]);
            acc[nb] = mfma16<DT>(vlo[ks], bop, acc[nb]);
        }
    }
    // D[token 4g+i][column m of the block]
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
    float *so = reinterpret_cast<float *>(sb);
#pragma unroll
    for (int nb = 0; nb < NBC; nb++)
#pragma unroll
        for (int i = 0; i < 4; i++) so[(4 * g + i) * OPITCH + nb * 16 + m] = acc[nb][i];
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int q = 0; q < 2; q++) {
        const int t = q * 8 + (lane >> 3);
        if (t >= ntok || yc >= hout) continue;
        const float4_t d0 = *reinterpret_cast<const float4_t *>(so + t * OPITCH + (lane & 7) * 8);
        const float4_t d1 = *reinterpret_cast<const float4_t *>(so + t * OPITCH + (lane & 7) * 8 + 4);
        float o[8];
        unpack8<DT>(yv[q], o);                                  // zeros when not accumulating
#pragma unroll
        for (int e = 0; e < 4; e++) { o[e] = fmaf(tl.scale, d0[e], o[e]); o[4 + e] = fmaf(tl.scale, d1[e], o[4 + e]); }
        stg16_stream(y + (size_t)(tok0 + t) * hout + yc, pack8<DT>(o));
    }
}

void sgmv_launch_shape(SgmvArgs &a, int max_rank, int phases)
{
    a.scaled = !(phases & SGMV_APPLY);                          // the base GEMM + LoRA kernel takes the scaled intermediate
    if (a.scaled) return;
    long long few_wgs = 0;
    int most = 1;
    for (int q = 0; q < a.n_proj; q++) {
        few_wgs += (long long)a.tiles * 4 * ((a.pr[q].hout + FEW_COLS - 1) / FEW_COLS);
        most = a.pr[q].ksplit > most ? a.pr[q].ksplit : most;
    }
    a.few = few_wgs <= few_expand(max_rank, a.seg_uniform_len > 0, most);
    // The expand sums the splits itself up to rank 32 and in launches of few tiles; rows outside every segment are zeroed by the
    // reduce launch only.
    a.fold = (max_rank <= 32 || a.few) && (a.accumulate || a.seg_uniform_len > 0);
    // Without splits the shrink has stored the halves itself, and the launch would only read the cover flags: two projections
    // of 25 x 64 tokens, rank 64, hin 512 15.6 -> 14.0 us a call, q/k/v/o of 16 x 500 tokens at hidden 4096 153.4 -> 151.7.
    a.reduce = !a.fold && (most > 1 || !(a.accumulate || a.seg_uniform_len > 0));
}

template <int DT, int RMAX>
static int launch_rmax(const SgmvArgs &a, int phases, hipStream_t s)
{
    int rc = 0;
    if ((phases & SGMV_PLAN) && a.seg_uniform_len == 0) {
        const int by_tiles = (a.max_tiles + PLAN_TILES - 1) / PLAN_TILES, by_tokens = (a.T + PLAN_TOKENS - 1) / PLAN_TOKENS;
        hipLaunchKernelGGL(sgmv_plan_kernel, dim3((unsigned)(by_tiles > by_tokens ? by_tiles : by_tokens)), dim3(PLAN_NT), 0, s, a);
        rc = (int)hipGetLastError();
        if (rc) return rc;
    }
    if (!(phases & (SGMV_APPLY | SGMV_SHRINK))) return 0;
    // The caller has filled pr[], the shrink groups, ksplit, cols and ncb; the rest of the shape and the grid ends are set here.
    SgmvArgs g = a;
    sgmv_launch_shape(g, RMAX, phases);
    for (int q = 0; q < g.n_proj; q++) {
        SgmvProj &pj = g.pr[q];
        const int nstage = (pj.hin + 63) / 64;
        pj.kper = (nstage + pj.ksplit - 1) / pj.ksplit;
        pj.ksplit_inv = inverse_of(pj.ksplit);
        pj.ncb_inv = inverse_of(tile_major(pj.ncb) && !few_tiles(g.max_tiles) ? (pj.ncb + 7) & ~7 : pj.ncb);
    }
    g.seg_tiles = (g.seg_uniform_len + TM - 1) / TM;
    g.seg_tiles_inv = inverse_of(g.seg_tiles);
    unsigned end = 0;
    const bool rows = tile_rows(g.max_tiles);
    for (int q = 0; q < MAX_PROJ; q++) {
        if (q < g.n_grp) {
            const int splits = g.pr[g.grp_first[q]].ksplit;
            end += (unsigned)((rows ? splits : place_grid(g.max_tiles, splits)) * (g.share_x ? 1 : g.grp_n[q]));
        }
        g.grp_end[q] = q < g.n_grp ? end : ~0u;
    }
    const dim3 sgrid(end, rows ? (unsigned)g.max_tiles : 1u);
    end = 0;
    for (int q = 0; q < MAX_PROJ; q++) {
        if (q < g.n_proj)
            end += g.few ? (unsigned)((g.pr[q].hout + FEW_COLS - 1) / FEW_COLS) : (unsigned)expand_grid(g.max_tiles, g.pr[q].ncb);
        g.ex_end[q] = q < g.n_proj ? end : ~0u;
    }
    const dim3 egrid(end, g.few ? (unsigned)g.max_tiles * 4u : 1u);
    if ((g.seg_uniform_len > 0) != (g.b_transposed != 0)) return (int)hipErrorInvalidValue;
    if (g.seg_uniform_len > 0 && g.share_x) return (int)hipErrorInvalidValue;
    const dim3 threads(SG_NT * (g.share_x ? SH_KG<true> : SH_KG<false>));
    if (g.seg_uniform_len > 0) hipLaunchKernelGGL((sgmv_shrink_kernel<DT, RMAX, true, false>), sgrid, threads, 0, s, g);
    else if (g.share_x) hipLaunchKernelGGL((sgmv_shrink_kernel<DT, RMAX, false, true>), sgrid, threads, 0, s, g);
    else hipLaunchKernelGGL((sgmv_shrink_kernel<DT, RMAX, false, false>), sgrid, threads, 0, s, g);
    rc = (int)hipGetLastError();
    if (rc || !(phases & SGMV_APPLY)) return rc;
    if (g.reduce) {
        const long long n = (long long)g.T * (RMAX / 8);
        hipLaunchKernelGGL((sgmv_reduce_kernel<DT, RMAX>), dim3((unsigned)((n + 255) / 256), (unsigned)g.n_proj), dim3(256), 0, s, g);
        rc = (int)hipGetLastError();
        if (rc) return rc;
    }
    if (g.few) {
        if (g.b_transposed) hipLaunchKernelGGL((sgmv_expand_few_kernel<DT, RMAX, true>), egrid, dim3(SG_NT), 0, s, g);
        else hipLaunchKernelGGL((sgmv_expand_few_kernel<DT, RMAX, false>), egrid, dim3(SG_NT), 0, s, g);
        return (int)hipGetLastError();
    }
    if (g.b_transposed)
        hipLaunchKernelGGL((sgmv_expand_kernel<DT, RMAX, true>), egrid, dim3(SG_NT), 0, s, g);
    else
        hipLaunchKernelGGL((sgmv_expand_kernel<DT, RMAX, false>), egrid, dim3(SG_NT), 0, s, g);
    return (int)hipGetLastError();
}

template <int DT>
static int launch_sg_dt(const SgmvArgs &a, int max_rank, int phases, hipStream_t s)
{
    if (max_rank <= 16) return launch_rmax<DT, 16>(a, phases, s);
    if (max_rank <= 32) return launch_rmax<DT, 32>(a, phases, s);
    return launch_rmax<DT, 64>(a, phases, s);
}

int launch_sgmv(const SgmvArgs &a, int dtype, int max_rank, int phases, hipStream_t s)
{
    if (dtype == DT_F16) return launch_sg_dt<DT_F16>(a, max_rank, phases, s);
    return launch_sg_dt<DT_BF16>(a, max_rank, phases, s);
}

}  // namespace mlora
