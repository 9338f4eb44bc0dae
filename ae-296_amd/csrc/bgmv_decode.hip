// BGMV decode kernel for gfx950: y[t] (+)= s_a * (x[t] . A_a) . B_a, shrink and expand
// fused in one launch.  One workgroup owns one work item = up to G tokens that use the
// same adapter (G = 1: one token per workgroup), so an adapter's rows are fetched once
// per item and the rank-r intermediate never leaves the CU (fp32 in LDS).
//
// Work items come in two forms:
//   - work records written by the gather kernel (WORK = true): one 320-byte record per
//     workgroup holding the tokens, the adapter's rank, scaling and the row index of every
//     rank row, already placed in launch order -- one dependent load before the streaming
//     starts, no table walk, no barrier;
//   - the plain form (WORK = false): workgroup t serves token t and walks the page table
//     (or the dense reference layout) itself.
//
// Shrink: a wavefront is split into four 16-lane DPP rows.  Each 16-lane row reads
// 256 contiguous bytes (two 128-byte lines) of one rank row per load, rank rows are
// dealt round-robin to the four lane rows, and wavefronts split the Hin columns.  The
// per-lane partial dot products are reduced with four DPP adds inside the 16-lane row
// and across wavefronts through LDS.
// Expand: every lane owns 8 contiguous output columns, so a wavefront reads 1 KiB
// contiguous from each B rank row and writes y with 16-byte stores.  With PF the first B rows
// and the y rows of a lane's first output chunk are requested ahead of the expand: with one or two tokens
// an item behind the first A rows (one round trip to memory less: 32 tokens of rank 16 9.0 -> 8.6 us a call,
// 64 tokens x 3 projections 10.4 -> 10.2), with more into the registers the A rows have just vacated
// (up to 20 % at four tokens per item and rank 64).
//
// Replaces punica.ops.add_lora_bgmv as called from lightllm/models/lora_gpu.py:138,150,162.
#include "mlora_args.hpp"
#include "mlora_dev.hpp"

namespace mlora {

__device__ __forceinline__ int pool_row(const int32_t *__restrict__ tbl, long long dense_stride, int adapter, int j,
                                        const PoolView &pv, long long n_rows)
{
    long long row;
    if (tbl) {
        int pg = tbl[(long long)adapter * pv.max_pages + (j >> pv.page_shift)];
        row = pg < 0 ? -1 : (((long long)pg << pv.page_shift) + (j & ((1 << pv.page_shift) - 1)));
    } else {
        row = (long long)adapter * dense_stride + j;
    }
    return (row < 0 || row >= n_rows) ? -1 : (int)row;
}

template <int DT, int G, int RMAX, int NT, bool BT, bool WORK, bool PF>
__global__ __launch_bounds__(NT) void bgmv_kernel(const BgmvArgs p)
{
    constexpr int NW = NT / 64;
    constexpr int RPG = RMAX / 4;                               // rank rows per 16-lane row
    constexpr int UB = 32 / (RPG + G);                          // ~128 VGPRs of loads in flight
    constexpr int U = UB >= 4 ? 4 : (UB >= 2 ? 2 : 1);          // column steps kept in flight
    constexpr int EB = RMAX < 16 ? RMAX : 16;                   // B rank rows in flight per lane
    __shared__ float s_part[NW][G][RMAX];
    __shared__ __attribute__((aligned(16))) float s_v[G][RMAX];
    __shared__ int s_arow[WORK ? 1 : RMAX];
    __shared__ int s_brow[WORK ? 1 : RMAX];

    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int cl = lane & 15, rg = lane >> 4;
    const PoolView &pv = p.pool;

    int proj, part = 0, ntok = 1, adapter, r;
    float scale;
    int tok[G];
    const int32_t *__restrict__ rows = nullptr;                 // WORK: row index of rank row j at rows[j]

    if constexpr (WORK) {
        // Records are stored in launch order: record b belongs to workgroup b of every projection.
        // The gather interleaves consecutive chunks over the 8 XCDs (workgroups are dealt to XCDs
        // round-robin by id), so the chunks of one hot adapter share one XCD's L2.
        const int b = (int)blockIdx.x;
        proj = (int)blockIdx.y;
        part = (int)blockIdx.z;
        const int32_t *__restrict__ rec = p.work + (size_t)b * WORK_WORDS;
        ntok = rec[0];
        if (ntok <= 0) return;
        ntok = ntok < G ? ntok : G;
        adapter = rec[1];
        r = rec[2];
        scale = __builtin_bit_cast(float, rec[3]);
#pragma unroll
        for (int k = 0; k < G; k++) {
            const int t = k < ntok ? rec[4 + k] : -1;
            tok[k] = (t >= 0 && t < p.T) ? t : -1;
        }
        rows = rec + WORK_ROWS_AT;
    } else {
        const int item = (int)blockIdx.x;
        proj = (int)blockIdx.y;
        tok[0] = item;
#pragma unroll
        for (int k = 1; k < G; k++) tok[k] = -1;
        if (p.tok_adapter) {
            // int32 ids: any negative id and any id beyond the pool mean "no adapter" (the row is
            // defined: kept when accumulating, zeros otherwise), as the work-record path treats them
            adapter = p.tok_adapter[item];
            if (adapter < 0 || adapter >= pv.n_adapters) adapter = -1;
        } else {
            // int64 ids of the reference-layout call: a bad index leaves the row untouched (-2)
            const long long a64 = p.tok_adapter64[item];
            adapter = (a64 < 0 || a64 >= pv.n_adapters) ? -2 : (int)a64;
        }
        r = 0;
        scale = 0.f;
        if (adapter >= 0) {
            r = pv.rank ? pv.rank[adapter] : pv.uniform_rank;
            scale = pv.scaling ? pv.scaling[adapter] : pv.uniform_scale;
            if (pv.a_tbl || pv.b_tbl) {
                const int cap = pv.max_pages << pv.page_shift;
                r = r > cap ? cap : r;
            }
        }
    }
    r = r < 0 ? 0 : (r > RMAX ? RMAX : r);

    const int hin = p.hin[proj], hout = p.hout[proj];
    const uint16_t *__restrict__ x = static_cast<const uint16_t *>(p.x[proj]);
    uint16_t *__restrict__ y = static_cast<uint16_t *>(p.y[proj]);
    const uint16_t *__restrict__ arows = static_cast<const uint16_t *>(p.a_rows[proj]);
    const uint16_t *__restrict__ brows = static_cast<const uint16_t *>(p.b_rows[proj]);
    // the 16-byte chunks of a row of y that this workgroup makes
    const int per_part = WORK ? ((hout >> 3) + (1 << p.part_shift) - 1) >> p.part_shift : hout >> 3;
    const int cc0 = part * per_part, cc1 = cc0 + per_part < (hout >> 3) ? cc0 + per_part : hout >> 3;

    if (adapter < 0) {
        // No adapter: y = delta mode must still define the row (zeros).  The reference-layout
        // call (tok_adapter64) leaves rows with a bad index untouched.
        if (!p.accumulate && adapter == -1) {
#pragma unroll
            for (int k = 0; k < G; k++)
                if (tok[k] >= 0)
                    for (int cc = cc0 + tid; cc < cc1; cc += NT) stg16(y + (size_t)tok[k] * hout + (size_t)cc * 8, zero16());
        }
        return;
    }

    if constexpr (!WORK) {
        // Row index of every rank row, looked up once per work item (-1 = absent / out of bounds).
        for (int j = tid; j < RMAX; j += NT) {
            s_arow[j] = j < r ? pool_row(pv.a_tbl, pv.a_dense_stride, adapter, j, pv, pv.n_rows_a) : -1;
            if constexpr (!BT) s_brow[j] = j < r ? pool_row(pv.b_tbl, pv.b_dense_stride, adapter, j, pv, pv.n_rows_b) : -1;
        }
        __syncthreads();
    }
    // Row lookups.  Records hold -1 for every absent rank row, so record reads need no rank guard
    // and are issued as plain (batched) loads.
    auto a_row = [&](int j) -> int {
        if constexpr (WORK) { const int row = rows[j]; return (row >= 0 && row < pv.n_rows_a) ? row : -1; }
        else return s_arow[j];
    };
    auto b_rows_of = [&](int j0, int (&out)[EB]) {     // rows of rank rows j0 .. j0+EB-1 (wavefront-uniform)
        if constexpr (WORK) {
            if constexpr (EB % 4 == 0) {
                const int4 *q = reinterpret_cast<const int4 *>(rows + j0);
#pragma unroll
                for (int m = 0; m < EB / 4; m++) {
                    const int4 v = q[m];
                    out[4 * m] = v.x; out[4 * m + 1] = v.y; out[4 * m + 2] = v.z; out[4 * m + 3] = v.w;
                }
            } else {
#pragma unroll
                for (int jj = 0; jj < EB; jj++) out[jj] = rows[j0 + jj];
            }
#pragma unroll
            for (int jj = 0; jj < EB; jj++) out[jj] = (out[jj] >= 0 && out[jj] < pv.n_rows_b) ? out[jj] : -1;
        } else {
#pragma unroll
            for (int jj = 0; jj < EB; jj++) out[jj] = __builtin_amdgcn_readfirstlane(s_brow[j0 + jj]);
        }
    };

    // ---------------------------------------------------------------- shrink
    // Loads are unconditional: an absent rank row reads row 0 of the slab and a token slot
    // beyond ntok reads token 0 (both discarded below), a column chunk past the end of the
    // row re-reads the last chunk with x forced to zero.
    const int ncc_in = hin >> 3;
    const int cpw = ((ncc_in + NW * 16 - 1) / (NW * 16)) * 16;   // 16-byte column chunks per wavefront
    const int n_it = cpw >> 4;
    const int c0 = wave * cpw + cl;
    const uint4 *ap[RPG];
    unsigned row_ok = 0;
#pragma unroll
    for (int i = 0; i < RPG; i++) {
        const int row = a_row(rg + 4 * i);
        row_ok |= (row >= 0 ? 1u : 0u) << i;
        ap[i] = reinterpret_cast<const uint4 *>(arows + (size_t)(row >= 0 ? row : 0) * hin);
    }
    const uint4 *xp[G];
#pragma unroll
    for (int k = 0; k < G; k++) xp[k] = reinterpret_cast<const uint4 *>(x + (size_t)(tok[k] >= 0 ? tok[k] : 0) * hin);
    float acc[G][RPG];
#pragma unroll
    for (int k = 0; k < G; k++)
#pragma unroll
        for (int i = 0; i < RPG; i++) acc[k][i] = 0.f;

    uint4 xv[G][U];
    uint4 av[RPG][U];
    auto request = [&](int it0) {
#pragma unroll
        for (int u = 0; u < U; u++) {
            const int c = c0 + (it0 + u) * 16, cs = c < ncc_in ? c : ncc_in - 1;
#pragma unroll
            for (int k = 0; k < G; k++) xv[k][u] = ldg16_stream(xp[k] + cs);
#pragma unroll
            for (int i = 0; i < RPG; i++) av[i][u] = ldg16_stream(ap[i] + cs);
        }
    };
    auto multiply = [&](int it0) {
#pragma unroll
        for (int u = 0; u < U; u++) {
            const bool cv = (it0 + u) < n_it && c0 + (it0 + u) * 16 < ncc_in;
#pragma unroll
            for (int k = 0; k < G; k++) {
                xv[k][u].x = cv ? xv[k][u].x : 0u; xv[k][u].y = cv ? xv[k][u].y : 0u;
                xv[k][u].z = cv ? xv[k][u].z : 0u; xv[k][u].w = cv ? xv[k][u].w : 0u;
            }
#pragma unroll
            for (int i = 0; i < RPG; i++)
#pragma unroll
                for (int k = 0; k < G; k++) acc[k][i] = dot8<DT>(av[i][u], xv[k][u], acc[k][i]);
        }
    };
    // First expand step: its rows and y are requested behind the first A rows of an item of one or two tokens, and arrive while
    // those are multiplied; with more tokens, when the A rows have left their registers.
    constexpr bool EARLY = PF && G <= 2;
    uint4 bpre[PF ? EB : 1];
    uint4 ypre[PF ? G : 1];
    auto request_expand = [&]() {
        if (cc0 + tid < cc1) {
            int br[EB];
            b_rows_of(0, br);
#pragma unroll
            for (int jj = 0; jj < EB; jj++)
                bpre[jj] = br[jj] >= 0 ? ldg16_stream(brows + (size_t)br[jj] * hout + (size_t)(cc0 + tid) * 8) : zero16();
#pragma unroll
            for (int k = 0; k < G; k++)
                ypre[k] = (p.accumulate && tok[k] >= 0) ? ldg16_stream(y + (size_t)tok[k] * hout + (size_t)(cc0 + tid) * 8) : zero16();
        }
    };
    request(0);
    if constexpr (EARLY) {
        request_expand();
        asm volatile("" ::: "memory");                          // the compiler leaves the requests there
    }
    multiply(0);
#pragma unroll 1
    for (int it0 = U; it0 < n_it; it0 += U) { request(it0); multiply(it0); }
    if constexpr (PF && !EARLY) request_expand();

#pragma unroll
    for (int k = 0; k < G; k++)
#pragma unroll
        for (int i = 0; i < RPG; i++) {
            const float a = ((row_ok >> i) & 1u) ? acc[k][i] : 0.f;
            const float s = row16_sum(a);
            if (cl == 0) s_part[wave][k][rg + 4 * i] = s;
        }
    __syncthreads();
    for (int e = tid; e < G * RMAX; e += NT) {
        const int k = e / RMAX, j = e - k * RMAX;
        float s = 0.f;
#pragma unroll
        for (int wv = 0; wv < NW; wv++) s += s_part[wv][k][j];
        s_v[k][j] = j < r ? s * scale : 0.f;
    }
    __syncthreads();

    // ---------------------------------------------------------------- expand
    if constexpr (!BT) {
#pragma unroll 1
        for (int cc = cc0 + tid; cc < cc1; cc += NT) {
            const bool pre = PF && cc == cc0 + tid;            // this step's first rows and y are already in registers
            float o[G][8];
#pragma unroll
            for (int k = 0; k < G; k++) {
                if (p.accumulate && tok[k] >= 0) {
                    uint4 yv;
                    if (pre) yv = ypre[k]; else yv = ldg16_stream(y + (size_t)tok[k] * hout + (size_t)cc * 8);
                    unpack8<DT>(yv, o[k]);
                } else {
#pragma unroll
                    for (int e = 0; e < 8; e++) o[k][e] = 0.f;
                }
            }
#pragma unroll 1
            for (int j0 = 0; j0 < r; j0 += EB) {
                uint4 bv[EB];
                if (pre && j0 == 0) {
#pragma unroll
                    for (int jj = 0; jj < EB; jj++) bv[jj] = bpre[jj];
                } else {
                    int br[EB];
                    b_rows_of(j0, br);
#pragma unroll
                    for (int jj = 0; jj < EB; jj++)
                        bv[jj] = br[jj] >= 0 ? ldg16_stream(brows + (size_t)br[jj] * hout + (size_t)cc * 8) : zero16();
                }
#pragma unroll
                for (int jj = 0; jj < EB; jj++) {
                    float f[8];
                    unpack8<DT>(bv[jj], f);
#pragma unroll
                    for (int k = 0; k < G; k++) {
                        const float vk = s_v[k][j0 + jj];
#pragma unroll
                        for (int e = 0; e < 8; e++) o[k][e] = fmaf(vk, f[e], o[k][e]);
                    }
                }
            }
#pragma unroll
            for (int k = 0; k < G; k++)
                if (tok[k] >= 0) stg16_stream(y + (size_t)tok[k] * hout + (size_t)cc * 8, pack8<DT>(o[k]));
        }
    } else {
        // B given as [hout, r] blocks (reference layout): output column c is the dot product
        // of v with the r contiguous values at brows + adapter * stride + c * r.
        const uint16_t *__restrict__ bt = brows + (size_t)adapter * (size_t)pv.b_dense_stride;
        if ((r & 7) == 0) {
            const int npair = hout >> 1;
            for (int cp = tid; cp < npair; cp += NT) {
                float o[G][2];
#pragma unroll
                for (int k = 0; k < G; k++) {
                    o[k][0] = 0.f; o[k][1] = 0.f;
                    if (p.accumulate && tok[k] >= 0) {
                        const uint32_t u = *reinterpret_cast<const uint32_t *>(y + (size_t)tok[k] * hout + (size_t)cp * 2);
                        o[k][0] = lo_f32<DT>(u); o[k][1] = hi_f32<DT>(u);
                    }
                }
                const uint16_t *b0 = bt + (size_t)cp * 2 * r;
#pragma unroll
                for (int j0 = 0; j0 < RMAX; j0 += 8) {
                    if (j0 < r) {
                        float f0[8], f1[8];
                        unpack8<DT>(ldg16(b0 + j0), f0);
                        unpack8<DT>(ldg16(b0 + r + j0), f1);
#pragma unroll
                        for (int k = 0; k < G; k++)
#pragma unroll
                            for (int e = 0; e < 8; e++) {
                                const float vk = s_v[k][j0 + e];
                                o[k][0] = fmaf(vk, f0[e], o[k][0]);
                                o[k][1] = fmaf(vk, f1[e], o[k][1]);
                            }
                    }
                }
#pragma unroll
                for (int k = 0; k < G; k++)
                    if (tok[k] >= 0)
                        *reinterpret_cast<uint32_t *>(y + (size_t)tok[k] * hout + (size_t)cp * 2) = pack2<DT>(o[k][0], o[k][1]);
            }
        } else {
            for (int c = tid; c < hout; c += NT) {
                float o[G];
#pragma unroll
                for (int k = 0; k < G; k++) {
                    o[k] = 0.f;
                    if (p.accumulate && tok[k] >= 0) {
                        const uint32_t u = y[(size_t)tok[k] * hout + c];
                        o[k] = lo_f32<DT>(u);
                    }
                }
                for (int j = 0; j < r; j++) {
                    const float b = lo_f32<DT>((uint32_t)bt[(size_t)c * r + j]);
#pragma unroll
                    for (int k = 0; k < G; k++) o[k] = fmaf(s_v[k][j], b, o[k]);
                }
#pragma unroll
                for (int k = 0; k < G; k++)
                    if (tok[k] >= 0) y[(size_t)tok[k] * hout + c] = (uint16_t)cvt16<DT>(o[k]);
            }
        }
    }
}

// Workgroups that share the output columns of an item: each repeats the shrink (the A rows come from L2, the items of a
// record run on one XCD) and takes a quarter or half of the expand, while all of them fit the device at once.  A unit pulls
// 256 KiB of an item's rows in about 4.5 us, so fewer bytes a unit is what shortens the launch.  Attention projections of
// Llama-7B in a graph, 1 / 2 / 4 / 8 workgroups an item, us a call: rank 16, one token 6.2 / 5.3 / 5.3 / 5.4, 32 tokens x 1 projection
// 8.6 / 7.2 / 6.6 / 6.7 (two launches 7.5), 16 x 3 9.3 / 7.8 / 7.2 / 11.7 (384 workgroups), 32 x 3 9.4 / 8.0 / 12.7 (384) / 17.7;
// rank 8, 8 x 4 7.1 / 6.1 / 6.2 / 6.3.
// Not where y lies over x: a workgroup that has stored its columns would have changed what the others of the item still read.
static int column_part_shift(const BgmvArgs &a)
{
    int widest = 0, shift = 0;
    for (int q = 0; q < a.n_proj; q++)
        for (int k = 0; k < a.n_proj; k++) {
            const uintptr_t y = (uintptr_t)a.y[q], x = (uintptr_t)a.x[k];
            if (y < x + (uintptr_t)a.T * a.hin[k] * 2 && x < y + (uintptr_t)a.T * a.hout[q] * 2) return 0;
        }
    for (int q = 0; q < a.n_proj; q++) widest = a.hout[q] > widest ? a.hout[q] : widest;
    while (shift < 2 && (2LL << shift) * a.n_proj * a.items_cap <= device_compute_units() && (2 << shift) * 512 <= widest) shift++;
    return shift;
}

template <int DT, int G, int RMAX, bool BT, bool WORK>
static int launch_one(const BgmvArgs &a0, hipStream_t s)
{
    BgmvArgs a = a0;
    a.part_shift = WORK ? column_part_shift(a) : 0;
    // Work items of one or two tokens are the small-batch form: a launch of at most about one
    // workgroup per CU, bound by the chain launch -> record -> page table -> rows -> y.  Twice the
    // threads halve the shrink's load rounds and the early expand requests overlap the reduction
    // (8.5 vs 9.9 us per call at 64 tokens, 10.8 vs 13.2 us at 128, three projections; before the requests moved ahead of
    // the shrink and items were shared).
    constexpr bool WIDE = WORK && !BT && G <= 2;
    constexpr int NT = WIDE ? 512 : 256;
    const long long per_proj = WORK ? a.items_cap : a.T;
    if (per_proj <= 0 || a.n_proj <= 0) return 0;
    if ((per_proj * a.n_proj << a.part_shift) > 0x7fffffffLL) return (int)hipErrorInvalidValue;
    // The id in three parts, in the same order as one flat id: two divisions by numbers of the arguments (and one by the parts)
    // at the head of the chain of loads cost 0.15 us a launch (1 token x 1 projection 5.39 -> 5.23, 32 x 3 7.97 -> 7.82).
    const dim3 grid((unsigned)per_proj, (unsigned)a.n_proj, 1u << a.part_shift);
    // Early expand requests pay for their registers when a work item carries several tokens, or when
    // the launch is latency-bound anyway.
    constexpr bool PF = WORK && !BT && (G >= 4 || WIDE);
    hipLaunchKernelGGL((bgmv_kernel<DT, G, RMAX, NT, BT, WORK, PF>), grid, dim3(NT), 0, s, a);
    return (int)hipGetLastError();
}

template <int DT, int RMAX>
static int launch_work(const BgmvArgs &a, int group, hipStream_t s)
{
    switch (group) {
    case 1: return launch_one<DT, 1, RMAX, false, true>(a, s);
    case 2: return launch_one<DT, 2, RMAX, false, true>(a, s);
    case 4: return launch_one<DT, 4, RMAX, false, true>(a, s);
    case 8:
        if constexpr (RMAX <= 32) return launch_one<DT, 8, RMAX, false, true>(a, s);
        else return (int)hipErrorInvalidValue;
    default: return (int)hipErrorInvalidValue;
    }
}

template <int DT>
static int launch_dt(const BgmvArgs &a, int group, int max_rank, bool bt, hipStream_t s)
{
    if (a.work) {
        if (bt) return (int)hipErrorInvalidValue;
        if (max_rank <= 16) return launch_work<DT, 16>(a, group, s);
        if (max_rank <= 32) return launch_work<DT, 32>(a, group, s);
        return launch_work<DT, 64>(a, group, s);
    }
    if (group != 1) return (int)hipErrorInvalidValue;      // the plain form is one token per work item
    if (bt) {
        if (max_rank <= 16) return launch_one<DT, 1, 16, true, false>(a, s);
        if (max_rank <= 32) return launch_one<DT, 1, 32, true, false>(a, s);
        return launch_one<DT, 1, 64, true, false>(a, s);
    }
    if (max_rank <= 16) return launch_one<DT, 1, 16, false, false>(a, s);
    if (max_rank <= 32) return launch_one<DT, 1, 32, false, false>(a, s);
    return launch_one<DT, 1, 64, false, false>(a, s);
}

int launch_bgmv(const BgmvArgs &a, int dtype, int group, int max_rank, bool b_transposed, hipStream_t s)
{
    if (dtype == DT_F16) return launch_dt<DT_F16>(a, group, max_rank, b_transposed, s);
    return launch_dt<DT_BF16>(a, group, max_rank, b_transposed, s);
}

}  // namespace mlora
