"""GPU parity: base projection + LoRA in one pass (MFMA GEMM with the expand riding along) through the C ABI,
against the fp32-accumulated oracle (rtol 1e-2 / atol 1e-3), bit-exact on integer-valued inputs, and against
the library GEMM followed by the SGMV kernels at full config-4 width."""
import zlib

import numpy as np
import pytest
import torch

from gpu_common import ATOL, RTOL, assert_close_bits, say, tdtype, upload_pool
from helpers import BF16, FP16, PagedPool, bits_of, bits_to_torch, f32_of, torch_to_bits
from mlora import AdapterPool, gemm_lora, plan_prefill, sgmv_multi
from oracle import oracle as orc

pytestmark = pytest.mark.gpu


def _oracle(pp, x, w, tok, **kw):
    return orc.gemm_lora_paged(x, w, pp.a_rows, pp.b_rows, tok, pp.page_tbl, pp.page_tbl, pp.ranks, pp.scaling,
                               pp.page_rows, pp.dtype, **kw)


def _layout(lens, gaps, adapters):
    """Segments laid out one after another with `gaps[i]` adapter-less tokens before segment i."""
    start, pos = [], 0
    for l, g in zip(lens, gaps):
        pos += g
        start.append(pos)
        pos += l
    return np.asarray(start, np.int32), np.asarray(lens, np.int32), np.asarray(adapters, np.int32), pos


def _tok_of(start, lens, adapters, T):
    tok = np.full(T, -1, np.int32)
    for s, l, a in zip(start, lens, adapters):
        tok[s:s + l] = a
    return tok


def _run(pp, x_bits, w_bits, seg, T, aligned=False):
    pool = upload_pool(pp)
    x = bits_to_torch(x_bits, pp.dtype, "cuda")
    w = bits_to_torch(w_bits, pp.dtype, "cuda")
    y = torch.full((T, pp.hout), float("nan"), dtype=tdtype(pp.dtype), device="cuda")
    ss, sl, sa = (torch.from_numpy(a).cuda() for a in seg)
    plan = plan_prefill(ss, sl, sa, T, pool, aligned=aligned)
    gemm_lora([y], [x], [w], pool, 0, ["p"], plan)
    torch.cuda.synchronize()
    return torch_to_bits(y)


CASES = [
    # name, segment lengths, gaps before them, tail tokens, pool ranks, hin, hout, dtype
    ("q slice 1024x1024 fp16 r16", [70, 128, 1, 57], [0, 0, 0, 0], 0, [16] * 4, 1024, 1024, FP16),
    ("bf16 r64, K tail 1032x520, gaps", [37, 44, 51, 64, 100], [3, 0, 5, 0, 1], 7, [64, 24, 8], 1032, 520, BF16),
    ("rank 32 pool, ragged N 512x776", [64, 64, 64, 9], [0, 0, 0, 0], 0, [32, 17, 32], 512, 776, FP16),
    ("one K step and a tail 72x72", [5], [0], 0, [8], 72, 72, BF16),
    ("tail only 40x264", [30, 3], [2, 0], 1, [16, 4], 40, 264, FP16),
    ("three row tiles 640x256", [300, 250, 130], [0, 20, 0], 0, [16, 16], 640, 256, FP16),
]


@pytest.mark.parametrize("name,lens,gaps,tail,ranks,hin,hout,dtype", CASES, ids=[c[0] for c in CASES])
def test_gemm_lora_vs_oracle(name, lens, gaps, tail, ranks, hin, hout, dtype):
    rng = np.random.default_rng(zlib.crc32(name.encode()))
    pp = PagedPool(rng, ranks, hin, hout, page_rows=8, dtype=dtype)
    adapters = rng.integers(0, len(ranks), len(lens))
    if len(lens) > 2:
        adapters[1] = -1                                   # a segment without adapter: base product only
    ss, sl, sa, T = _layout(lens, gaps, adapters)
    T += tail
    tok = _tok_of(ss, sl, sa, T)
    x = bits_of(rng.standard_normal((T, hin)).astype(np.float32), dtype)
    w = bits_of((rng.standard_normal((hin, hout)) / np.sqrt(hin)).astype(np.float32), dtype)
    say(f"gemm_lora {name}")
    got = _run(pp, x, w, (ss, sl, sa), T)
    assert_close_bits(got, _oracle(pp, x, w, tok), dtype, name)
    say(f"gemm_lora {name}, tiles cut at multiples of 64")
    assert_close_bits(_run(pp, x, w, (ss, sl, sa), T, aligned=True), _oracle(pp, x, w, tok), dtype, name + " aligned")
    # much closer than the tolerance: within one 16-bit ulp of the fp64 result (+ fp32 accumulation noise)
    want64 = f32_of(_oracle(pp, x, w, tok, acc64=True), dtype).astype(np.float64)
    err = np.abs(f32_of(got, dtype) - want64)
    mant = 10 if dtype == FP16 else 7
    assert np.all(err <= 2.0 ** -mant * np.abs(want64) + 2e-5), "not within one ulp of the exact result"


def test_gemm_lora_integer_inputs_bit_exact():
    rng = np.random.default_rng(81)
    ranks = [8, 16, 3, 64, 5]
    pp = PagedPool(rng, ranks, hin=512, hout=384, page_rows=8, dtype=FP16, integer=True)
    pp.scaling[:] = [1, 2, 0.5, -1, 4]
    lens, gaps = [33, 64, 65, 1, 130], [0, 2, 0, 0, 4]
    ss, sl, sa, T = _layout(lens, gaps, [4, 0, 1, 3, 2])
    tok = _tok_of(ss, sl, sa, T)
    xi = (rng.integers(-2, 3, (T, 512)) * (rng.random((T, 512)) < 0.05)).astype(np.float32)
    wi = (rng.integers(-1, 2, (512, 384)) * (rng.random((512, 384)) < 0.5)).astype(np.float32)
    x, w = bits_of(xi, FP16), bits_of(wi, FP16)
    want = _oracle(pp, x, w, tok)
    assert np.abs(f32_of(want, FP16)).max() < 2048
    say("gemm_lora integer-valued inputs")
    assert np.array_equal(_run(pp, x, w, (ss, sl, sa), T), want)
    assert np.array_equal(_run(pp, x, w, (ss, sl, sa), T, aligned=True), want)


@pytest.mark.parametrize("dtype", [FP16, BF16])
def test_gemm_base_only_matches_library_product(dtype):
    """No plan: the base products alone, against torch.mm in fp32 on the same 16-bit inputs."""
    torch.manual_seed(5)
    td = tdtype(dtype)
    T, hin, hout = 333, 1096, 840
    x = torch.randn(T, hin, device="cuda").to(td)
    w = (torch.randn(hin, hout, device="cuda") / hin ** 0.5).to(td)
    y = torch.full((T, hout), float("nan"), dtype=td, device="cuda")
    say(f"gemm base only {td}")
    gemm_lora([y], [x], [w], None, 0, ["p"], None)
    want = (x.float() @ w.float())
    err = (y.float() - want).abs()
    assert bool((err <= ATOL + RTOL * want.abs()).all())
    assert bool((err <= 2.0 ** (-10 if dtype == FP16 else -7) * want.abs() + 2e-5).all())


def test_gemm_lora_three_projections_one_launch():
    """q, k (same x) and a wider projection with its own x in one call, each against the oracle."""
    rng = np.random.default_rng(83)
    dims = {"q": (512, 512), "k": (512, 256), "g": (768, 1376)}
    ranks = [16, 8, 32]
    pps = {p: PagedPool(np.random.default_rng(90), ranks, hin, hout, page_rows=8, dtype=FP16) for p, (hin, hout) in dims.items()}
    first = pps["q"]
    pool = AdapterPool(1, dims, first.n, first.n_pages, page_rows=8, max_rank=32, dtype=torch.float16, device="cuda")
    pool.h_page_tbl[:] = first.page_tbl
    pool.h_rank[:] = first.ranks
    pool.h_scaling[:] = first.scaling
    pool._dirty = True
    pool.sync()
    for p, pp in pps.items():
        assert np.array_equal(pp.page_tbl, first.page_tbl)
        pool.a_rows[p][0].copy_(bits_to_torch(pp.a_rows, FP16))
        pool.b_rows[p][0].copy_(bits_to_torch(pp.b_rows, FP16))
    ss, sl, sa, T = _layout([100, 64, 200], [0, 3, 0], [2, 0, 1])
    tok = _tok_of(ss, sl, sa, T)
    xb = {512: bits_of(rng.standard_normal((T, 512)).astype(np.float32), FP16),
          768: bits_of(rng.standard_normal((T, 768)).astype(np.float32), FP16)}
    xt = {k: bits_to_torch(v, FP16, "cuda") for k, v in xb.items()}
    wb = {p: bits_of((rng.standard_normal(d) / np.sqrt(d[0])).astype(np.float32), FP16) for p, d in dims.items()}
    ws = [bits_to_torch(wb[p], FP16, "cuda") for p in dims]
    ys = [torch.full((T, d[1]), float("nan"), dtype=torch.float16, device="cuda") for d in dims.values()]
    plan = plan_prefill(*(torch.from_numpy(a).cuda() for a in (ss, sl, sa)), T, pool, n_proj=3)
    say("gemm_lora three projections")
    gemm_lora(ys, [xt[d[0]] for d in dims.values()], ws, pool, 0, list(dims), plan)
    torch.cuda.synchronize()
    for i, (p, d) in enumerate(dims.items()):
        assert_close_bits(torch_to_bits(ys[i]), _oracle(pps[p], xb[d[0]], wb[p], tok), FP16, p)


def test_gemm_lora_config4_width_against_library_products():
    """Full config-4 attention width (5120 x 5120, rank 64, bf16, 2048 tokens): the one-pass result against
    fp32 library products of the same 16-bit operands, within the tolerance; and the SGMV kernels' delta added
    to the base-only result reproduces it to the roundings involved."""
    torch.manual_seed(7)
    T, H, r, n_seg = 2048, 5120, 64, 8
    pool = AdapterPool(1, {"q": (H, H)}, n_seg, n_seg * 8 + 2, page_rows=8, max_rank=64, dtype=torch.bfloat16, device="cuda")
    AB = []
    for a in range(n_seg):
        pool.allocate(a, r, 0.5)
        AB.append(((torch.randn(H, r) * 0.02).bfloat16(), (torch.randn(r, H) * 0.02).bfloat16()))
        pool.load(a, 0, "q", *AB[-1])
    x = torch.randn(T, H, device="cuda").bfloat16()
    w = (torch.randn(H, H, device="cuda") / H ** 0.5).bfloat16()
    L = T // n_seg
    ss = torch.arange(0, T, L, dtype=torch.int32, device="cuda")
    sl = torch.full((n_seg,), L, dtype=torch.int32, device="cuda")
    sa = torch.arange(n_seg, dtype=torch.int32, device="cuda")
    plan = plan_prefill(ss, sl, sa, T, pool)
    y = torch.full((T, H), float("nan"), dtype=torch.bfloat16, device="cuda")
    say("gemm_lora config-4 width, one pass")
    gemm_lora([y], [x], [w], pool, 0, ["q"], plan)
    ref = torch.mm(x.float(), w.float())
    for a in range(n_seg):
        A, B = (m.cuda().float() for m in AB[a])
        ref[a * L:(a + 1) * L] += 0.5 * ((x[a * L:(a + 1) * L].float() @ A) @ B)
    torch.cuda.synchronize()
    assert bool(torch.isfinite(y.float()).all())
    err = (y.float() - ref).abs()
    assert bool((err <= ATOL + RTOL * ref.abs()).all()), float(err.max())
    assert bool((err <= 2.0 ** -8 * ref.abs() + 1e-4).all()), "not within one bf16 ulp of the fp32 reference"
    say("base only + sgmv delta")
    yb = torch.empty_like(y)
    gemm_lora([yb], [x], [w], None, 0, ["q"], None)
    delta = torch.empty_like(y)
    sgmv_multi([delta], [x], pool, 0, ["q"], plan, accumulate=False)
    torch.cuda.synchronize()
    assert float(delta.float().abs().max()) > 0.05                      # the delta is not negligible here
    # three bf16 roundings (y, base, delta) apart at most
    assert bool(((y.float() - yb.float() - delta.float()).abs() <= 2.0 ** -7 * (ref.abs() + delta.float().abs()) + 1e-4).all())


@pytest.mark.parametrize("aligned", [False, True])
def test_plan_tile_list_matches_oracle(aligned):
    """The tile list the plan kernel writes (first words of the workspace: segment, first token and token count
    per tile, then the count) is the oracle's, bit for bit, in both cutting modes; and SGMV gives the same
    result with either plan."""
    rng = np.random.default_rng(91)
    lens = rng.integers(0, 300, 37).astype(np.int32)
    gaps = (rng.integers(0, 2, 37) * rng.integers(0, 50, 37)).astype(np.int32)
    ss, sl, sa, T = _layout(lens, gaps, rng.integers(-1, 3, 37))
    T += 5
    pp = PagedPool(rng, [16, 8, 4], 64, 64, page_rows=8, dtype=FP16)
    pool = upload_pool(pp)
    say(f"plan tile list aligned={aligned}")
    plan = plan_prefill(*(torch.from_numpy(a).cuda() for a in (ss, sl, sa)), T, pool, aligned=aligned)
    torch.cuda.synchronize()
    want_s, want_t0, want_n = orc.sgmv_plan(ss, sl, 64, aligned=aligned)
    max_tiles = T // 64 + 2 * len(lens) + 1
    words = plan.workspace[:(3 * max_tiles + 1) * 4].cpu().numpy().view(np.int32)
    n = int(words[3 * max_tiles])
    assert n == len(want_s)
    assert np.array_equal(words[:n], want_s)
    assert np.array_equal(words[max_tiles:max_tiles + n], want_t0)
    assert np.array_equal(words[2 * max_tiles:2 * max_tiles + n], want_n)


@pytest.mark.parametrize("T,hin,hout,n_proj,ranks,dtype,splits", [
    (1, 2056, 264, 1, [64, 8], FP16, 8),          # one row of a 64-row tile, uneven K ranges and a partial last step
    (64, 2088, 4104, 3, [16, 8], BF16, 3),        # a full 64-row tile, a column tile of eight columns
    (65, 2056, 4096, 3, [64, 24], FP16, 4),       # 128-row tiles, one row in the upper half's first block
    (128, 3080, 4096, 3, [32, 17], BF16, 2),      # two full 64-row tiles
    (128, 3592, 4104, 3, [32, 17], BF16, 4),      # a full 128-row tile
    (129, 4104, 4096, 3, [32, 16], FP16, 4),      # 192-row tiles, one row in the third block
    (192, 4096, 4352, 3, [64, 40], BF16, 4),
    (351, 4104, 1288, 7, [16, 8], FP16, 2),       # three tiles of 128 rows, the last with a ragged end
])
def test_gemm_lora_short_batches(T, hin, hout, n_proj, ranks, dtype, splits):
    """Tiles of 64 to 192 rows with K cut into ranges: the rows at the tiles' edges against the oracle, every projection
    alike, and the same result as the call without room for partial sums up to the last rounding."""
    from mlora import _ext
    import ctypes as C
    rng = np.random.default_rng(T * 7 + hin)
    pp = PagedPool(rng, ranks, hin, hout, page_rows=8, dtype=dtype)
    names = [f"p{i}" for i in range(n_proj)]
    pool = upload_pool(pp, projections={nm: (hin, hout) for nm in names})
    for nm in names:
        pool.a_rows[nm][0].copy_(bits_to_torch(pp.a_rows, dtype))
        pool.b_rows[nm][0].copy_(bits_to_torch(pp.b_rows, dtype))
    cut = max(1, T // 3)
    lens = [cut] + ([T - cut] if T > cut else [])
    ss, sl, sa, _ = _layout(lens, [0] * len(lens), [0, 1][:len(lens)])
    tok = _tok_of(ss, sl, sa, T)
    x = bits_of(rng.standard_normal((T, hin)).astype(np.float32), dtype)
    w = bits_of((rng.standard_normal((hin, hout)) / np.sqrt(hin)).astype(np.float32), dtype)
    xt, wt = bits_to_torch(x, dtype, "cuda"), bits_to_torch(w, dtype, "cuda")
    arr = [(C.c_int32 * 8)(*([v] * n_proj)) for v in (hin, hout)]
    assert _ext.lib().mlora_gemm_lora_partial_bytes(n_proj, *arr, T) == splits * n_proj * T * hout * 4          # K ranges
    plan = plan_prefill(*(torch.from_numpy(a).cuda() for a in (ss, sl, sa)), T, pool, n_proj=n_proj)
    ys = [torch.full((T, hout), float("nan"), dtype=tdtype(dtype), device="cuda") for _ in names]
    say(f"gemm_lora short T={T} {hin}x{hout} n_proj={n_proj} ranks={ranks} dtype={dtype}")
    gemm_lora(ys, [xt] * n_proj, [wt] * n_proj, pool, 0, names, plan)
    torch.cuda.synchronize()
    got = torch_to_bits(ys[0])
    rows = np.unique(np.clip([0, cut - 1, cut, 31, 32, 63, 64, 65, 127, 128, 191, 192, T - 2, T - 1], 0, T - 1))
    assert_close_bits(got[rows], _oracle(pp, x[rows], w, tok[rows]), dtype, "rows at the edges")
    for y in ys[1:]:
        assert torch.equal(y, ys[0])
    # without room for partial sums: K whole, the same products summed in another order.  Both round one fp32 sum to 16
    # bits; sums differ by no more than hin roundings of 2^-24 of their terms' size, about one, so by less than 1e-3 at
    # these widths, and the results by that and one rounding step.
    ptr = lambda ts: (C.c_void_p * 8)(*[t.data_ptr() for t in ts])
    whole = [torch.empty_like(y) for y in ys]
    rc = _ext.lib().mlora_gemm_lora_planned(
        n_proj, ptr(whole), ptr([xt] * n_proj), ptr([wt] * n_proj), ptr([pool.a_rows[nm][0] for nm in names]),
        ptr([pool.b_rows[nm][0] for nm in names]), *arr, plan.seg_start.data_ptr(), plan.seg_len.data_ptr(),
        plan.seg_adapter.data_ptr(), len(lens), pool.page_tbl.data_ptr(), pool.rank.data_ptr(), pool.scaling.data_ptr(), T,
        pool.n_slots, pool.max_pages, pool.page_rows, pool.n_pages, pool.max_rank, pool.dtype_code,
        plan.workspace.data_ptr(), plan.workspace.numel(), _ext.current_stream_ptr())
    _ext.check(rc)
    torch.cuda.synchronize()
    ulp = 2.0 ** (-10 if dtype == FP16 else -7)
    for y in whole:
        a, b = y.double(), ys[0].double()
        assert bool(((a - b).abs() <= ulp * b.abs() + 1e-3).all())


@pytest.mark.parametrize("T,hins,houts,splits,ranks,dtype", [
    # K ranges per projection, as the rule chooses them: cut and whole projections in one launch, the cut ones ...
    (100, [4096, 512, 4104, 320, 2048], [264, 520, 256, 768, 512], [8, 1, 8, 1, 4], [16, 5], FP16),      # first, in the middle and last
    (200, [352, 4104, 512, 2080, 416], [512, 264, 1032, 520, 768], [1, 8, 1, 4, 1], [64, 24], BF16),     # between whole ones
    (260, [4104, 4096, 1024], [4096, 4096, 4104], [3, 3, 1], [32, 8], FP16),                             # two tiles of 192 rows
])
def test_gemm_lora_short_batches_of_unlike_projections(T, hins, houts, splits, ranks, dtype):
    """Projections of other widths, each with its own number of K ranges: the room of the cut ones side by side, the sum
    launch over them alone, the whole ones written by the product itself."""
    from mlora import _ext
    import ctypes as C
    n = len(hins)
    names = [f"p{i}" for i in range(n)]
    pps = [PagedPool(np.random.default_rng(31), ranks, hi, ho, page_rows=8, dtype=dtype) for hi, ho in zip(hins, houts)]
    pool = upload_pool(pps[0], projections={nm: (hi, ho) for nm, hi, ho in zip(names, hins, houts)})
    rng = np.random.default_rng(T)
    xs, ws = [], []
    for nm, pp in zip(names, pps):
        pool.a_rows[nm][0].copy_(bits_to_torch(pp.a_rows, dtype))
        pool.b_rows[nm][0].copy_(bits_to_torch(pp.b_rows, dtype))
        xs.append(bits_of(rng.standard_normal((T, pp.hin)).astype(np.float32), dtype))
        ws.append(bits_of((rng.standard_normal((pp.hin, pp.hout)) / np.sqrt(pp.hin)).astype(np.float32), dtype))
    arr = [(C.c_int32 * 8)(*v) for v in (hins, houts)]
    room = sum(s * T * ho * 4 for s, ho in zip(splits, houts) if s > 1)
    assert _ext.lib().mlora_gemm_lora_partial_bytes(n, *arr, T) == room
    ss, sl, sa, _ = _layout([T // 3, T - T // 3 - 7], [0, 7], [0, 1])
    tok = _tok_of(ss, sl, sa, T)
    plan = plan_prefill(*(torch.from_numpy(a).cuda() for a in (ss, sl, sa)), T, pool, n_proj=n)
    ys = [torch.full((T, ho), float("nan"), dtype=tdtype(dtype), device="cuda") for ho in houts]
    say(f"gemm_lora short T={T} {hins}x{houts} ranges={splits}")
    gemm_lora(ys, [bits_to_torch(x, dtype, "cuda") for x in xs], [bits_to_torch(w, dtype, "cuda") for w in ws], pool, 0, names, plan)
    torch.cuda.synchronize()
    rows = np.unique(np.clip([0, T // 3 - 1, T // 3, T // 3 + 6, T // 3 + 7, 63, 64, 127, 128, 191, 192, T - 1], 0, T - 1))
    for nm, pp, x, w, y in zip(names, pps, xs, ws, ys):
        assert bool(torch.isfinite(y).all())
        assert_close_bits(torch_to_bits(y)[rows], _oracle(pp, x[rows], w, tok[rows]), dtype, nm)
