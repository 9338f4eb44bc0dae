"""GPU parity: SGMV prefill kernels (MFMA) through the C ABI against the fp32-accumulated oracle, and
against the decode kernel at full config-4 size."""
import numpy as np
import pytest
import torch

from gpu_common import ATOL, RTOL, assert_close_bits, oracle_apply, say, tdtype, upload_pool
from helpers import (BF16, FP16, PagedPool, bits_of, bits_to_torch, f32_of, sgmv_shape, torch_to_bits,
                     workspace_for_splits)
from mlora import bgmv, plan_prefill, sgmv

pytestmark = pytest.mark.gpu


def _assert_shape(want, widths, inputs, T, n_seg, max_rank):
    """The case is the one it is meant to be: the accumulating call takes the launches that `want` names."""
    got = sgmv_shape(widths, inputs, T, n_seg, max_rank)
    got["most"] = max(got["splits"])
    assert {k: got[k] for k in want} == want, got


def _segments(lens, adapters):
    lens = np.asarray(lens, np.int32)
    start = np.concatenate([[0], np.cumsum(lens)[:-1]]).astype(np.int32)
    return start, lens, np.asarray(adapters, np.int32)


def _tok_of(start, lens, adapters, T):
    tok = np.full(T, -1, np.int32)
    for s, l, a in zip(start, lens, adapters):
        tok[s:s + l] = a
    return tok


def _run(pp, x_bits, seg, y0_bits, accumulate=True):
    pool = upload_pool(pp)
    T = x_bits.shape[0]
    x = bits_to_torch(x_bits, pp.dtype, "cuda")
    y = bits_to_torch(y0_bits, pp.dtype, "cuda") if y0_bits is not None else \
        torch.full((T, pp.hout), float("nan"), dtype=tdtype(pp.dtype), device="cuda")
    ss, sl, sa = (torch.from_numpy(a).cuda() for a in seg)
    sgmv(y, x, pool, 0, "p", ss, sl, sa, accumulate=accumulate)
    torch.cuda.synchronize()
    return torch_to_bits(y)


CASES = [
    # name, segment lengths, ranks of the pool, hin, hout, dtype
    ("C4 slice q 5120x5120 bf16 r64", [70, 128, 1, 300, 64, 65], [64] * 8, 5120, 5120, BF16),
    ("C4 slice gate 5120x13824 bf16 r64", [130, 33], [64] * 4, 5120, 13824, BF16),
    ("C4 slice down 13824x5120 bf16 r64", [90, 17, 64], [64] * 4, 13824, 5120, BF16),
    ("fp16 hetero ranks 4096x4096", [40, 100, 7, 64, 129], [8, 16, 32, 64, 24], 4096, 4096, FP16),
    ("rank 16 pool 1024x2048", [63, 64, 65, 1], [16, 8, 16, 3], 1024, 2048, FP16),
    ("odd widths 200x72 bf16", [5, 70], [32, 5], 200, 72, BF16),
    ("tile boundaries 127/128/129 r32 2048x1024", [127, 128, 129, 63, 64, 65], [32, 32, 16, 32], 2048, 1024, FP16),
]


@pytest.mark.parametrize("name,lens,ranks,hin,hout,dtype", CASES, ids=[c[0] for c in CASES])
def test_sgmv_vs_oracle(name, lens, ranks, hin, hout, dtype):
    import zlib
    rng = np.random.default_rng(zlib.crc32(name.encode()))
    pp = PagedPool(rng, ranks, hin, hout, page_rows=8, dtype=dtype)
    adapters = rng.integers(0, len(ranks), len(lens))
    seg = _segments(lens, adapters)
    T = int(np.sum(lens))
    tok = _tok_of(*seg, T)
    x = bits_of(rng.standard_normal((T, hin)).astype(np.float32), dtype)
    y0 = bits_of(rng.standard_normal((T, hout)).astype(np.float32), dtype)
    say(f"sgmv {name} accumulate")
    got = _run(pp, x, seg, y0)
    assert_close_bits(got, oracle_apply(pp, x, tok, y0), dtype, name)
    say(f"sgmv {name} delta")
    got_d = _run(pp, x, seg, None, accumulate=False)
    want_d = oracle_apply(pp, x, tok, None)
    assert_close_bits(got_d, want_d, dtype, name + " delta")
    # the hi+lo split keeps the intermediate at fp32 accuracy: the delta is much closer to the
    # fp64-accumulated oracle than a 16-bit intermediate would allow
    want64 = f32_of(oracle_apply(pp, x, tok, None, acc64=True), dtype).astype(np.float64)
    err = np.abs(f32_of(got_d, dtype) - want64)
    mant = 10 if dtype == FP16 else 7
    assert np.all(err <= 2.0 ** -mant * np.abs(want64) + 1e-5), "delta is not within one ulp of the exact result"


def test_sgmv_integer_inputs_bit_exact():
    rng = np.random.default_rng(71)
    ranks = [8, 16, 3, 64, 5]
    pp = PagedPool(rng, ranks, hin=512, hout=384, page_rows=8, dtype=FP16, integer=True)
    pp.scaling[:] = [1, 2, 0.5, -1, 4]
    lens = [64, 3, 100, 65, 1]
    seg = _segments(lens, [3, 0, 1, 2, 4])
    T = sum(lens)
    tok = _tok_of(*seg, T)
    xi = (rng.integers(-2, 3, (T, 512)) * (rng.random((T, 512)) < 0.05)).astype(np.float32)
    y0 = bits_of(rng.integers(-8, 9, (T, 384)).astype(np.float32), FP16)
    x = bits_of(xi, FP16)
    want = oracle_apply(pp, x, tok, y0)
    assert np.abs(f32_of(want, FP16)).max() < 2048
    say("sgmv integer-valued inputs")
    assert np.array_equal(_run(pp, x, seg, y0), want)


def test_sgmv_segments_without_adapter_and_gaps():
    rng = np.random.default_rng(72)
    pp = PagedPool(rng, [16, 32], 256, 256, page_rows=8, dtype=FP16)
    # tokens 0..9 uncovered, then a segment with no adapter, an empty one, and two real ones
    ss = np.array([10, 40, 40, 104], np.int32)
    sl = np.array([30, 0, 64, 20], np.int32)
    sa = np.array([-1, 1, 0, 1], np.int32)
    T = 130
    tok = _tok_of(ss, sl, sa, T)
    x = bits_of(rng.standard_normal((T, 256)).astype(np.float32), FP16)
    y0 = bits_of(rng.standard_normal((T, 256)).astype(np.float32), FP16)
    say("sgmv gaps / adapter-less segment, accumulate")
    got = _run(pp, x, (ss, sl, sa), y0)
    assert np.array_equal(got[tok < 0], y0[tok < 0])
    assert_close_bits(got, oracle_apply(pp, x, tok, y0), FP16)
    say("sgmv gaps / adapter-less segment, delta")
    got_d = _run(pp, x, (ss, sl, sa), None, accumulate=False)
    assert np.all(got_d[10:40] == 0)                       # adapter-less segment is defined as zeros
    assert np.all(got_d[tok < 0] == 0)                     # ... and so are tokens 0..9 and 124..129, which no segment covers
    assert_close_bits(got_d, oracle_apply(pp, x, tok, None), FP16)


def test_sgmv_delta_defines_rows_outside_every_segment():
    """y = delta mode over NaN-filled memory: rows between, before and after the segments (given out of
    order) come back as zeros from the one-projection, the planned and the multi-projection calls."""
    from mlora import plan_prefill, sgmv, sgmv_multi
    rng = np.random.default_rng(75)
    hin, hout = 256, 392
    pp = PagedPool(rng, [8, 64, 24], hin, hout, page_rows=8, dtype=BF16)
    ss = np.array([200, 5, 70], np.int32)                  # gaps: 0..4, 69, 135..199, 263..299
    sl = np.array([63, 64, 65], np.int32)
    sa = np.array([2, 0, 1], np.int32)
    T = 300
    tok = _tok_of(ss, sl, sa, T)
    x = bits_of(rng.standard_normal((T, hin)).astype(np.float32), BF16)
    want = oracle_apply(pp, x, tok, None)
    assert np.all(want[tok < 0] == 0) and (tok < 0).sum() == 108
    say("sgmv delta with gaps: self-planning call")
    got = _run(pp, x, (ss, sl, sa), None, accumulate=False)
    assert np.all(got[tok < 0] == 0)
    assert_close_bits(got, want, BF16)
    pool = upload_pool(pp)
    seg = tuple(torch.from_numpy(a).cuda() for a in (ss, sl, sa))
    xt = bits_to_torch(x, BF16, "cuda")
    plan = plan_prefill(*seg, T, pool, n_proj=2)
    nan = lambda: torch.full((T, hout), float("nan"), dtype=torch.bfloat16, device="cuda")
    say("sgmv delta with gaps: planned and multi-projection calls")
    y1, y2, y3 = nan(), nan(), nan()
    sgmv(y1, xt, pool, 0, "p", accumulate=False, plan=plan)
    sgmv_multi([y2, y3], [xt, xt], pool, 0, ["p", "p"], plan, accumulate=False)
    torch.cuda.synchronize()
    for y in (y1, y2, y3):
        bits = torch_to_bits(y)
        assert np.all(bits[tok < 0] == 0)
        assert_close_bits(bits, want, BF16)


def test_sgmv_plan_once_apply_many():
    """One plan serves several projections and layers, and matches the self-planning call bit for bit."""
    rng = np.random.default_rng(73)
    ranks = [64, 16, 32, 8]
    hin, hout = 512, 768
    pp = PagedPool(rng, ranks, hin, hout, page_rows=8, dtype=BF16)
    from mlora import AdapterPool
    pool = upload_pool(pp, projections={"p": (hin, hout), "o": (hout, hin)}, n_layers=2)
    for l in range(2):
        pool.a_rows["o"][l].normal_(0, 0.02)
        pool.b_rows["o"][l].normal_(0, 0.02)
    pool.a_rows["p"][1].normal_(0, 0.02)
    pool.b_rows["p"][1].normal_(0, 0.02)
    lens = [70, 3, 128, 65]
    ss, sl, sa = (torch.from_numpy(a).cuda() for a in _segments(lens, [2, 0, 3, 1]))
    T = sum(lens)
    say("sgmv: one plan, two layers x two projections")
    plan = plan_prefill(ss, sl, sa, T, pool)
    for l in range(2):
        for proj, (hi, ho) in (("p", (hin, hout)), ("o", (hout, hin))):
            x = torch.randn(T, hi, device="cuda").bfloat16()
            y0 = torch.randn(T, ho, device="cuda").bfloat16()
            y_plan, y_self = y0.clone(), y0.clone()
            sgmv(y_plan, x, pool, l, proj, plan=plan)
            sgmv(y_self, x, pool, l, proj, ss, sl, sa)
            torch.cuda.synchronize()
            assert torch.equal(y_plan, y_self)
            assert not torch.equal(y_plan, y0)


def test_sgmv_equals_bgmv_at_config4_size():
    """Config 4 at full size (16 requests, lengths U[128,1024], 32 rank-64 adapters, hidden 5120, bf16):
    the prefill kernels and the decode kernel must agree within tolerance on every token."""
    rng = np.random.default_rng(1004)
    lens = rng.integers(128, 1025, 16)
    adapters = rng.integers(0, 32, 16)
    seg = _segments(lens, adapters)
    T = int(lens.sum())
    pp = PagedPool(rng, [64] * 32, 5120, 5120, page_rows=8, dtype=BF16)
    pool = upload_pool(pp)
    x = (torch.randn(T, 5120, device="cuda")).to(torch.bfloat16)
    y0 = (torch.randn(T, 5120, device="cuda")).to(torch.bfloat16)
    tok = torch.from_numpy(_tok_of(*seg, T)).cuda()
    ys, yb = y0.clone(), y0.clone()
    say(f"sgmv vs bgmv at config-4 size T={T}")
    sgmv(ys, x, pool, 0, "p", *(torch.from_numpy(a).cuda() for a in seg))
    bgmv([yb], [x], pool, 0, ["p"], tok)
    torch.cuda.synchronize()
    assert torch.allclose(ys.float(), yb.float(), rtol=RTOL, atol=ATOL)
    # linearity of the delta in x at full size
    d1, d2 = torch.zeros_like(y0), torch.zeros_like(y0)
    sgmv(d1, x, pool, 0, "p", *(torch.from_numpy(a).cuda() for a in seg), accumulate=False)
    sgmv(d2, (2 * x).contiguous(), pool, 0, "p", *(torch.from_numpy(a).cuda() for a in seg), accumulate=False)
    torch.cuda.synchronize()
    assert torch.equal(d2, 2 * d1)


def test_sgmv_multi_projection_call():
    """q, k, v (one x) and o (own x, other widths) in one call of three launches: every projection against the
    oracle, bit for bit on integer-valued inputs, and no effect on rows outside the segments."""
    from mlora import sgmv_multi
    rng = np.random.default_rng(74)
    ranks = [64, 16, 32, 8, 24]
    shapes = {"q": (512, 512), "k": (512, 256), "v": (512, 256), "o": (768, 512)}
    ss = np.array([5, 75, 78, 78, 206], np.int32)
    sl = np.array([70, 3, 0, 128, 65], np.int32)
    sa = np.array([2, 0, 1, 3, -1], np.int32)
    T = 280
    tok = _tok_of(ss, sl, sa, T)
    for integer in (False, True):
        pps = {p: PagedPool(np.random.default_rng(80), ranks, hin, hout, page_rows=8, dtype=FP16, integer=integer)
               for p, (hin, hout) in shapes.items()}
        for i, p in enumerate(shapes):                # same page table, different weights per projection
            r2 = np.random.default_rng(90 + i)
            if integer:
                pps[p].a_rows = bits_of(r2.integers(-2, 3, pps[p].a_rows.shape).astype(np.float32), FP16)
                pps[p].b_rows = bits_of(r2.integers(-2, 3, pps[p].b_rows.shape).astype(np.float32), FP16)
                pps[p].scaling[:] = [1, 2, 0.5, -1, 4]
            else:
                pps[p].a_rows = bits_of((r2.standard_normal(pps[p].a_rows.shape) * 0.02).astype(np.float32), FP16)
                pps[p].b_rows = bits_of((r2.standard_normal(pps[p].b_rows.shape) * 0.02).astype(np.float32), FP16)
        pool = upload_pool(pps["q"], projections=shapes)
        pool.h_scaling[:] = pps["q"].scaling
        pool._dirty = True
        for p in shapes:
            pool.a_rows[p][0].copy_(bits_to_torch(pps[p].a_rows, FP16))
            pool.b_rows[p][0].copy_(bits_to_torch(pps[p].b_rows, FP16))
        if integer:
            mk = lambda h: bits_of((rng.integers(-2, 3, (T, h)) * (rng.random((T, h)) < 0.04)).astype(np.float32), FP16)
            y0 = {p: bits_of(rng.integers(-8, 9, (T, shapes[p][1])).astype(np.float32), FP16) for p in shapes}
        else:
            mk = lambda h: bits_of(rng.standard_normal((T, h)).astype(np.float32), FP16)
            y0 = {p: bits_of(rng.standard_normal((T, shapes[p][1])).astype(np.float32), FP16) for p in shapes}
        x_qkv, x_o = mk(512), mk(768)
        xt_qkv, xt_o = bits_to_torch(x_qkv, FP16, "cuda"), bits_to_torch(x_o, FP16, "cuda")
        ys = {p: bits_to_torch(y0[p], FP16, "cuda") for p in shapes}
        d = [torch.from_numpy(a).cuda() for a in (ss, sl, sa)]
        plan = plan_prefill(d[0], d[1], d[2], T, pool, n_proj=4)
        say(f"sgmv_multi q,k,v,o integer={integer}")
        sgmv_multi([ys[p] for p in "qkvo"], [xt_qkv, xt_qkv, xt_qkv, xt_o], pool, 0, list("qkvo"), plan)
        torch.cuda.synchronize()
        for p in "qkvo":
            pps[p].scaling[:] = pps["q"].scaling
            want = oracle_apply(pps[p], x_o if p == "o" else x_qkv, tok, y0[p])
            got = torch_to_bits(ys[p])
            assert np.array_equal(got[tok < 0], y0[p][tok < 0])
            if integer:
                assert np.abs(f32_of(want, FP16)).max() < 2048
                assert np.array_equal(got, want), p
            else:
                assert_close_bits(got, want, FP16, f"projection {p}")
        # the same plan still serves single-projection calls
        y1 = bits_to_torch(y0["k"], FP16, "cuda")
        sgmv(y1, xt_qkv, pool, 0, "k", plan=plan)
        torch.cuda.synchronize()
        if integer:
            assert torch.equal(y1, ys["k"])
        else:
            assert torch.allclose(y1.float(), ys["k"].float(), rtol=RTOL, atol=ATOL)


@pytest.mark.parametrize("dtype", [FP16, BF16])
@pytest.mark.parametrize("lens,ranks,hin,hout,n_proj,shape", [
    ([1], [64], 4096, 640, 3, dict(share=0, few=1, most=8)),                # one tile, eight K splits, projections kept apart
    ([65, 3], [16, 32], 264, 1032, 3, dict(few=1, most=1)),                 # a short K; a width that ends inside a column block
    ([64] * 20 + [17], [33, 8], 4096, 128, 1, dict(few=1, most=8)),         # eight splits, one column block
    ([300, 150], [32, 24, 8], 1024, 2048, 7, dict(few=1, reduce=0, most=2)),    # the expand of 16-token pieces sums the splits
    ([300, 400], [32, 24, 8], 1096, 5128, 7, dict(few=0, reduce=0, most=2)),    # so does that of 64-token tiles
    ([64] * 25, [64], 512, 512, 2, dict(few=0, reduce=0, most=1)),          # 76 tiles at most: the numbering in runs
    ([64] * 30, [16], 384, 256, 3, dict(share=1, few=1)),                   # projections that share x in one workgroup
])
def test_sgmv_launch_shapes(lens, ranks, hin, hout, n_proj, shape, dtype):
    """Both sides of the size rules of the prefill launches: K splits, column blocks, numbering of the workgroups,
    shared x, and who sums the splits, with and without accumulation; a gap of rows no segment covers at the end."""
    from mlora import sgmv_multi
    rng = np.random.default_rng(sum(lens) + hin)
    pp = PagedPool(rng, ranks, hin, hout, page_rows=8, dtype=dtype)
    pool = upload_pool(pp, projections={f"p{i}": (hin, hout) for i in range(n_proj)})
    names = list(pool.projections)
    for nm in names:
        pool.a_rows[nm][0].copy_(bits_to_torch(pp.a_rows, dtype))
        pool.b_rows[nm][0].copy_(bits_to_torch(pp.b_rows, dtype))
    seg = _segments(lens, rng.integers(0, len(ranks), len(lens)))
    T = sum(lens) + 5
    tok = _tok_of(*seg, T)
    dev = [torch.from_numpy(a).cuda() for a in seg]
    x = bits_of(rng.standard_normal((T, hin)).astype(np.float32), dtype)
    y0 = bits_of(rng.standard_normal((T, hout)).astype(np.float32), dtype)
    xt = bits_to_torch(x, dtype, "cuda")
    _assert_shape(shape, [(hin, hout)] * n_proj, [0] * n_proj, T, len(lens), pool.max_rank)
    plan = plan_prefill(*dev, T, pool, n_proj=n_proj)
    for accumulate in (True, False):
        say(f"sgmv launch shapes lens={lens[:4]}x{len(lens)} {hin}->{hout} n_proj={n_proj} dtype={dtype} accumulate={accumulate}")
        ys = [bits_to_torch(y0, dtype, "cuda") for _ in names]
        sgmv_multi(ys, [xt] * n_proj, pool, 0, names, plan, accumulate=accumulate)
        torch.cuda.synchronize()
        want = oracle_apply(pp, x, tok, y0 if accumulate else None)
        for nm, y in zip(names, ys):
            assert_close_bits(torch_to_bits(y), want, dtype, nm)


@pytest.mark.parametrize("splits", [1, 3])
def test_sgmv_workspace_of_a_longer_batch(splits):
    """A workspace with room for fewer splits than a short prompt takes by itself, as a longer batch can leave."""
    from mlora import sgmv_multi
    rng = np.random.default_rng(5)
    T, hin, hout = 255, 4096, 264
    pp = PagedPool(rng, [64], hin, hout, page_rows=8, dtype=FP16)
    pool = upload_pool(pp)
    seg = _segments([T], [0])
    dev = [torch.from_numpy(a).cuda() for a in seg]
    ws = torch.empty(workspace_for_splits(T, 1, 1, splits), dtype=torch.uint8, device="cuda")
    assert sgmv_shape([(hin, hout)], [0], T, 1, 64)["splits"] == [8]
    assert sgmv_shape([(hin, hout)], [0], T, 1, 64, workspace_bytes=ws.numel())["splits"] == [splits]
    x = bits_of(rng.standard_normal((T, hin)).astype(np.float32), FP16)
    y0 = bits_of(rng.standard_normal((T, hout)).astype(np.float32), FP16)
    y = bits_to_torch(y0, FP16, "cuda")
    say(f"sgmv workspace of a longer batch T={T} {hin}->{hout} splits={splits}")
    plan = plan_prefill(*dev, T, pool, workspace=ws)
    sgmv_multi([y], [bits_to_torch(x, FP16, "cuda")], pool, 0, ["p"], plan)
    torch.cuda.synchronize()
    assert_close_bits(torch_to_bits(y), oracle_apply(pp, x, _tok_of(*seg, T), y0), FP16, "short prompt")


@pytest.mark.parametrize("splits", [None, 1])
@pytest.mark.parametrize("long,T,n_seg,n_proj", [(6848, 6144, 1, 1), (3648, 2880, 8, 7), (3648, 3648, 8, 6), (300, 250, 1, 1)])
def test_a_workspace_of_a_larger_call_serves_a_smaller_one(long, T, n_seg, n_proj, splits):
    """A batch in the workspace of a larger call, and in one that is cut to fewer splits than the batch takes by itself, through
    the LoRA call and the one-pass base product; (3648, 3648): fewer projections than it was sized for."""
    from mlora import gemm_lora, sgmv_multi, sgmv_workspace
    rng = np.random.default_rng(long + T)
    hin, hout = 4104, 72
    names = [f"p{i}" for i in range(n_proj)]
    pp = PagedPool(rng, [64, 16, 40], hin, hout, page_rows=8, dtype=FP16)
    pool = upload_pool(pp, projections={nm: (hin, hout) for nm in names})
    for nm in names:
        pool.a_rows[nm][0].copy_(bits_to_torch(pp.a_rows, FP16))
        pool.b_rows[nm][0].copy_(bits_to_torch(pp.b_rows, FP16))
    taken = lambda size: sgmv_shape([(hin, hout)] * n_proj, [0] * n_proj, T, n_seg, 64, workspace_bytes=size)["splits"]  # noqa: E731
    if splits is None:
        ws = sgmv_workspace(long, n_seg, "cuda", 7 if n_seg == 8 else n_proj)
    else:
        ws = torch.empty(workspace_for_splits(T, n_seg, n_proj, splits), dtype=torch.uint8, device="cuda")
        assert taken(ws.numel()) == [splits] * n_proj and min(taken(1 << 50)) > splits
    cuts = np.sort(rng.choice(np.arange(1, T), n_seg - 1, replace=False)) if n_seg > 1 else np.empty(0, np.int64)
    lens = np.diff(np.concatenate([[0], cuts, [T]])).astype(int)
    seg = _segments(lens, rng.integers(0, 3, n_seg))
    dev = [torch.from_numpy(a).cuda() for a in seg]
    x = bits_of(rng.standard_normal((T, hin)).astype(np.float32), FP16)
    y0 = bits_of(rng.standard_normal((T, hout)).astype(np.float32), FP16)
    xt = bits_to_torch(x, FP16, "cuda")
    ys = [bits_to_torch(y0, FP16, "cuda") for _ in names]
    say(f"sgmv_multi T={T} in a workspace for {long}, splits={splits}")
    plan = plan_prefill(*dev, T, pool, workspace=ws)
    sgmv_multi(ys, [xt] * n_proj, pool, 0, names, plan)
    torch.cuda.synchronize()
    tok = _tok_of(*seg, T)
    want = oracle_apply(pp, x, tok, y0)
    for y in ys:
        assert_close_bits(torch_to_bits(y), want, FP16, "sgmv_multi")
    w = (torch.randn(hin, hout, device="cuda") / hin ** 0.5).half()
    outs = [torch.zeros(T, hout, device="cuda").half() for _ in names]
    say(f"gemm_lora T={T} in a workspace for {long}, splits={splits}")
    plan = plan_prefill(*dev, T, pool, workspace=ws, aligned=True)
    gemm_lora(outs, [xt] * n_proj, [w] * n_proj, pool, 0, names, plan)
    torch.cuda.synchronize()
    base = xt.double().cpu().numpy() @ w.double().cpu().numpy()
    for a in range(3):
        v = (f32_of(x, FP16).astype(np.float64)[tok == a] @ pp.A(a)) * np.float64(pp.scaling[a])
        base[tok == a] += v @ pp.B(a)
    for y in outs:
        got = y.double().cpu().numpy()
        assert (np.abs(got - base) <= ATOL + RTOL * np.abs(base)).all()


@pytest.mark.parametrize("lens,ranks,hin,inputs,share,most", [
    ([30], [16], 8, [0], 0, 1),                              # no whole stage of 64 columns
    ([64, 1], [8, 16], 72, [0, 1], 0, 1),                    # one whole stage and a short one; a group of wavefronts without any
    ([129], [32, 20], 1096, [0, 0], 0, 3),                   # ranges of unlike length, the last with the short stage
    ([100, 28], [64], 4160, [0, 0, 0, 0], 0, 8),             # eight splits, four projections of one input
    ([64] * 70 + [17], [64, 40], 200, [0, 0, 0, 1], 1, 1),   # one workgroup for three projections, and for one beside it
    ([64] * 70 + [33], [32], 136, [0, 0, 1, 1, 1], 1, 1),    # for two and for three
    ([64] * 90, [16, 5], 640, [0, 0, 0, 0], 1, 1),           # a fourth projection of the same input starts a new group
    ([64] * 40 + [30], [64, 24], 1032, [0, 0, 0, 1, 1], 1, 2),   # three and two of them in two ranges, the last with a short stage
    ([64] * 41, [32, 8], 2056, [0, 0], 1, 4),                # two in four ranges
])
@pytest.mark.parametrize("dtype", [FP16, BF16])
def test_sgmv_shrink_stages_and_groups(lens, ranks, hin, inputs, share, most, dtype):
    """The ring of stages at its ends (rows shorter than a stage, a last stage of fewer columns, more slots than stages) and
    every number of projections that a workgroup serves, with one K split and with several."""
    from mlora import sgmv_multi
    rng = np.random.default_rng(sum(lens) + hin)
    hout = 136
    pp = PagedPool(rng, ranks, hin, hout, page_rows=8, dtype=dtype)
    names = [f"p{i}" for i in range(len(inputs))]
    pool = upload_pool(pp, projections={nm: (hin, hout) for nm in names})
    for nm in names:
        pool.a_rows[nm][0].copy_(bits_to_torch(pp.a_rows, dtype))
        pool.b_rows[nm][0].copy_(bits_to_torch(pp.b_rows, dtype))
    seg = _segments(lens, rng.integers(0, len(ranks), len(lens)))
    T = sum(lens) + 3
    tok = _tok_of(*seg, T)
    _assert_shape(dict(share=share, most=most), [(hin, hout)] * len(inputs), inputs, T, len(lens), pool.max_rank)
    plan = plan_prefill(*(torch.from_numpy(a).cuda() for a in seg), T, pool, n_proj=len(inputs))
    xs = [bits_of(rng.standard_normal((T, hin)).astype(np.float32), dtype) for _ in range(max(inputs) + 1)]
    xt = [bits_to_torch(x, dtype, "cuda") for x in xs]
    y0 = bits_of(rng.standard_normal((T, hout)).astype(np.float32), dtype)
    for accumulate in (True, False):
        say(f"sgmv stages lens={lens[:2]}x{len(lens)} hin={hin} inputs={inputs} dtype={dtype} accumulate={accumulate}")
        ys = [bits_to_torch(y0, dtype, "cuda") for _ in names]
        sgmv_multi(ys, [xt[i] for i in inputs], pool, 0, names, plan, accumulate=accumulate)
        torch.cuda.synchronize()
        want = [oracle_apply(pp, x, tok, y0 if accumulate else None) for x in xs]
        for i, y in zip(inputs, ys):
            assert_close_bits(torch_to_bits(y), want[i], dtype, f"input {i}")


@pytest.mark.parametrize("lens,gap,ranks,hin,hout,n_proj,shape", [
    ([1], 2, [40], 64, 8, 1, dict(few=1, most=1)),                     # one token, one piece of y
    ([17, 15, 33], 2, [64, 8], 520, 264, 3, dict(few=1, most=2)),      # pieces of 16 tokens with a remainder; a last column block of 8
    ([48], 2, [48], 4096, 2568, 2, dict(few=1, most=8)),               # eight splits
    ([128], 0, [33], 72, 4096, 4, dict(few=1, most=1)),                # one split: halves from the shrink; 512 workgroups
    ([128], 0, [33], 72, 4104, 4, dict(few=0, most=1)),                # 544 workgroups: the expand of 64 tokens
    ([64, 64], 2, [33], 72, 4096, 4, dict(few=0, most=1)),             # 768 by the estimate of two segments in 130 tokens
])
@pytest.mark.parametrize("dtype", [FP16, BF16])
def test_sgmv_few_tiles(lens, gap, ranks, hin, hout, n_proj, shape, dtype):
    """The expand of 16-token pieces on both sides of its limit, summing the splits itself, behind the reduce launch (y = delta) and
    on one split; a segment without an adapter and rows outside every segment."""
    from mlora import sgmv_multi
    rng = np.random.default_rng(sum(lens) + hin)
    pp = PagedPool(rng, ranks, hin, hout, page_rows=8, dtype=dtype)
    names = [f"p{i}" for i in range(n_proj)]
    pool = upload_pool(pp, projections={nm: (hin, hout) for nm in names})
    for nm in names:
        pool.a_rows[nm][0].copy_(bits_to_torch(pp.a_rows, dtype))
        pool.b_rows[nm][0].copy_(bits_to_torch(pp.b_rows, dtype))
    adapters = rng.integers(0, len(ranks), len(lens))
    if len(lens) > 2:
        adapters[1] = -1
    seg = _segments(lens, adapters)
    T = sum(lens) + gap
    tok = _tok_of(*seg, T)
    _assert_shape(shape, [(hin, hout)] * n_proj, [0] * n_proj, T, len(lens), pool.max_rank)
    plan = plan_prefill(*(torch.from_numpy(a).cuda() for a in seg), T, pool, n_proj=n_proj)
    x = bits_of(rng.standard_normal((T, hin)).astype(np.float32), dtype)
    y0 = bits_of(rng.standard_normal((T, hout)).astype(np.float32), dtype)
    xt = bits_to_torch(x, dtype, "cuda")
    for accumulate in (True, False):
        say(f"sgmv few tiles lens={lens} {hin}->{hout} n_proj={n_proj} dtype={dtype} accumulate={accumulate}")
        ys = [bits_to_torch(y0, dtype, "cuda") for _ in names]
        sgmv_multi(ys, [xt] * n_proj, pool, 0, names, plan, accumulate=accumulate)
        torch.cuda.synchronize()
        want = oracle_apply(pp, x, tok, y0 if accumulate else None)
        for y in ys:
            assert_close_bits(torch_to_bits(y), want, dtype)


@pytest.mark.parametrize("lens,ranks,hin,hout,n_proj,few,many", [
    ([64] * 11 + [30, 1], [64, 40], 1096, 4096, 3, 0, True),       # 18 tiles by the estimate, 3456 workgroups
    ([64] * 9 + [30, 1], [64, 40], 1096, 4096, 3, 1, True),        # 2880
    ([64] * 13 + [30], [64], 1096, 5128, 2, 0, True),              # 3360
    ([64] * 22, [48], 4096, 4104, 3, 0, True),
    ([700], [16, 5], 72, 4104, 7, 1, False),                       # 11 tiles, 5236 workgroups
    ([700], [16], 1096, 6152, 7, 0, True),                         # 7700
    ([33, 640], [32, 20], 1096, 4104, 7, 1, True),
    ([1000], [24], 72, 4104, 7, 0, False),
    ([641], [32, 20], 1096, 6152, 7, 0, True),
])
@pytest.mark.parametrize("dtype", [FP16, BF16])
def test_sgmv_both_expands(lens, ranks, hin, hout, n_proj, few, many, dtype):
    """Both kernels at the ranks of every instance, on either side of the number of workgroups at which they change, summing the
    splits themselves (up to rank 32, or few) and behind the reduce launch (y = delta); rows at the end outside every segment."""
    from mlora import sgmv_multi
    rng = np.random.default_rng(sum(lens) + hout)
    pp = PagedPool(rng, ranks, hin, hout, page_rows=8, dtype=dtype)
    names = [f"p{i}" for i in range(n_proj)]
    pool = upload_pool(pp, projections={nm: (hin, hout) for nm in names})
    for nm in names:
        pool.a_rows[nm][0].copy_(bits_to_torch(pp.a_rows, dtype))
        pool.b_rows[nm][0].copy_(bits_to_torch(pp.b_rows, dtype))
    seg = _segments(lens, rng.integers(0, len(ranks), len(lens)))
    x = bits_of(rng.standard_normal((sum(lens) + 3, hin)).astype(np.float32), dtype)
    y0 = bits_of(rng.standard_normal((sum(lens) + 3, hout)).astype(np.float32), dtype)
    for gap, accumulate in ((0, True), (3, True), (3, False)):
        T = sum(lens) + gap
        shape = sgmv_shape([(hin, hout)] * n_proj, [0] * n_proj, T, len(lens), pool.max_rank, accumulate)
        assert shape["few"] == few and (max(shape["splits"]) > 1) == many, shape
        assert shape["reduce"] == (not accumulate or (many and pool.max_rank > 32 and not few)), shape
        plan = plan_prefill(*(torch.from_numpy(a).cuda() for a in seg), T, pool, n_proj=n_proj)
        say(f"sgmv both expands lens={lens[:2]}x{len(lens)} ranks={ranks} {hin}->{hout} n_proj={n_proj} dtype={dtype} accumulate={accumulate}")
        ys = [bits_to_torch(y0[:T], dtype, "cuda") for _ in names]
        sgmv_multi(ys, [bits_to_torch(x[:T], dtype, "cuda")] * n_proj, pool, 0, names, plan, accumulate=accumulate)
        torch.cuda.synchronize()
        want = oracle_apply(pp, x[:T], _tok_of(*seg, T), y0[:T] if accumulate else None)
        for y in ys:
            assert_close_bits(torch_to_bits(y), want, dtype)


@pytest.mark.parametrize("aligned", [False, True])
@pytest.mark.parametrize("n_seg,longest", [(300, 5), (17, 1100), (1, 1)])
def test_plan_over_several_workgroups(n_seg, longest, aligned):
    """More segments than a workgroup looks at together, more tiles and more tokens than one writes: the tile list is the
    oracle's, and y = delta is zero exactly in the rows outside every segment."""
    from oracle import oracle as orc
    rng = np.random.default_rng(n_seg)
    lens = rng.integers(1, longest + 1, n_seg).astype(np.int32)
    gaps = rng.integers(0, 3, n_seg).astype(np.int32)
    ss = (np.cumsum(lens + gaps) - lens).astype(np.int32)
    T = int(ss[-1] + lens[-1]) + 4
    pp = PagedPool(rng, [16, 8, 4], 64, 64, page_rows=8, dtype=FP16)
    pool = upload_pool(pp)
    sa = rng.integers(0, 3, n_seg).astype(np.int32)
    say(f"plan of {n_seg} segments, {T} tokens, aligned={aligned}")
    plan = plan_prefill(*(torch.from_numpy(a).cuda() for a in (ss, lens, sa)), T, pool, aligned=aligned)
    torch.cuda.synchronize()
    want = orc.sgmv_plan(ss, lens, 64, aligned=aligned)
    max_tiles = T // 64 + 2 * n_seg + 1
    words = plan.workspace[:(3 * max_tiles + 1) * 4].cpu().numpy().view(np.int32)
    n = int(words[3 * max_tiles])
    assert n == len(want[0])
    for i in range(3):
        assert np.array_equal(words[i * max_tiles:i * max_tiles + n], want[i])
    x = torch.ones(T, 64, device="cuda", dtype=torch.float16)
    y = torch.full((T, 64), float("nan"), device="cuda", dtype=torch.float16)
    sgmv(y, x, pool, 0, "p", plan=plan, accumulate=False)
    torch.cuda.synchronize()
    covered = np.zeros(T, bool)
    for s, ln in zip(ss, lens):
        covered[s:s + ln] = True
    assert np.array_equal((y != 0).any(1).cpu().numpy(), covered) and bool(torch.isfinite(y).all())
