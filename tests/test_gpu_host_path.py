"""The native launch path of the eager calls: what it rejects, and that it reads the pool it is given on every call."""
import numpy as np
import pytest
import torch

import mlora
from gpu_common import assert_close_bits, oracle_apply, say, upload_pool
from helpers import FP16, PagedPool, bits_of, bits_to_torch, torch_to_bits

pytestmark = pytest.mark.gpu


def _setup(T=5, hin=64, hout=96):
    pp = PagedPool(np.random.default_rng(7), [8, 16], hin, hout, page_rows=8, dtype=FP16)
    pool = upload_pool(pp)
    tok = torch.tensor([0, 1, -1, 1, 0][:T], dtype=torch.int32, device="cuda")
    x = torch.randn(T, hin, device="cuda").half()
    y = torch.zeros(T, hout, device="cuda").half()
    return pp, pool, tok, x, y


BAD = {
    "cpu tensor": (ValueError, lambda x, y: ([x.cpu()], [y])),
    "not contiguous": (ValueError, lambda x, y: ([x.t().contiguous().t()], [y])),
    "dtype": (TypeError, lambda x, y: ([x.float()], [y])),
    "rows": (ValueError, lambda x, y: ([x[:-1]], [y])),
    "width": (ValueError, lambda x, y: ([x], [y[:, :-8].contiguous()])),
    "dim": (ValueError, lambda x, y: ([x], [y[None]])),
    "count": (ValueError, lambda x, y: ([x, x], [y])),
}


@pytest.mark.parametrize("what", list(BAD))
def test_calls_reject_what_they_cannot_take(what):
    pp, pool, tok, x, y = _setup()
    error, change = BAD[what]
    xs, ys = change(x, y)
    plan = mlora.plan_decode(tok, pool)
    seg = tuple(torch.tensor(v, dtype=torch.int32, device="cuda") for v in ([0], [5], [1]))
    pplan = mlora.plan_prefill(*seg, 5, pool)
    with pytest.raises(error):
        mlora.bgmv(ys, xs, pool, 0, ["p"], tok, plan=plan)
    with pytest.raises(error):
        mlora.sgmv_multi(ys, xs, pool, 0, ["p"], pplan)


def test_calls_reject_other_bad_arguments():
    pp, pool, tok, x, y = _setup()
    plan = mlora.plan_decode(tok, pool)
    for error, kw in ((TypeError, dict(tok=tok.long())), (KeyError, dict(projs=["none"])), (IndexError, dict(layer=1)),
                      (ValueError, dict(plan=None, fused=False)), (ValueError, dict(plan=mlora.plan_decode(tok[:4].contiguous(), pool)))):
        a = dict(layer=0, projs=["p"], tok=tok, plan=plan, fused=None)
        a.update(kw)
        with pytest.raises(error):
            mlora.bgmv([y], [x], pool, a["layer"], a["projs"], a["tok"], plan=a["plan"], fused=a["fused"])
    with pytest.raises(TypeError):
        mlora.plan_prefill(*(torch.tensor(v, dtype=torch.int64, device="cuda") for v in ([0], [5], [1])), 5, pool,
                           workspace=mlora.sgmv_workspace(5, 1, "cuda"))


def test_slabs_are_read_from_the_pool_on_every_call():
    """A pool whose slab tensor is replaced between two calls: the second call uses the new one."""
    pp, pool, tok, x, y = _setup()
    plan = mlora.plan_decode(tok, pool)
    say("bgmv before and after the B slab is replaced")
    mlora.bgmv([y], [x], pool, 0, ["p"], tok, plan=plan, accumulate=False)
    pool.b_rows["p"] = pool.b_rows["p"] * 2
    y2 = torch.zeros_like(y)
    mlora.bgmv([y2], [x], pool, 0, ["p"], tok, plan=plan, accumulate=False)
    torch.cuda.synchronize()
    want = oracle_apply(pp, torch_to_bits(x), tok.cpu().numpy())
    assert_close_bits(torch_to_bits(y), want, FP16, "first slab")
    # Doubling is exact where y is a normal fp16 number.  Below 2^-14 the spacing no longer falls with the value: y is up
    # to half a step (2^-25) from its sum, which doubling doubles, and y2 up to half a step from twice that sum.
    normal = y.abs() >= 2.0 ** -14
    assert torch.equal(y2[normal], (y * 2)[normal])
    assert bool(((y2.float() - 2 * y.float())[~normal].abs() <= 3 * 2.0 ** -25).all())


def test_a_plan_refuses_a_larger_batch_and_stays_usable():
    """A batch larger than the plan's buffers is refused before anything is launched, and leaves the plan its own batch."""
    pp, pool, tok, x, y = _setup(T=4)
    plan = mlora.plan_decode(tok, pool)
    with pytest.raises(ValueError):
        mlora.plan_decode(torch.zeros(300, dtype=torch.int32, device="cuda"), pool, out=plan)
    assert plan.tok_adapter is tok
    say("bgmv on a plan that refused a larger batch")
    mlora.bgmv([y], [x], pool, 0, ["p"], tok, plan=plan, accumulate=False)
    torch.cuda.synchronize()
    assert_close_bits(torch_to_bits(y), oracle_apply(pp, torch_to_bits(x), tok.cpu().numpy()), FP16, "own batch")


def test_a_prefill_workspace_in_host_memory_is_refused():
    """Every prefill entry point writes its workspace from the device: one in host memory is refused before a launch."""
    pp, pool, tok, x, y = _setup()
    seg = tuple(torch.tensor(v, dtype=torch.int32, device="cuda") for v in ([0], [5], [1]))
    host = mlora.sgmv_workspace(5, 1, "cpu")
    strided = torch.empty((host.numel(), 2), dtype=torch.uint8, device="cuda")[:, 0]
    w = torch.zeros(64, 96, device="cuda").half()
    for ws in (host, strided):
        plan = mlora.PrefillPlan(*seg, 5, ws)
        for call in (lambda: mlora.plan_prefill(*seg, 5, pool, workspace=ws), lambda: mlora.sgmv_multi([y], [x], pool, 0, ["p"], plan),
                     lambda: mlora.sgmv(y, x, pool, 0, "p", plan=plan), lambda: mlora.sgmv(y, x, pool, 0, "p", *seg, workspace=ws),
                     lambda: mlora.gemm_lora([y], [x], [w], pool, 0, ["p"], plan),
                     lambda: mlora.lora_prefill_ref(x[None], torch.zeros(1, 1, 8, 64, device="cuda").half(),
                                                    torch.zeros(1, 1, 96, 8, device="cuda").half(), 0, workspace=ws)):
            with pytest.raises(ValueError):
                call()


def _small_batch(n_proj, T=6, hin=2048, hout=1536, ranks=(64, 16, 40)):
    """A batch that mlora_bgmv_form runs as two launches, and its projections' names."""
    pp = PagedPool(np.random.default_rng(17), list(ranks), hin, hout, page_rows=8, dtype=FP16)
    names = [f"p{i}" for i in range(n_proj)]
    pool = upload_pool(pp, projections={nm: (hin, hout) for nm in names})
    gen = torch.Generator(device="cuda").manual_seed(3)
    for nm in names:
        pool.a_rows[nm].copy_(torch.randn(pool.a_rows[nm].shape, device="cuda", generator=gen) * 0.02)
        pool.b_rows[nm].copy_(torch.randn(pool.b_rows[nm].shape, device="cuda", generator=gen) * 0.02)
    tok = torch.tensor([i % (len(ranks) + 1) - 1 for i in range(T)], dtype=torch.int32, device="cuda")
    xs = [torch.randn(T, hin, device="cuda", generator=gen).half() for _ in range(8)]
    return pool, names, tok, xs, lambda: [torch.zeros(T, hout, device="cuda").half() for _ in names]


@pytest.mark.parametrize("fused", [None, False, True])
def test_a_call_leaves_its_plan_as_it_was(fused):
    pool, names, tok, xs, zeros = _small_batch(3)
    plan = mlora.plan_decode(tok, pool)
    before = dict(vars(plan))
    say(f"bgmv on a plan that stays as it was, fused={fused}")
    mlora.bgmv(zeros(), xs[:3], pool, 0, names, tok, plan=plan, fused=fused)
    torch.cuda.synchronize()
    assert vars(plan).keys() == before.keys() and all(v is before[k] for k, v in vars(plan).items())


def test_small_batches_that_share_a_plan_on_several_streams_and_threads():
    """Calls of one plan that overlap, from one thread on two streams and from four threads on a stream each."""
    import threading
    pool, names, tok, xs, zeros = _small_batch(3)
    plan = mlora.plan_decode(tok, pool)
    want = []
    for x in xs:
        y = zeros()
        mlora.bgmv(y, [x] * 3, pool, 0, names, tok, plan=plan, accumulate=False)
        want.append(y)
    torch.cuda.synchronize()

    def run(which, stream, out, reps=40):
        with torch.cuda.stream(stream):
            for i in range(reps):
                k = (which + i) % len(xs)
                mlora.bgmv(out[i], [xs[k]] * 3, pool, 0, names, tok, plan=plan, accumulate=False)

    say("bgmv on two streams and one plan")
    outs = [[zeros() for _ in range(40)] for _ in range(4)]
    streams = [torch.cuda.Stream() for _ in range(4)]
    torch.cuda.synchronize()
    for i in range(40):
        for j in range(2):
            with torch.cuda.stream(streams[j]):
                mlora.bgmv(outs[j][i], [xs[(j + i) % len(xs)]] * 3, pool, 0, names, tok, plan=plan, accumulate=False)
    torch.cuda.synchronize()
    for j in range(2):
        for i in range(40):
            assert all(torch.equal(a, b) for a, b in zip(outs[j][i], want[(j + i) % len(xs)])), (j, i)
    say("bgmv from four threads and one plan")
    threads = [threading.Thread(target=run, args=(j, streams[j], outs[j])) for j in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    torch.cuda.synchronize()
    for j in range(4):
        for i in range(40):
            assert all(torch.equal(a, b) for a, b in zip(outs[j][i], want[(j + i) % len(xs)])), (j, i)


def test_a_captured_step_keeps_its_intermediate():
    """Eager calls of other sizes on the plan of a captured step, and new tensors after them: the replay gives the same
    bits and writes to none of the new tensors."""
    pool, names, tok, xs, zeros = _small_batch(7)
    plan = mlora.plan_decode(tok, pool, n_proj=7)
    y = zeros()
    step = lambda: mlora.bgmv(y, xs[:7], pool, 0, names, tok, plan=plan, accumulate=False)  # noqa: E731
    say("bgmv captured, then eager calls on the same plan")
    step()
    torch.cuda.synchronize()
    want = [t.clone() for t in y]
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        step()
    for n in (1, 3, 7):
        mlora.bgmv(zeros()[:n], xs[:n], pool, 0, names[:n], tok, plan=plan, fused=False)
    fresh = [torch.full((1 << 20,), 7.0, device="cuda") for _ in range(8)]
    for rep in range(3):
        for t in y:
            t.fill_(float(rep))
        torch.cuda.synchronize()
        g.replay()
        torch.cuda.synchronize()
        assert all(torch.equal(a, b) for a, b in zip(y, want)), rep
        assert all(bool((t == 7.0).all()) for t in fresh), rep
