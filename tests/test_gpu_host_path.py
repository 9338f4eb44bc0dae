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
