"""GPU check of the allocation-free decode entry point (mlora_bgmv_multi_noalloc) through the C ABI: its
output equals, bit for bit, that of mlora_bgmv_multi with a caller workspace (the same kernels), on two
calls in a row, the second on a smaller batch, and both meet the oracle's tolerance."""
import ctypes as C

import numpy as np
import pytest
import torch

from gpu_common import assert_close_bits, oracle_apply, say, upload_pool
from helpers import FP16, PagedPool, bits_of, bits_to_torch, torch_to_bits
from mlora import _ext, plan_decode

pytestmark = pytest.mark.gpu


def _call(pool, plan, tok, xs, ys, hins, houts, noalloc, ws=None):
    n = len(xs)
    VP, IP = C.c_void_p * _ext.MAX_PROJ, C.c_int32 * _ext.MAX_PROJ
    yv, xv, av, bv, hi, ho = VP(), VP(), VP(), VP(), IP(), IP()
    a_ptr, b_ptr = pool.slab_ptrs(0, "p")
    for i in range(n):
        yv[i], xv[i], av[i], bv[i], hi[i], ho[i] = ys[i].data_ptr(), xs[i].data_ptr(), a_ptr, b_ptr, hins[i], houts[i]
    T = tok.numel()
    lib = _ext.lib()
    common = (n, yv, xv, av, bv, hi, ho, tok.data_ptr(), T, pool.page_tbl.data_ptr(), pool.rank.data_ptr(),
              pool.scaling.data_ptr(), pool.n_slots, pool.max_pages, pool.page_rows, pool.n_pages, pool.max_rank,
              plan.work.data_ptr(), plan.group)
    stream = torch.cuda.current_stream().cuda_stream
    if noalloc:
        rc = lib.mlora_bgmv_multi_noalloc(*common, pool.dtype_code, 1, stream)
    else:
        rc = lib.mlora_bgmv_multi(*common, ws.data_ptr(), ws.numel(), pool.dtype_code, 1, stream)
    _ext.check(rc)


def test_noalloc_matches_workspace_form_on_two_calls():
    rng = np.random.default_rng(777)
    hin = hout = 2048
    ranks = rng.choice([8, 16, 32, 64], 24)
    pp = PagedPool(rng, ranks, hin, hout, page_rows=8, dtype=FP16)
    pool = upload_pool(pp)
    lib = _ext.lib()
    for T in (300, 41):                                   # second call: smaller batch over the array the first one used
        tok_np = rng.integers(-1, len(ranks), T).astype(np.int32)
        tok = torch.from_numpy(tok_np).cuda()
        plan = plan_decode(tok, pool, group=4)
        x_bits = [bits_of(rng.standard_normal((T, hin)).astype(np.float32), FP16) for _ in range(2)]
        y0_bits = [bits_of(rng.standard_normal((T, hout)).astype(np.float32), FP16) for _ in range(2)]
        xs = [bits_to_torch(b, FP16, "cuda") for b in x_bits]
        ws = torch.empty(lib.mlora_bgmv_workspace_bytes(2, T, hin, pool.max_rank), dtype=torch.uint8, device="cuda")
        y_ws = [bits_to_torch(b, FP16, "cuda") for b in y0_bits]
        y_na = [bits_to_torch(b, FP16, "cuda") for b in y0_bits]
        torch.cuda.synchronize()
        say(f"noalloc decode T={T}: workspace form")
        _call(pool, plan, tok, xs, y_ws, [hin] * 2, [hout] * 2, noalloc=False, ws=ws)
        torch.cuda.synchronize()
        before = torch.cuda.memory_allocated()
        say(f"noalloc decode T={T}: allocation-free form")
        _call(pool, plan, tok, xs, y_na, [hin] * 2, [hout] * 2, noalloc=True)
        torch.cuda.synchronize()
        assert torch.cuda.memory_allocated() == before
        for i in range(2):
            got = torch_to_bits(y_na[i])
            assert np.array_equal(got, torch_to_bits(y_ws[i])), f"T={T} projection {i}: differs from the workspace form"
            assert_close_bits(got, oracle_apply(pp, x_bits[i], tok_np, y0_bits[i]), FP16, f"noalloc T={T}")


@pytest.mark.parametrize("T", [1, 5, 24])
def test_results_do_not_depend_on_the_size_of_the_workspace(T):
    """A small batch, which mlora_bgmv_form would run in 512-column slices: mlora_bgmv_multi gives the same bits with a
    workspace of the size it asks for and with one many times as large, and so does the allocation-free form."""
    rng = np.random.default_rng(779 + T)
    hin, hout, ranks = 4096, 4096, [16, 64, 32]
    pp = PagedPool(rng, ranks, hin, hout, page_rows=8, dtype=FP16)
    pool = upload_pool(pp)
    tok_np = rng.integers(-1, len(ranks), T).astype(np.int32)
    tok = torch.from_numpy(tok_np).cuda()
    plan = plan_decode(tok, pool, group=1)
    x = bits_of(rng.standard_normal((T, hin)).astype(np.float32), FP16)
    y0 = bits_of(rng.standard_normal((T, hout)).astype(np.float32), FP16)
    need = _ext.lib().mlora_bgmv_workspace_bytes(1, T, hin, pool.max_rank)
    outs = []
    for size in (need, 64 * need, None):
        y = bits_to_torch(y0, FP16, "cuda")
        ws = None if size is None else torch.empty(size, dtype=torch.uint8, device="cuda")
        say(f"decode T={T} with a workspace of {size} bytes")
        _call(pool, plan, tok, [bits_to_torch(x, FP16, "cuda")], [y], [hin], [hout], noalloc=size is None, ws=ws)
        torch.cuda.synchronize()
        outs.append(torch_to_bits(y))
    assert_close_bits(outs[0], oracle_apply(pp, x, tok_np, y0), FP16, f"workspace form T={T}")
    assert np.array_equal(outs[0], outs[1]) and np.array_equal(outs[0], outs[2])


def test_noalloc_rejects_a_batch_beyond_its_array():
    rng = np.random.default_rng(778)
    pp = PagedPool(rng, [64] * 4, 64, 64, page_rows=8, dtype=FP16)
    pool = upload_pool(pp)
    T = 8192
    tok = torch.zeros(T, dtype=torch.int32, device="cuda")
    plan = plan_decode(tok, pool, group=4)
    x = torch.zeros((T, 64), dtype=torch.float16, device="cuda")
    y = torch.zeros((T, 64), dtype=torch.float16, device="cuda")
    # widths are validated against the arrays passed here, not dereferenced: 8 projections of hin 11008 need 184 MB
    with pytest.raises(_ext.MloraError) as e:
        _call(pool, plan, tok, [x] * 8, [y] * 8, [11008] * 8, [64] * 8, noalloc=True)
    assert e.value.code == _ext.MLORA_ENOSPACE
