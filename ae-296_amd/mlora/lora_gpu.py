"""Host-side mirror of the reference's ``Lora_GPU`` (``lightllm/models/lora_gpu.py``) for the
apply path: same constructor keys, same pool attributes and shapes, same
``invoke_one_layer_{q,k,v}(x, layer_id, prefill)`` calls that
``LlamaTransformerLayerInfer._get_qkv`` makes
(``lightllm/models/llama/layer_infer/transformer_layer_infer.py:76-81,101-111``) -- with the
decode branch on the HIP BGMV kernel instead of ``punica.ops.add_lora_bgmv`` and the prefill
branch on the HIP SGMV kernels instead of ``torch.bmm(torch.bmm(...))`` plus two weight
transposes per call.

Left out on purpose (not part of the apply path): the zmq / CUDA-IPC sharing with the
swapper process (``lora_gpu.py:76-118,246-296``) and the progress polling (``:298-339``).
"""
from __future__ import annotations

import itertools
from operator import attrgetter

import numpy as np
import torch

from . import _ext, ops

_QKV_WEIGHTS = attrgetter("q_down", "q_up", "k_down", "k_up", "v_down", "v_up")


class Lora_GPU:
    def __init__(self, configJson, shared: bool = False, device: str = "cuda", seed: int = 0):
        self.device = torch.device(device)
        self.n_layers = configJson["n_layers"]
        self.batch_size = configJson["batch_size"]
        self.lora_rank = configJson["lora_rank"]
        self.in_size = configJson["hidden_dim"]
        self.output_size = configJson["hidden_dim"] // configJson["tp_degree"]
        self.tp_degree = configJson["tp_degree"]
        self.max_prefill_batch_size = configJson["max_prefill_batch_size"]
        self.dtype = configJson.get("dtype", torch.float16)
        self._gen = torch.Generator(device=self.device)
        self._gen.manual_seed(seed)

        # Decode pool, reference layout (lora_gpu.py:33-40): down [N, L, r, Hin], up [N, L, Hout, r].
        # The reference leaves these uninitialised (torch.empty); they are given small random values here.
        for name in ("q", "k", "v"):
            setattr(self, f"{name}_down", self._rand(self.batch_size, self.in_size, self.lora_rank))
            setattr(self, f"{name}_up", self._rand(self.batch_size, self.lora_rank, self.output_size))
            setattr(self, f"{name}_down_prefill", None)
            setattr(self, f"{name}_up_prefill", None)
        mode = configJson.get("mode", [])
        if shared or "aaas-cached" in mode or "aaas-gpu" in mode:
            self.prepare_lora_prefill(self.max_prefill_batch_size)

        # Per-batch-size index vectors (lora_gpu.py:120).  The reference draws from [0, 32) whatever the
        # pool size, which reads out of bounds when batch_size < 32; indices are kept inside the pool here.
        hi = min(32, self.batch_size)
        self.select_inds = [torch.randint(0, hi, (i + 1,), device=self.device, generator=self._gen)
                            for i in range(self.batch_size)]
        self._workspace = None                         # of the newest prefill call ...
        self._workspace_for = (0, 0, None, None)       # ... the rows and requests it was sized for, the order it belongs to, itself
        # Grouping of the current decode batch by adapter: (plan, the index tensor it was made from, its torch version, the
        # order it belongs to, its number).  It is served again only for the very tensor object it was made from (kept
        # alive here so that neither its address nor its Python identity can pass to another tensor) at the same version
        # counter: a serving loop builds `lora_ids` afresh every step (pre_process.py:50,100), and a new tensor of the same
        # size often gets the freed one's address.  A plan that an invoke call made by itself belongs to that call's thread,
        # stream and graph capture (mlora._host.order): a call elsewhere is not ordered behind the launch that writes it, and
        # makes its own.  One that plan_decode made (order None) serves wherever the program has ordered its calls behind that.
        self._plan_state = (None, None, None, None, 0)
        self._plan_gen = 0                             # number of the newest plan
        self._plan_numbers = itertools.count(1)
        # q, k, v deltas of the last decode input that were not asked for yet: (what they were computed from, the deltas, the
        # input tensor itself and the six weight tensors (kept alive for the same reason))
        self._qkv = None

    def _rand(self, n, rows, cols):
        """[n, L, rows, cols] * 0.001, stored transposed and contiguous as the reference does."""
        w = torch.randn((n, self.n_layers, rows, cols), device=self.device, dtype=torch.float32,
                        generator=self._gen) * 0.001
        return w.to(self.dtype).transpose(-1, -2).contiguous()

    # ------------------------------------------------------------------ apply
    def _index_source(self, bsz, lora_ids):
        # The reference drops the request's adapter ids (``infer_state.lora_ids``, built at
        # pre_process.py:50,100) and applies a random stand-in; pass ``lora_ids`` to use the real ones.
        if lora_ids is None:
            return self.select_inds[bsz - 1]
        if lora_ids.numel() != bsz:
            raise ValueError("lora_ids must hold one adapter slot per row of x")
        return lora_ids

    def _indices(self, bsz, lora_ids, device):
        """The index vector as the kernels take it: int64 on the device (int32 ids, pre_process.py:100, are widened)."""
        src = self._index_source(bsz, lora_ids)
        if src.dtype == torch.int64 and src.device == device:
            return src
        return src.to(device=device, dtype=torch.int64)

    def plan_decode(self, bsz, lora_ids=None):
        """Group the decode batch by adapter (one gather launch): the step boundary.  A serving loop calls it once
        per step; ``invoke_one_layer_*`` call it themselves when they are handed another index tensor than the one
        the current plan was made from, or the same one after torch has written to it.  A tensor whose contents
        were changed behind torch's back (a raw kernel writing through its pointer) needs this call."""
        return self._group(bsz, lora_ids, None)[0]

    def _group(self, bsz, lora_ids, order):
        """A new plan and its number.  It takes the buffers of the plan before it only where no call elsewhere may read them."""
        src = self._index_source(bsz, lora_ids)
        cur_inds = self._indices(bsz, lora_ids, self.q_down.device)
        last, _, _, belongs, _ = self._plan_state
        mine = belongs == order or (order is None and belongs == _ext.host().order())
        reuse = last if (last is not None and mine and last.T == bsz) else None
        plan = ops.plan_decode_ref(cur_inds, self.batch_size, self.n_layers, self.lora_rank, out=reuse)
        self._plan_gen = number = next(self._plan_numbers)
        self._plan_state = (plan, src, src._version, order, number)
        self._qkv = None
        return plan, number

    def _plan_for(self, bsz, lora_ids):
        src = self._index_source(bsz, lora_ids)
        plan, made_from, version, belongs, number = self._plan_state
        if plan is None or made_from is not src or version != src._version or plan.T != bsz or (
                belongs is not None and belongs != _ext.host().order()):
            return self._group(bsz, lora_ids, _ext.host().order())
        return plan, number

    def invoke_one_layer_qkv(self, x, layer_id, lora_ids=None):
        """The q, k and v deltas of one decode layer in one call pair (the reference makes three
        ``add_lora_bgmv`` calls with a ``torch.zeros`` each, lora_gpu.py:137-138,149-150,161-162): returns
        ``(q_lora, k_lora, v_lora)``, each ``[bsz, hidden / tp]``."""
        bsz = x.shape[0]
        if not ops.ref_rank_supported(self.lora_rank):
            return tuple(self._invoke_single(n, x, layer_id, lora_ids) for n in "qkv")
        return self._deltas(x, layer_id, self._plan_for(bsz, lora_ids)[0], _QKV_WEIGHTS(self))

    @staticmethod
    def _deltas(x, layer_id, plan, weights):
        """The deltas of one input and the projections whose down and up tensors `weights` lists, in new tensors."""
        if not x.is_contiguous():
            x = x.contiguous()
        ys = _ext.host().deltas_ref(plan, x, weights, layer_id, plan.T, plan.N, plan.L, plan.r)
        if ys.__class__ is int:
            _ext.check(ys)
        return ys

    def _invoke_single(self, name, x, layer_id, lora_ids):
        bsz = x.shape[0]
        cur_inds = self._indices(bsz, lora_ids, x.device)
        y = torch.zeros(bsz, self.output_size, device=x.device, dtype=x.dtype)
        ops.add_lora_bgmv(y, x, getattr(self, f"{name}_down"), getattr(self, f"{name}_up"), cur_inds, layer_id, 1)
        return y

    def _invoke(self, name, x, layer_id, prefill, lora_ids=None):
        bsz = x.shape[0]
        if prefill:
            down, up = getattr(self, f"{name}_down_prefill"), getattr(self, f"{name}_up_prefill")
            if down is None:
                raise RuntimeError("prefill adapters are not loaded (call prepare_lora_prefill)")
            if not x.is_contiguous():
                x = x.contiguous()
            # A shorter batch than it was sized for keeps the workspace.  It serves one thread, stream and capture
            # (mlora._host.order): calls elsewhere may overlap, and a captured call goes on using the one it was given.
            order = _ext.host().order()
            had_rows, had_reqs, belongs, ws = self._workspace_for
            if belongs != order:
                had_rows = had_reqs = 0
            rows, reqs = max(bsz * x.shape[1], had_rows), max(bsz, had_reqs)
            if (rows, reqs) != (had_rows, had_reqs):
                ws = ops.sgmv_workspace(rows, reqs, x.device)
                self._workspace, self._workspace_for = ws, (rows, reqs, order, ws)
            return ops.lora_prefill_ref(x, down, up, layer_id, workspace=ws)
        if not ops.ref_rank_supported(self.lora_rank):
            return self._invoke_single(name, x, layer_id, lora_ids)
        # ``_get_qkv`` asks for q, k and v of the same input one after the other
        # (transformer_layer_infer.py:109-111): the first of the three calls computes all of them in one call pair,
        # the other two are answered from that result as long as it is the same input tensor object at the same
        # torch version, the same layer, the same plan, the same weight tensors at the same versions, and the same thread,
        # stream and graph capture: a call elsewhere is not ordered behind the launches that write the result.
        plan, number = self._plan_for(bsz, lora_ids)
        weights = _QKV_WEIGHTS(self)
        key = (_ext.host().state(x, weights), x.shape, layer_id, number)
        kept = self._qkv
        if kept is not None and kept[0] == key:
            y = kept[1].pop(name, None)
            if y is not None:
                return y
        q, k, v = self._deltas(x, layer_id, plan, weights)
        left = {"q": q, "k": k, "v": v}
        y = left.pop(name)
        self._qkv = (key, left, x, weights)
        return y

    def invoke_one_layer_q(self, x, layer_id, prefill=False, lora_ids=None):
        return self._invoke("q", x, layer_id, prefill, lora_ids)

    def invoke_one_layer_k(self, x, layer_id, prefill=False, lora_ids=None):
        return self._invoke("k", x, layer_id, prefill, lora_ids)

    def invoke_one_layer_v(self, x, layer_id, prefill=False, lora_ids=None):
        return self._invoke("v", x, layer_id, prefill, lora_ids)

    # ------------------------------------------------------------------ slot management
    def prepare_lora_prefill(self, batch_size):
        """lora_gpu.py:190-200: fresh random prefill adapters, one slot per request."""
        self._qkv = None
        for name in ("q", "k", "v"):
            setattr(self, f"{name}_down_prefill", self._rand(batch_size, self.in_size, self.lora_rank))
            setattr(self, f"{name}_up_prefill", self._rand(batch_size, self.lora_rank, self.output_size))

    def merge_lora_prefill(self, bsz, re_inds=None):
        """lora_gpu.py:202-217: copy the first bsz prefill slots into decode slots (random targets
        in the reference; pass re_inds to choose them)."""
        self._qkv = None                        # weights change: results computed from the old ones are not served again
        if re_inds is None:
            re_inds = np.random.randint(0, self.batch_size, size=bsz)
        for idx, re_ind in enumerate(re_inds):
            for name in ("q", "k", "v"):
                getattr(self, f"{name}_down")[re_ind].copy_(getattr(self, f"{name}_down_prefill")[idx])
                getattr(self, f"{name}_up")[re_ind].copy_(getattr(self, f"{name}_up_prefill")[idx])
        return re_inds

    def remove_lora(self, rm_ids, running_bsz, chosen=None):
        """lora_gpu.py:229-242 shifts slices of the *second* axis of [N, L, ...] tensors, i.e. layers, which
        looks unintended; the documented intent (drop the adapters of finished requests, closing the gap)
        is applied to the adapter axis here."""
        if running_bsz <= 0:
            return
        self._qkv = None
        if chosen is None:
            chosen = np.random.randint(0, running_bsz, size=len(rm_ids))
        for rm_id in chosen:
            for name in ("q", "k", "v"):
                for side in ("down", "up"):
                    w = getattr(self, f"{name}_{side}")
                    w[rm_id:-1] = w[rm_id + 1:].clone()
