"""What Lora_GPU keeps between the q, k and v calls of a layer, and for whom: the launches are replaced by stand-ins that
count, so no GPU is needed."""
import threading

import pytest
import torch

from mlora import Lora_GPU, _ext, ops


class _Host:
    """mlora._host as far as Lora_GPU uses it; a delta says which call made it, and from which plan."""
    def __init__(self):
        self.at, self.calls, self.lock = (0, 0, 0, 0), [], threading.Lock()

    def order(self):
        return (threading.get_ident(),) + self.at[1:]

    def state(self, x, weights):
        return self.order() + tuple((id(t), t._version) for t in (x, *weights))

    def deltas_ref(self, plan, x, weights, layer, T, N, L, r):
        with self.lock:
            made = len(self.calls)
            self.calls.append((plan, plan.indicies, layer))
        return tuple(torch.tensor([made, i]) for i in range(3))


@pytest.fixture
def gpu(monkeypatch):
    host = _Host()

    def plan(ids, N, L, r, group=None, out=None):
        if out is not None:
            out.indicies = ids
            return out
        return ops.RefDecodePlan(ids, 1, N, L, r, torch.zeros(1, dtype=torch.uint8))
    monkeypatch.setattr(_ext, "host", lambda: host)
    monkeypatch.setattr(ops, "plan_decode_ref", plan)
    g = Lora_GPU(dict(n_layers=2, batch_size=4, lora_rank=8, hidden_dim=16, tp_degree=1, max_prefill_batch_size=1), device="cpu")
    return g, host


@pytest.mark.parametrize("elsewhere", [(0, 1, 0, 0), (0, 0, 7, 0), (0, 0, 0, 3)], ids=["device", "stream", "capture"])
@pytest.mark.parametrize("planned", [False, True])
def test_a_call_elsewhere_is_computed_there(gpu, planned, elsewhere):
    """k on another stream, or in a graph capture that q was not part of: nothing orders it behind q's launches."""
    g, host = gpu
    x, ids = torch.zeros(3, 16, dtype=torch.float16), torch.tensor([0, 1, 2])
    if planned:
        g.plan_decode(3, ids)
    q = g.invoke_one_layer_q(x, 0, False, lora_ids=ids)
    k = g.invoke_one_layer_k(x, 0, False, lora_ids=ids)
    assert len(host.calls) == 1 and q.tolist() == [0, 0] and k.tolist() == [0, 1]
    host.at = elsewhere
    v = g.invoke_one_layer_v(x, 0, False, lora_ids=ids)
    assert len(host.calls) == 2 and v.tolist() == [1, 2]
    # a plan of plan_decode serves wherever the program orders its calls behind it; one made by the way is not shared
    assert (host.calls[0][0] is host.calls[1][0]) == planned
    host.at = (0, 0, 0, 0)
    assert g.invoke_one_layer_q(x, 0, False, lora_ids=ids).tolist() == [2, 0]


def test_steps_in_order_share_their_plan_buffers(gpu):
    g, host = gpu
    x = torch.zeros(3, 16, dtype=torch.float16)
    for step in range(3):
        ids = torch.tensor([step, 0, 0])
        for layer in range(2):
            for name in "qkv":
                getattr(g, f"invoke_one_layer_{name}")(x, layer, False, lora_ids=ids)
    assert len(host.calls) == 6 and all(c[0] is host.calls[0][0] for c in host.calls)


def test_threads_get_results_of_their_own_input(gpu):
    """Four threads on one object, each with its own input, ids and layer, each call between other threads' calls."""
    g, host = gpu
    gate, bad = threading.Barrier(4, timeout=60), []

    def run(j):
        x, ids = torch.zeros(3, 16, dtype=torch.float16), torch.tensor([j, j, j])
        for _ in range(50):
            for i, name in enumerate("qkv"):
                gate.wait()
                y = getattr(g, f"invoke_one_layer_{name}")(x, j % 2, False, lora_ids=ids)
                made, which = y.tolist()
                if which != i or host.calls[made][2] != j % 2 or host.calls[made][1].tolist() != [j, j, j]:
                    bad.append((j, name, made))
    threads = [threading.Thread(target=run, args=(j,)) for j in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad


def test_a_prefill_workspace_serves_one_stream_and_one_capture(gpu, monkeypatch):
    g, host = gpu
    g.prepare_lora_prefill(2)
    used = []
    monkeypatch.setattr(ops, "sgmv_workspace", lambda rows, reqs, device: torch.empty(rows * 10 + reqs))
    monkeypatch.setattr(ops, "lora_prefill_ref", lambda x, down, up, layer, workspace: used.append(workspace))
    call = lambda n, length: g.invoke_one_layer_q(torch.zeros(n, length, 16).half(), 0, True)  # noqa: E731
    call(1, 300), call(1, 250), call(2, 100)
    assert used[0] is used[1] and used[2] is not used[1] and used[2].numel() == 3002     # grows, and covers what it covered before
    for elsewhere in ((0, 0, 7, 0), (0, 0, 7, 2), (0, 0, 7, 0)):
        host.at = elsewhere
        call(1, 50), call(1, 40)
        assert used[-1] is used[-2] and all(used[-1] is not w for w in used[:-2]) and used[-1].numel() == 501
