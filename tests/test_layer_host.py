"""What SimpleMoE's forward and backward do on the host around their native
calls, with the native calls recorded instead of made: the streams are joined
when a step after the call fails."""
import pytest
import torch

import smoe
from smoe import _C, layer, ops

T, H, I, E, K = 8, 256, 128, 8, 2


class FakeStream:
    cuda_stream, device = 0, torch.device("cpu")

    def __init__(self, log):
        self.log = log

    def wait_stream(self, other):
        self.log.append(("wait", self, other))


@pytest.fixture
def host(monkeypatch):
    """(calls, main stream): the layer on CPU tensors, native calls recorded."""
    calls = []
    main = FakeStream(calls)
    monkeypatch.setattr(ops, "_check", lambda *a, **k: None)
    monkeypatch.setattr(ops, "_stream", lambda: 0)
    monkeypatch.setattr(_C, "call", lambda name, *a: calls.append(name))
    monkeypatch.setattr(ops, "_status_workspace", lambda n, dev: torch.empty(n, dtype=torch.uint8))
    monkeypatch.setattr(torch.cuda, "current_stream", lambda *a: main)
    monkeypatch.setattr(layer.SimpleMoE, "_side_stream", lambda self, device: FakeStream(calls))
    return calls, main


def module(E=E, I=I, H=H):
    m = smoe.SimpleMoE(H, I, E, K, device="cpu")
    set_weights(m, E, I, H)
    return m


def set_weights(m, E, I, H):
    """Unquantised stand-ins of the layer's fp8 weights (only shapes matter)."""
    w = lambda *s: torch.zeros(s, dtype=torch.uint8)
    s = lambda e, n, k: torch.ones(e, ops.nblocks(n), ops.nblocks(k))
    Hp, Ip, Np = ops.pad128(H), ops.pad128(I), ops.pad128(2 * I)
    m._fp8 = m._gemm = (w(E, 2 * I, Hp), s(E, 2 * I, H), w(E, H, Ip), s(E, H, I))
    m._gemm_t = (w(E, H, Np), s(E, H, 2 * I), w(E, I, Hp), s(E, I, H))
    m._fp8_key = m._weights_key()


def intermediates(m):
    with torch.no_grad():
        return m(torch.zeros(T, H, dtype=torch.bfloat16), torch.zeros(T, E), return_intermediates=True)[1]


def test_streams_are_joined_when_the_gate_gradient_fails(host):
    """The backward leaves the join to its gating-linear gradients; an error
    there (out of memory, say) must not free memory the side stream still uses."""
    calls, main = host
    m = module()
    st = dict(intermediates(m), logits_from_gate=True)
    m.w_gate = torch.nn.Parameter(torch.zeros(3, 5))  # the product below raises
    with pytest.raises(RuntimeError):
        m.backward_from(st, torch.zeros(T, H, dtype=torch.bfloat16))
    assert calls[-2] == "smoe_layer_backward" and calls[-1][:2] == ("wait", main)


@pytest.mark.parametrize("change", [
    dict(E=4), dict(I=64), dict(H=128),                       # all weights of another layer
    dict(w1=(E, 2 * I, 128)), dict(w1=(E - 1, 2 * I, H)),     # one tensor that does not fit the rest
    dict(w2=(E, H, 256)), dict(w2=(E - 1, H, I))])
@pytest.mark.parametrize("save", [False, True])
def test_forward_never_runs_on_weights_of_other_shapes(host, change, save):
    """The native call takes the sizes as numbers: it is made only with
    weights of exactly those shapes.  Weights a caller replaced by others run
    with their own sizes or are refused, as the operators did."""
    calls, _ = host
    m = module()
    set_weights(m, change.get("E", E), change.get("I", I), change.get("H", H))
    w1, w1s, w2, w2s = m._gemm
    w1 = torch.zeros(change.get("w1", w1.shape), dtype=torch.uint8)
    w2 = torch.zeros(change.get("w2", w2.shape), dtype=torch.uint8)
    m._fp8 = m._gemm = (w1, w1s, w2, w2s)
    x, logits = torch.zeros(T, H, dtype=torch.bfloat16), torch.zeros(T, E)
    if change == dict(I=64):  # a consistent layer of another width: runs, with its own sizes
        with torch.no_grad():
            out = m(x, logits, return_intermediates=save)
        if save:
            assert out[1]["c1"].shape == (T * K, 128) and out[1]["hq"].shape == (T * K, 128)
        return
    with pytest.raises(ValueError), torch.no_grad():
        m(x, logits, return_intermediates=save)
    assert "smoe_layer_forward" not in calls


def test_forward_takes_the_sizes_of_replaced_weights(host):
    """Experts dropped from all three parameters, as a pruned layer has it."""
    calls, _ = host
    m = module()
    set_weights(m, 4, I, H)
    with torch.no_grad():
        _, st = m(torch.zeros(T, H, dtype=torch.bfloat16), torch.zeros(T, 4), return_intermediates=True)
    assert st["offsets"].shape == (5,) and calls == ["smoe_layer_forward"]


@pytest.mark.parametrize("t", range(4))
def test_backward_never_runs_on_weights_of_other_shapes(host, t):
    calls, _ = host
    m = module()
    st = intermediates(m)
    bad = list(m._gemm_t)
    bad[t] = torch.zeros([n - 1 for n in bad[t].shape], dtype=bad[t].dtype)
    m._gemm_t = tuple(bad)
    with pytest.raises(ValueError):
        m.backward_from(st, torch.zeros(T, H, dtype=torch.bfloat16))
    assert "smoe_layer_backward" not in calls


def test_backward_refuses_other_gradient_types(host):
    m = module()
    with pytest.raises(TypeError):
        m.backward_from(intermediates(m), torch.zeros(T, H, dtype=torch.bfloat16), wgrad_dtype=torch.float16)
