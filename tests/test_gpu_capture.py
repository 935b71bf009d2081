"""Graph capture at more rows than a stream was warmed up with, on an MI355X (-m gpu)."""
import numpy as np
import pytest
import torch

from exl3rocm import kernels as E, ops, plugin, synth

pytestmark = [pytest.mark.gpu,
              pytest.mark.skipif(not torch.cuda.is_available(), reason="needs a GPU")]

K_IN, N, BITS = 5120, 5120, 4


def same(a, b):
    return torch.equal(a.view(torch.int16), b.view(torch.int16))


def capture(s, op):
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=s):
        y = op()
    return g, y


@pytest.fixture
def default_routes(monkeypatch):
    if ops.MR_MAX is not None or ops.PREFILL_ROUTE != "fused" or ops.GEMM_KERNEL or ops.GEMV_APPROX:
        pytest.skip("a knob chooses the route")


@pytest.mark.parametrize("m", [16, 48])
def test_layer_warmed_with_one_row(m, default_routes):
    """Load, one eager row on stream S, capture m rows on S: what an eager call of m rows gives, bitwise."""
    method = plugin.Exl3LinearMethod(plugin.Exl3Config("mul1"), [("o", BITS, K_IN, N)])
    layer = torch.nn.Module()
    method.create_weights(layer, K_IN, [N], K_IN, N, torch.float16)
    layer.to("cuda")
    tr, su, sv = synth.layer("capture", 0, K_IN, N, BITS)
    for name, w in (("trellis", tr.view(np.int16)), ("suh", su), ("svh", sv)):
        target = getattr(layer, name)
        target.weight_loader(target, torch.from_numpy(w))
    layer.mul1.weight_loader(layer.mul1, torch.tensor(0x83DCD12D - 2 ** 32))
    method.process_weights_after_loading(layer)
    x = torch.from_numpy(synth.activations(synth.key_of("capture", "x", m), m, K_IN)).cuda()
    want = method.apply(layer, x)
    torch.cuda.synchronize()
    s = torch.cuda.Stream()
    with torch.cuda.stream(s):
        method.apply(layer, x[:1])
    s.synchronize()
    g, y = capture(s, lambda: method.apply(layer, x))
    for _ in range(3):
        y.zero_()
        torch.cuda.synchronize()
        g.replay()
        torch.cuda.synchronize()
        assert same(y, want)
        method.apply(layer, x)
        torch.cuda.synchronize()


@pytest.mark.parametrize("m", [9, 16])
def test_stream_with_the_gemv_workspace_only(m, monkeypatch, default_routes):
    """No layer has reserved anything: a capture at m rows on a stream that has the GEMV's workspace records the
    GEMV, as it does for the rows that were warmed up; on one that has none it is refused."""
    monkeypatch.setattr(E, "_pf_reserved", set())
    tr, su, sv = synth.layer("capture", 1, K_IN, N, BITS)
    t, su, sv = (torch.from_numpy(a).cuda() for a in (tr.view(np.int16), su, sv))
    x = torch.from_numpy(synth.activations(synth.key_of("capture", "x", m), m, K_IN)).cuda()
    want = torch.empty(m, N, dtype=torch.float16, device="cuda")
    assert E.exl3_gemv_mr(x, t, want, su, None, sv, BITS, False, True) == 0
    torch.cuda.synchronize()
    s = torch.cuda.Stream()
    monkeypatch.setattr(E, "_pf_workspaces", {})
    with torch.cuda.stream(s):
        ops.reserve_workspace(x.device, K_IN, N, BITS, m=m)
        torch.ops.exl3rocm.linear(x[:1], t, su, sv, BITS, False, True)
    s.synchronize()
    assert not E._pf_workspaces
    g, y = capture(s, lambda: torch.ops.exl3rocm.linear(x, t, su, sv, BITS, False, True))
    for _ in range(3):
        y.zero_()
        torch.cuda.synchronize()
        g.replay()
        torch.cuda.synchronize()
        assert same(y, want)
    monkeypatch.setattr(E, "_workspaces", {})
    with pytest.raises(RuntimeError, match="before graph capture"):
        capture(torch.cuda.Stream(), lambda: torch.ops.exl3rocm.linear(x, t, su, sv, BITS, False, True))
    torch.cuda.synchronize()
