"""The prefill GEMM's split tiles (csrc/exl3_gemm.hip): tiles of three or more K pieces, whose rows the
pieces' workgroups share out among them, and of two, on an MI355X (-m gpu).

Shapes sit where the sharing can go wrong: one live row tile, live row tiles that the pieces don't
divide, more pieces than row tiles, split tiles behind whole ones, groups, pieces that are not equal; and
with no polls at all (EXL3_GEMM_POLLS=0: every workgroup but the last to land gives up at once).
"""
import os

import pytest
import torch

from exl3rocm import kernels as E

pytestmark = [pytest.mark.gpu,
              pytest.mark.skipif(not torch.cuda.is_available(), reason="needs a GPU")]

CASES = [(1792, [128], 3, 9),                # 3 pieces of 9 steps, one live row tile
         (1792, [256], 6, 33),               # 3 live row tiles
         (17408, [128], 4, 200),             # 34 pieces, 13 live row tiles
         (5120, [1024], 5, 257),             # 16 tiles of 10 pieces, the second row tile with one live
         (6144, [5120], 4, 200),             # 6 pieces
         (5120, [5120, 1024, 1024], 3, 130),  # groups, 4 pieces
         (5120, [10240], 2, 1000),           # 256 whole tiles, then 64 of 4 pieces
         (5120, [5120], 4, 700),             # 2 pieces
         (5120, [17408], 4, 200)]            # 2 unequal pieces


def make(k, widths, bits, m):
    g = torch.Generator(device="cuda").manual_seed(k + sum(widths) + m)
    T = [torch.randint(-2 ** 31, 2 ** 31, (k // 16, n // 16, 8 * bits), device="cuda", dtype=torch.int32, generator=g).view(torch.int16)
         for n in widths]
    su = [torch.randn(k, device="cuda", generator=g).sign().half() for _ in widths]
    sv = [(torch.randn(n, device="cuda", generator=g).sign() * k ** -0.5).half() for n in widths]
    return torch.randn(m, k, device="cuda", generator=g).half(), T, su, sv


def gemm(x, T, su, sv, bits, y=None):
    m, k = x.shape
    if y is None:
        y = torch.empty(m, sum(s.shape[0] for s in sv), dtype=torch.float16, device="cuda")
    E.exl3_gemm_trellis_grouped(x, T, y, su, torch.empty(len(T), m, k, dtype=torch.float16, device="cuda"), sv, bits, False, True)
    return y


def head():
    """The workspace's counters."""
    return E.prefill_workspace(torch.device("cuda", torch.cuda.current_device()), 1)[:4096]


@pytest.mark.parametrize("k,widths,bits,m", CASES)
def test_split_tiles(monkeypatch, k, widths, bits, m):
    monkeypatch.setenv("EXL3_GEMM_KERNEL", "pc")
    x, T, su, sv = make(k, widths, bits, m)
    print(f"split tiles k={k} n={widths} bits={bits} m={m}", flush=True)
    y = gemm(x, T, su, sv, bits)
    torch.cuda.synchronize()
    assert not bool(head().any())                          # every counter zero again
    # without a workspace no tile is split: the same products, another order of the float32 sums.  An
    # fp16 rounding of C (half an ulp, 2^-12 of its value rms at most) may fall the other way, and one
    # of the output: rel-L2 below 2^-11
    n0 = 0
    for t, u, v in zip(T, su, sv):
        want = torch.empty(m, v.shape[0], dtype=torch.float16, device="cuda")
        E.exl3_gemm_trellis(x, t, want, u, torch.empty(m, k, dtype=torch.float16, device="cuda"), v, bits, False, True)
        got = y[:, n0:n0 + v.shape[0]].double()
        assert (got - want.double()).norm() <= 2.0 ** -11 * want.double().norm(), (k, widths, bits, m)
        n0 += v.shape[0]
    # whoever sums a row tile, in whatever order the pieces land: the same bits
    for polls in (None, "0"):
        if polls is not None:
            monkeypatch.setenv("EXL3_GEMM_POLLS", polls)
        for _ in range(3):
            again = gemm(x, T, su, sv, bits)
            torch.cuda.synchronize()
            assert torch.equal(again.view(torch.int16), y.view(torch.int16)), polls
            assert not bool(head().any()), polls


def test_split_tiles_on_two_streams_and_in_a_graph(monkeypatch):
    """Launches that wait for their own pieces, on two streams at once, and replayed from a graph."""
    monkeypatch.setenv("EXL3_GEMM_KERNEL", "pc")
    sides = [(torch.cuda.Stream(), make(6144, [5120], 4, 200)), (torch.cuda.Stream(), make(5120, [10240], 4, 300))]
    want = [gemm(*a, 4) for _, a in sides]
    outs = [torch.empty_like(w) for w in want]
    torch.cuda.synchronize()
    for _ in range(10):
        for (s, a), y in zip(sides, outs):
            with torch.cuda.stream(s):
                gemm(*a, 4, y)
    torch.cuda.synchronize()
    for y, w in zip(outs, want):
        assert torch.equal(y.view(torch.int16), w.view(torch.int16))
    s, a = sides[0]
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=s):
        y = gemm(*a, 4)
    for _ in range(3):
        y.zero_()
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(y.view(torch.int16), want[0].view(torch.int16))
        gemm(*sides[1][1], 4)
        torch.cuda.synchronize()
