"""The register-decode GEMM (csrc/exl3_gemm_rd.hip): its unit split and its completion protocol on the
CPU, its numbers against the oracle on an MI355X (-m gpu).

GPU cases sit where the kernel can go wrong: row counts at the edges of its 32-row tiles and of the
exact-transform range (64), every bitrate and codebook, launches of a few units, pieces that cross
tiles and pieces that do not, groups of different widths, row-strided operands, the SiLU input.
"""
import ctypes
import os

import numpy as np
import pytest
import torch

import cpu
import isa_waits as W
from exl3rocm import _lib, kernels as E, ops, synth

REPO = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LIB = os.path.join(REPO, "qwen38-27b-exl3-rdna4_amd", "exl3rocm", "libexl3_mi355x.so")
gpu = pytest.mark.gpu
needs_gpu = pytest.mark.skipif(not torch.cuda.is_available(), reason="needs a GPU")


def check(m, k, widths):
    return _lib.lib().exl3_gemm_rd_check(m, k, (ctypes.c_int * len(widths))(*widths), len(widths))


@pytest.mark.parametrize("widths", [[128], [1024], [5120], [5120, 1024, 1024], [17408], [17408, 17408], [12288, 128, 256],
                                    [128 * 255], [128 * 256], [128 * 257, 128], [248320]])
@pytest.mark.parametrize("k", [2048, 2304, 5120, 17408])
def test_unit_split(k, widths):
    """Every unit has one workgroup and every tile's contributors are the formulas'."""
    for m in (1, 33, 128):
        assert check(m, k, widths) == 0, (m, k, widths)


def test_shapes_not_served():
    assert check(129, 5120, [5120]) == -1 and check(64, 1792, [5120]) == -1 and check(64, 5120 + 128, [5120]) == -1
    assert check(64, 5120, [100]) == -1 and check(64, 5120, [128 * 4097]) == -1 and check(0, 5120, [128]) == -1


@pytest.mark.parametrize("m", [33, 64, 128])
def test_input_range(m):
    """The rotated input's byte offsets have 32 bits: m * k * 2 stays below 2^31 (the prefill GEMM's 64-bit
    kernel takes what is larger)."""
    k = ((1 << 30) - 1) // m // 256 * 256                          # the largest k of that many rows
    assert check(m, k, [128]) == 0 and check(m, k + 256, [128]) == -1
    assert check(m, 1 << 25, [128]) == -1


def test_workspace_max_holds_every_plan():
    lib = _lib.lib()
    assert lib.exl3_gemm_trellis_workspace_max() == lib.exl3_gemm_trellis_workspace_bound() + 4 * 4096
    # at most 256 workgroups (and one more for each small group of a launch of many tiles), two partial
    # tiles of 128 x 128 floats each
    assert 4096 + (256 + 3) * 2 * 128 * 128 * 4 <= lib.exl3_gemm_trellis_workspace_bound()


def test_completion_protocol():
    """The rules of test_completion_protocol.py on every instantiation: stores carry sc1, partials
    have landed before the count, loads after it carry sc1."""
    if not os.path.exists(f"{W.LLVM}/llvm-objdump"):
        pytest.skip("ROCm llvm tools not installed")
    rep = W.protocol_report(LIB, kinds=("gemm_rd_kernel",))
    assert len(rep) == 8 * 3 * 4                                  # bits x codebooks x row tiles
    for name, r in rep.items():
        assert r.atomics >= 1 and r.loads_after >= 1 and r.stores >= 2, name
    assert not {n: r.violations[:3] for n, r in rep.items() if r.violations}


# ---------------------------------------------------------------------------------------------- GPU
def module(tag, k, widths, bits, m):
    mats = [synth.layer(tag, i, k, n, bits) for i, n in enumerate(widths)]
    x = synth.activations(synth.key_of(tag, "x", m), m, k, heavy_tail=True)
    dev = [[torch.from_numpy(a).cuda() for a in (t.view(np.int16), su, sv)] for t, su, sv in mats]
    return x, mats, torch.from_numpy(x).cuda(), [list(c) for c in zip(*dev)]


def grouped(X, T, SU, SV, bits, cb):
    m, k = X.shape
    y = torch.full((m, sum(s.shape[0] for s in SV)), float("nan"), dtype=torch.float16, device="cuda")
    E.exl3_gemm_trellis_grouped(X, T, y, SU, torch.empty(len(T), m, k, dtype=torch.float16, device="cuda"), SV, bits,
                                cb == 1, cb == 2)
    return y


def assert_close(got, ref, what):
    """The repository's parity bar (test_gpu_parity.assert_close): rel-L2 1e-3, and each element within
    four fp16 steps of the output's scale."""
    from test_gpu_parity import assert_close as bar
    bar(got, ref, what)


CASES = [  # m, k, widths, bits, cb
    (9, 5120, [5120], 4, 2), (31, 2048, [128], 1, 0), (32, 2304, [384], 2, 1), (33, 2048, [256, 128], 3, 2),
    (63, 4096, [512], 5, 0), (64, 5120, [1024, 1024], 6, 1), (65, 2560, [640], 7, 2), (96, 3072, [256], 8, 0),
    (97, 2048, [1024, 128, 128], 4, 1), (127, 5120, [256], 3, 0), (128, 2048, [384], 8, 2), (1, 2048, [256], 5, 1),
    (40, 2048, [128 * 260], 2, 2),          # more tiles than workgroups: pieces cross tiles, next to whole tiles
    (100, 5120, [17408], 4, 2),             # 136 tiles in 256 pieces that cross them
    (48, 17408, [768], 3, 2),
]


@gpu
@needs_gpu
@pytest.mark.parametrize("m,k,widths,bits,cb", CASES, ids=[f"m{c[0]}-k{c[1]}-n{'+'.join(map(str, c[2]))}-K{c[3]}-cb{c[4]}" for c in CASES])
def test_against_the_oracle(m, k, widths, bits, cb):
    print(f"register-decode m={m} k={k} widths={widths} bits={bits} cb={cb}", flush=True)
    assert check(m, k, widths) == 0
    x, mats, X, (T, SU, SV) = module(f"rd{k}x{sum(widths)}", k, widths, bits, m)
    y, again = grouped(X, T, SU, SV, bits, cb), grouped(X, T, SU, SV, bits, cb)
    torch.cuda.synchronize()
    assert torch.equal(y.view(torch.int16), again.view(torch.int16))      # deterministic, counters left zero
    rows = sorted({0, m // 2, min(m - 1, 31), min(m - 1, 32), m - 1})
    n0 = 0
    for (tr, su, sv), n in zip(mats, widths):
        assert_close(y[rows, n0:n0 + n].cpu().numpy(), cpu.linear(x[rows], tr, bits, su, sv, cb), (m, k, n0))
        n0 += n


def segments(tiles, upt, G=256):
    """Each workgroup's segments where pieces cross tiles: [(tile, whole)], of an even share of the units."""
    out = []
    for c in range(G):
        u, end, seg = tiles * upt * c // G, tiles * upt * (c + 1) // G, []
        while u < end:
            t = u // upt
            stop = min(end, (t + 1) * upt)
            seg.append((t, u == t * upt and stop == (t + 1) * upt))
            u = stop
        out.append(seg)
    return out


WIDE = 700                                                        # tiles of 8 units in 256 workgroups


def test_wide_launch_has_every_segment_order():
    """What the next test runs: a shared first tile, one or two whole tiles, a shared last one, and each of
    these orders without its first or last."""
    orders = {"".join("W" if w else "P" for _, w in seg) for seg in segments(WIDE, 8)}
    assert orders == {"WWP", "PWP", "PWWP", "PWW"}
    assert check(20, 2048, [128 * WIDE]) == 0


@gpu
@needs_gpu
@pytest.mark.parametrize("m", [20, 40, 80, 128])                  # one case for each count of row tiles
def test_whole_tiles_between_shared_ones(m):
    """Every tile of a launch of 700 against the unsplit prefill GEMM, and the tiles of workgroups that
    have whole tiles between shared ones against the oracle."""
    k, n, bits, cb = 2048, 128 * WIDE, 1, 2
    print(f"register-decode whole tiles between m={m}", flush=True)
    x, mats, X, (T, SU, SV) = module("rd-wide", k, [n], bits, m)
    y, again = grouped(X, T, SU, SV, bits, cb), grouped(X, T, SU, SV, bits, cb)
    want = torch.empty_like(y)
    E.exl3_gemm_trellis(X, T[0], want, SU[0], torch.empty_like(X), SV[0], bits, False, True)
    torch.cuda.synchronize()
    assert torch.equal(y.view(torch.int16), again.view(torch.int16))
    # two routes, each within the bar (rel-L2 1e-3) of the oracle: 2e-3 of each other, tile by tile
    d, w = ((v.double().view(m, WIDE, 128) ** 2).sum((0, 2)).sqrt() for v in (y.double() - want.double(), want))
    assert bool((d <= 2e-3 * w).all()), [int(t) for t in (~(d <= 2e-3 * w)).nonzero()[:8]]
    tr, su, sv = mats[0]
    rows = sorted({0, min(m - 1, 31), min(m - 1, 32), m - 1})
    for seg in [g for g in segments(WIDE, 8) if len(g) >= 3][::80]:
        c0, c1 = 128 * seg[0][0], 128 * (seg[-1][0] + 1)
        ref = cpu.linear(x[rows], np.ascontiguousarray(tr[:, c0 // 16:c1 // 16]), bits, su, np.ascontiguousarray(sv[c0:c1]), cb)
        assert_close(y[rows, c0:c1].cpu().numpy(), ref, (m, seg))


@gpu
@needs_gpu
def test_rows_do_not_interact_and_strides():
    """Every row of a 70-row call with NaN and infinite rows among the others equals its row of a clean
    call; row-strided input and output slices equal contiguous ones, with nothing written outside."""
    m, k, n, bits = 70, 2048, 384, 4
    x, mats, X, (T, SU, SV) = module("rd-rows", k, [n], bits, m)
    y = grouped(X, T, SU, SV, bits, 2)
    bad = X.clone()
    bad[5], bad[40], bad[69] = float("nan"), float("inf"), 65504.0
    yb = grouped(bad, T, SU, SV, bits, 2)
    keep = [r for r in range(m) if r not in (5, 40, 69)]
    assert torch.equal(y[keep].view(torch.int16), yb[keep].view(torch.int16))
    assert bool(torch.isnan(yb[5]).all()) and not bool(torch.isfinite(yb[40]).any())
    wide = torch.full((m, k + 72), 7.0, dtype=torch.float16, device="cuda")
    wide[:, 8:8 + k] = X
    out = torch.full((m, n + 64), 7.0, dtype=torch.float16, device="cuda")
    E.exl3_gemm_trellis_grouped(wide[:, 8:8 + k], T, out[:, 32:32 + n], SU, torch.empty(1, m, k, dtype=torch.float16, device="cuda"), SV,
                                bits, False, True)
    torch.cuda.synchronize()
    assert torch.equal(out[:, 32:32 + n].contiguous().view(torch.int16), y.view(torch.int16))
    assert bool((out[:, :32] == 7.0).all()) and bool((out[:, 32 + n:] == 7.0).all())


@gpu
@needs_gpu
def test_rows_are_the_same_in_every_batch():
    """A row's bits do not depend on the batch: up to 64 rows (exact transforms), and from 65 (float32 ones).
    The split of the work is by shape alone and every row is summed in the same order."""
    k, widths, bits = 5120, [640, 128], 4
    x, mats, X, (T, SU, SV) = module("rd-batch", k, widths, bits, 128)
    y64, y128 = grouped(X[:64], T, SU, SV, bits, 2), grouped(X, T, SU, SV, bits, 2)
    for m in (1, 9, 32, 33):
        assert torch.equal(grouped(X[:m], T, SU, SV, bits, 2).view(torch.int16), y64[:m].view(torch.int16)), m
    for m in (65, 97):
        assert torch.equal(grouped(X[:m], T, SU, SV, bits, 2).view(torch.int16), y128[:m].view(torch.int16)), m


@gpu
@needs_gpu
@pytest.mark.parametrize("m", [20, 90])
def test_silu_input_and_graph_replays(m):
    """The SiLU-input form equals silu_mul and the plain form bitwise; replays of a captured call equal
    the eager one, eager work between them."""
    if ops.PREFILL_ROUTE != "fused" or ops.GEMM_KERNEL or ops.MR_MAX is not None:
        pytest.skip("a knob chooses the route")
    k, n, bits = 4096, 768, 4
    x, mats, X, (T, SU, SV) = module("rd-silu", k, [n], bits, m)
    gu = torch.cat([X, X.flip(0)], 1).contiguous()
    act = torch.empty(m, k, dtype=torch.float16, device="cuda")
    E.silu_mul(gu[:, :k], gu[:, k:], act)
    want = grouped(act, T, SU, SV, bits, 2)

    def op():
        return torch.ops.exl3rocm.silu_mul_linear(gu, T[0], SU[0], SV[0], bits, False, True)

    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        eager = op()
    s.synchronize()
    assert torch.equal(eager.view(torch.int16), want.view(torch.int16))
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=s):
        y = op()
    for _ in range(3):
        y.zero_()
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(y.view(torch.int16), want.view(torch.int16))
        grouped(act, T, SU, SV, bits, 2)
        torch.cuda.synchronize()
