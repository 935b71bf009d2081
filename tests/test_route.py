"""The route of a launch (GEMV, register-decode GEMM, prefill GEMM), on the CPU: the GEMV keeps its boundary
against the prefill GEMM wherever the register-decode GEMM is not what the other route runs."""
import ctypes

import pytest
import torch

from exl3rocm import _lib, ops
from test_host import _Launches

CHECKPOINT = sorted(ops.GEMV_CROSSOVER)


def serves(m, k, widths, K, ldy=None):
    return _lib.lib().exl3_gemm_rd_serves(m, k, (ctypes.c_int * len(widths))(*widths), len(widths), K, ldy or sum(widths))


@pytest.fixture(autouse=True)
def defaults(monkeypatch):
    for name, value in (("MR_MAX", None), ("PREFILL_ROUTE", "fused"), ("GEMM_KERNEL", ""), ("GEMV_APPROX", ""), ("GATED_ROUTE", "unfused")):
        monkeypatch.setattr(ops, name, value)


def test_boundaries():
    """No boundary below MID_MR (the ops ask nothing at those rows), none against the prefill GEMM
    below the one against the register-decode GEMM, which starts to win earlier."""
    assert sorted(ops.PREFILL_CROSSOVER) == CHECKPOINT
    for s in CHECKPOINT:
        assert ops.MID_MR <= ops.GEMV_CROSSOVER[s] <= ops.PREFILL_CROSSOVER[s] <= _lib.GEMV_MAX_ROWS
    assert ops.MID_MR <= ops.DEFAULT_MR


def test_small_launches():
    """Launches of at most 2^24 weights that the register-decode GEMM does not speed up keep the GEMV's
    first 16-row tile; neighbours on each side of the rule do not."""
    for k, w, K in ((4096, 4096, 6), (4096, 4096, 5), (3072, 128, 4), (8192, 1024, 1), (5120, 1024, 4), (5120, 2048, 4), (3072, 5376, 8)):
        assert ops.gemv_max_rows(k, w, K) == 16, (k, w, K)
    for k, w, K in ((4096, 4096, 4), (4096, 4224, 6), (3072, 1152, 4), (8448, 1024, 8), (12288, 128, 4), (5120, 5120, 8)):
        assert ops.gemv_max_rows(k, w, K) == 8, (k, w, K)
    for k, w in ((2048, 2048), (3072 + 128, 1024), (2816, 128)):
        assert ops.gemv_max_rows(k, w, 8) == ops.DEFAULT_MR
    assert ops.gemv_rows(16, 4096, 4096, 6) and not ops.gemv_rows(17, 4096, 4096, 6)


@pytest.mark.parametrize("knob,value", [("PREFILL_ROUTE", "recon"), ("GEMM_KERNEL", "tile"), ("GEMM_KERNEL", "pc")])
def test_knobs_that_take_another_gemm(monkeypatch, knob, value):
    """EXL3_PREFILL=recon rebuilds the whole weight on each call and EXL3_GEMM_KERNEL takes the prefill's
    kernels: the GEMV's rows end where those begin to win."""
    monkeypatch.setattr(ops, knob, value)
    for (k, w), b in ops.PREFILL_CROSSOVER.items():
        assert ops.gemv_rows(b, k, w) and not ops.gemv_rows(b + 1, k, w), (k, w)
    assert ops.gemv_rows(32, 4096, 4096) and not ops.gemv_rows(33, 4096, 4096)
    assert ops.fused_rows(30, 6144, 5120) and not ops.fused_rows(31, 6144, 5120) and not ops.fused_rows(33, 17408, 5120)


@pytest.mark.parametrize("k,widths,K,ldy", [(8192, (262144,), 8, None),         # a trellis of 2 GiB
                                            (8192, (262144, 128), 8, None),
                                            (5120, (128 * 4097,), 1, None),     # more tiles than counters
                                            (4096, (4096,), 4, 1 << 24),        # output rows too far apart
                                            (1 << 24, (128,), 1, None)])        # 64 rows of input: 2 GiB
def test_launches_beyond_the_register_decode_gemm(k, widths, K, ldy):
    w = sum(widths)
    assert not serves(64, k, widths, K, ldy)
    for m in (9, 16, 32):
        assert ops.gemv_rows(m, k, w, K, widths, ldy), m
    assert not ops.gemv_rows(33, k, w, K, widths, ldy)


def test_serves_fewer_rows_too():
    """The boundary asks at the GEMV's most rows: what is served there is served at fewer."""
    for k, widths, K in ((5120, (5120,), 4), (5120, (248320,), 4), (3072, (128,), 1), (17408, (128 * 300, 128), 8), (2048, (128 * 4096,), 2)):
        assert serves(64, k, widths, K)
        assert all(serves(m, k, widths, K) for m in range(1, 64))
    assert not serves(0, 5120, (5120,), 4) and not serves(129, 5120, (5120,), 4) and not serves(64, 5120, (5120,), 9)
    assert not serves(64, 5120, (100,), 4)


def launches(monkeypatch, widths, Ks, m, k=5120):
    rec = _Launches()
    monkeypatch.setattr(ops, "E", rec)
    monkeypatch.setattr(ops, "_weight_buffer", lambda dev, n: torch.empty(n, dtype=torch.float16))
    tr = [torch.zeros(k // 16, n // 16, 16 * K, dtype=torch.int16) for n, K in zip(widths, Ks)]
    su = [torch.ones(k, dtype=torch.float16)] * len(widths)
    sv = [torch.ones(n, dtype=torch.float16) for n in widths]
    y = torch.ops.exl3rocm.linear_groups(torch.zeros(m, k, dtype=torch.float16), tr, su, sv, list(Ks), False, True)
    assert tuple(y.shape) == (m, sum(widths))
    return [name for name, _ in rec.calls]


def test_groups_under_recon(monkeypatch):
    monkeypatch.setattr(ops, "PREFILL_ROUTE", "recon")
    assert launches(monkeypatch, (1024, 1024), (5, 5), 40) == ["exl3_gemv_mr_grouped"]
    monkeypatch.setattr(ops, "PREFILL_ROUTE", "fused")
    assert launches(monkeypatch, (1024, 1024), (5, 5), 40) == ["exl3_gemm_trellis_grouped"]


@pytest.mark.parametrize("m,k,n,approx", [(9, 5120, 17408, True), (32, 5120, 17408, True), (33, 5120, 17408, False),
                                          (17, 5120, 5120, True), (18, 5120, 5120, False), (32, 4096, 4096, True)])
def test_approximate_gemv_keeps_its_rows(monkeypatch, m, k, n, approx):
    """EXL3_GEMV_APPROX: up to 32 rows of the boundary against the prefill GEMM, in every op; mcg and
    3inst modules take the faithful routes."""
    monkeypatch.setattr(ops, "GEMV_APPROX", "affine")
    want = "exl3_gemv_mr_approx" if approx else "exl3_gemm_trellis_grouped"
    assert launches(monkeypatch, (n,), (4,), m, k) == [want]
    rec = _Launches()
    monkeypatch.setattr(ops, "E", rec)
    t, su, sv = torch.zeros(k // 16, n // 16, 64, dtype=torch.int16), torch.ones(k, dtype=torch.float16), torch.ones(n, dtype=torch.float16)
    x = torch.zeros(m, k, dtype=torch.float16)
    torch.ops.exl3rocm.linear(x, t, su, sv, 4, True, False)
    assert rec.calls.pop()[0] == "exl3_gemm_trellis_grouped"
    torch.ops.exl3rocm.linear(x, t, su, sv, 4, False, True)
    assert rec.calls.pop()[0] == want


class _Mlp(_Launches):
    """_Launches for the SiLU forms too, whose arguments lie elsewhere."""

    def __getattr__(self, name):
        def launch(*args, **kw):
            self.calls.append((name, None))
            return 0
        return launch


@pytest.mark.parametrize("m", [9, 30, 31, 32, 33, 40])
def test_silu_input_forms(monkeypatch, m):
    """The down projection: the approximate GEMV forms up to their rows, else the GEMM's SiLU input."""
    k, n = 6144, 5120                                             # boundary against the prefill GEMM: 30
    gu, t = torch.zeros(m, 2 * k, dtype=torch.float16), torch.zeros(k // 16, n // 16, 64, dtype=torch.int16)
    su, sv = torch.ones(k, dtype=torch.float16), torch.ones(n, dtype=torch.float16)
    rec = _Mlp()
    monkeypatch.setattr(ops, "E", rec)
    torch.ops.exl3rocm.silu_mul_linear(gu, t, su, sv, 4, False, True)
    assert [c for c, _ in rec.calls] == ["exl3_gemm_trellis_silu_in"]
    monkeypatch.setattr(ops, "GEMV_APPROX", "affine")
    rec.calls.clear()
    torch.ops.exl3rocm.silu_mul_linear(gu, t, su, sv, 4, False, True)
    assert [c for c, _ in rec.calls] == (["silu_mul", "exl3_gemv_mr_approx"] if m <= 30 else ["exl3_gemm_trellis_silu_in"])


@pytest.mark.parametrize("m", [8, 9, 32, 33])
def test_gated_form_keeps_its_rows(monkeypatch, m):
    """EXL3_GATED=fused: the one-launch form up to 32 rows, and linear_groups of gate and up on the GEMV at
    those rows, whose bits it has; without the knob both take the GEMM from 9 rows."""
    k, n = 5120, 17408
    x, t = torch.zeros(m, k, dtype=torch.float16), torch.zeros(k // 16, n // 16, 64, dtype=torch.int16)
    su, sv = torch.ones(k, dtype=torch.float16), torch.ones(n, dtype=torch.float16)

    def calls(op):
        rec = _Mlp()
        monkeypatch.setattr(ops, "E", rec)
        op(x, [t, t], [su, su], [sv, sv], [4, 4], False, True)
        return [c for c, _ in rec.calls]

    small = "exl3_gemv_mr_grouped" if m <= 8 else "exl3_gemm_trellis_grouped"
    assert calls(torch.ops.exl3rocm.linear_groups) == [small] and calls(torch.ops.exl3rocm.linear_silu_mul) == [small, "silu_mul"]
    monkeypatch.setattr(ops, "GATED_ROUTE", "fused")
    fused = m <= 32
    assert calls(torch.ops.exl3rocm.linear_groups) == (["exl3_gemv_mr_grouped"] if fused else ["exl3_gemm_trellis_grouped"])
    assert calls(torch.ops.exl3rocm.linear_silu_mul) == (["exl3_gemv_silu_mul"] if fused else ["exl3_gemm_trellis_grouped", "silu_mul"])


# ---------------------------------------------------------------------------------- workspaces and capture
from exl3rocm import kernels as E  # noqa: E402

CPU = torch.device("cpu")


@pytest.fixture
def workspaces(monkeypatch):
    """Empty workspace tables, on the CPU."""
    for name, empty in (("_workspaces", {}), ("_reserved", {}), ("_pf_workspaces", {}), ("_pf_reserved", set())):
        monkeypatch.setattr(E, name, empty)
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: False)


def test_first_eager_call_brings_both_workspaces(monkeypatch, workspaces):
    """A layer's reservation at load reaches every stream with its first eager call, whatever its rows; without
    one a small GEMV call allocates its own workspace only."""
    E.workspace(CPU, 100, 6)
    assert list(E._workspaces) == [(CPU, 6)] and not E._pf_workspaces
    E.reserve_prefill_workspace(CPU, 0)
    E.workspace(CPU, 5000, 7)
    assert sorted(s for _, s in E._pf_workspaces) == [0, 7]
    assert all(b.numel() == E.prefill_workspace_bound() for b in E._pf_workspaces.values())
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: True)
    with pytest.raises(RuntimeError):
        E.workspace(CPU, 100, 8)
    assert E.prefill_workspace(CPU, 100, 8) is None and (CPU, 8) not in E._pf_workspaces


@pytest.mark.parametrize("m,gemv", [(8, True), (9, True), (17, True), (18, False)])
def test_capture_without_the_prefill_workspace(monkeypatch, m, gemv):
    """A stream that captures without it keeps the boundary against the prefill GEMM, which is what it would
    record above."""
    k, n = 5120, 5120
    rec = _Mlp()
    rec.captures_without_prefill_workspace = lambda x: True

    class Input:                                                  # _hold's questions to a GPU tensor
        shape, is_cuda = (m, k), True

    monkeypatch.setattr(ops, "E", rec)
    assert ops.gemv_rows(m, k, n, hold=ops._hold(Input, True)) == gemv
    rec.captures_without_prefill_workspace = lambda x: False
    assert ops.gemv_rows(m, k, n, hold=ops._hold(Input, True)) == (m <= 8)


@pytest.mark.parametrize("knobs", [{}, {"MR_MAX": 16}, {"PREFILL_ROUTE": "recon"}, {"GEMM_KERNEL": "pc"}, {"GEMV_APPROX": "affine"}])
@pytest.mark.parametrize("captures", [False, True])
def test_the_ops_question_is_the_rule(monkeypatch, knobs, captures):
    """_gemv, which leaves out what cannot decide a call, against gemv_rows with every question asked."""
    for name, value in knobs.items():
        monkeypatch.setattr(ops, name, value)
    rec = _Mlp()
    rec.captures_without_prefill_workspace = lambda x: captures
    monkeypatch.setattr(ops, "E", rec)
    shapes = CHECKPOINT + [(4096, 4096), (2048, 2048), (512, 512), (3200, 1024), (8192, 262144)]
    for k, w in shapes:
        for m in [*range(1, 66), 128, 2048]:
            x = type("Rows", (), dict(shape=(m, k), is_cuda=True))
            for K in (2, 8):
                for held in (False, True):
                    want = ops.gemv_rows(m, k, w, K, hold=held or ops._hold(x, True))
                    assert ops._gemv(m, x, True, k, w, K, held=held) == want, (m, k, w, K, held)


def test_launches_that_need_no_workspace_allocate_none(workspaces):
    def ws(m, k, widths, K=4, stream=5):
        return E._launch_workspace(CPU, stream, m, k, (ctypes.c_int * len(widths))(*widths), len(widths), K, sum(widths))

    assert ws(300, 512, (512, 384)) is None and ws(2048, 5120, (128 * 256,)) is None and ws(96, 896, (512,)) is None
    assert not E._pf_workspaces
    assert ws(256, 1024, (128 * 260,)) is not None                # a split tail
    first = E._pf_workspaces[(CPU, 5)]
    assert ws(300, 512, (512,)) is first and ws(20, 5120, (5120,)) is first
    assert ws(20, 5120, (5120,), stream=6) is not None and len(E._pf_workspaces) == 2   # the register-decode GEMM
