"""
EXL3 linear on MI355X as opaque torch custom ops, so torch.compile and HIP-graph capture treat
each call as one node.  Same op names, schemas and routing contract as the reference plugin's
ops (vllm_plugin/exl3rocm/ops.py:65-180); kernels come from libexl3_mi355x.so.

One call computes one checkpoint tensor ("group"): y = had(had(x * suh) @ W_inner) * svh.
Routing by rows M, per launch (gemv_rows: the measured GEMV / GEMM crossover of the launch's shape, 8 to
32 rows, or EXL3_MR_MAX rows for every shape when set):
  M <= the crossover     -> fused GEMV (input Hadamard, trellis decode + MFMA dot, split-K
                            reduction and output Hadamard in one launch); every row is bitwise
                            equal to the M == 1 call of that row; EXL3_GEMV_APPROX=affine|int8
                            selects the opt-in approximate mul1 forms (unrounded weights, or
                            int8 activations as the reference's EXL3_ROCM_GFX1201_INT8 path)
  otherwise              -> input Hadamard pass, then a GEMM launch (fp16 MFMA, fp32 accumulate, output
                            Hadamard and svh in its epilogue): up to 128 rows the register-decode GEMM
                            (k from 2048 in multiples of 256), else the prefill GEMM (trellis decoded
                            into LDS);
                            a fused module's groups share one GEMM launch; EXL3_PREFILL=recon takes
                            the reference's reconstruct + hgemm route instead
"""
from __future__ import annotations

import functools
import os
from ctypes import c_int as C_int
from typing import Optional

import torch

from . import _lib
from . import kernels as E

def _env_rows(name: str) -> Optional[int]:
    v = os.environ.get(name)
    return None if v is None or not v.strip() else min(int(v), _lib.GEMV_MAX_ROWS)


# EXL3_MR_MAX (the reference's knob) fixes the GEMV / GEMM boundary for every launch; unset, each launch
# takes a measured crossover of its shape: against the register-decode GEMM (up to 128 rows) where that
# serves the launch, else against the prefill GEMM
MR_MAX: Optional[int] = _env_rows("EXL3_MR_MAX")
# the library's comparison knob; set, the register-decode GEMM is not taken
GEMM_KERNEL = os.environ.get("EXL3_GEMM_KERNEL", "")
DEFAULT_MR = 32
# Largest row count of the fused GEMV where the register-decode GEMM serves the launch, by (k, output columns
# of the launch: all its groups).  The GEMV's cost grows with every row and steps at 17, its second
# 16-row tile; the GEMM's (up to 128 rows) only with each 32-row tile.  Measured on MI355X, GEMV / GEMM in us,
# graphs of 16 launches over cold weights, 4 bpw: 5120 -> 5120 14.4 / 15.1 at 8 rows, 17.4 / 15.1 at 9, 26.5 /
# 15.4 at 20; gate 25.8 / 24.8, 27.3 / 24.7, 36.2 / 26.0; down 24.2 / 25.4, 26.6 / 25.4, 36.5 / 25.6; gate/up
# 38.4 / 37.7, 39.6 / 37.8, 51.8 / 40.9: the layers' launches of a 27B decoder cross at 8 to 9 rows, and
# so do other shapes from 3072 to 17408 inputs and 128 to 17408 columns (MID_MR).
# Where the launch is small the two end within a few us of each other up to the GEMV's step, and a graph
# of this launch alone pays ~2.3 us for the GEMM's second node, so the GEMV keeps its first 16-row tile
# (SMALL_MR: up to 2^24 weights of at most 8192 inputs, and either at most 1024 columns or 5 bpw and more,
# whose pieces take the GEMM longer).  In a graph of 16 / of one launch: 5120 -> 1024 at 4 bpw 13.4 / 14.0 and
# 17.9 / 19.9 at 9 rows, 14.2 / 13.8 and 18.8 / 19.9 at 16, 17.5 / 14.2 and 21.4 / 20.2 at 20; 4096 -> 4096 at 6 bpw
# 17.2 / 15.4 and 21.3 / 21.7 at 9, 17.9 / 15.6 and 22.0 / 21.6 at 16, 21.0 / 16.0 and 25.6 / 22.0 at 20.  The k/v
# pair of 5120 inputs is one of these by the table (15.2 / 14.9 and 19.5 / 20.7 at 10 rows).
# Two boundaries are there for their rows, which are bitwise their one-row calls, and not for speed: lm_head's
# 32 rows (216 / 222 us at 9, 229 / 221 at 16, 300 / 232 at 32), and DEFAULT_MR, the boundary of the library's
# own dispatcher exl3_gemm, below 3072 inputs (2048 -> 2048 11.1 / 11.4 at 9, 16.8 / 11.9 at 32); it is the
# prefill GEMM's too where k is no multiple of 256.
MID_MR, MID_K, SMALL_MR = 8, 3072, 16
GEMV_CROSSOVER = {
    (5120, 1024): 16, (5120, 2048): 16, (5120, 5120): 8, (5120, 6144): 8, (5120, 7168): 8,
    (5120, 10240): 8, (5120, 12288): 8, (5120, 14336): 8, (5120, 16384): 8, (5120, 17408): 8,
    (5120, 34816): 8, (5120, 248320): 32, (6144, 5120): 8, (17408, 5120): 8,
}


def _crossover(k: int, width: int, K: int) -> int:
    b = GEMV_CROSSOVER.get((k, width))
    if b is not None:
        return b
    if k < MID_K or k % 256:
        return DEFAULT_MR
    return SMALL_MR if k * width <= 1 << 24 and k <= 8192 and (width <= 1024 or K >= 5) else MID_MR


# The same against the prefill GEMM (other shapes: DEFAULT_MR), for launches that the register-decode GEMM
# does not serve: both routes at every row count from 2 to 64, graphs of 24 launches over 8 weight
# copies, 4 bpw, and 2 / 3 bpw where a checkpoint holds them (the boundary moved by <= 4 rows).  Each
# entry is within 1 % of the least summed time, with no step above 5 % from the GEMV to the GEMM: the
# prefill GEMM's cost is flat within each 16-row MFMA tile, so it wins early where its 128-column tiles fill
# the chip (5120 - 7168 columns: 17 - 19) and late where they do not (the k/v launches, 2 x 17408 columns
# and lm_head: 58 to the GEMV's 64-row limit).
PREFILL_CROSSOVER = {
    (5120, 1024): 64, (5120, 2048): 58, (5120, 5120): 17, (5120, 6144): 17, (5120, 7168): 19,
    (5120, 10240): 31, (5120, 12288): 33, (5120, 14336): 25, (5120, 16384): 33, (5120, 17408): 46,
    (5120, 34816): 64, (5120, 248320): 64, (6144, 5120): 30, (17408, 5120): 39,
}


@functools.lru_cache(maxsize=4096)
def _rd_serves(k: int, widths: tuple, K: int, ldy: int) -> bool:
    """Whether the library's register-decode GEMM serves such a launch at every row count of the GEMV."""
    return bool(_lib.lib().exl3_gemm_rd_serves(_lib.GEMV_MAX_ROWS, k, (C_int * len(widths))(*widths), len(widths), K, ldy))


def gemv_max_rows(k: int, width: int, K: int = 4, widths: Optional[tuple] = None, ldy: Optional[int] = None,
                  hold: bool = False) -> int:
    """Most rows a launch of k inputs and `width` output columns (groups of `widths`, output rows ldy
    apart) takes on the fused GEMV.  Where the register-decode GEMM is not what the other route runs
    (EXL3_PREFILL=recon, EXL3_GEMM_KERNEL, shapes beyond its limits) the boundary is the prefill
    GEMM's: the register-decode GEMM's own is up to 56 rows lower.  hold: that boundary (_hold)."""
    if MR_MAX is not None:
        return MR_MAX
    if hold or PREFILL_ROUTE == "recon" or GEMM_KERNEL or not _rd_serves(k, widths or (width,), K, ldy or width):
        b = PREFILL_CROSSOVER.get((k, width), DEFAULT_MR)
    else:
        b = _crossover(k, width, K)
    return min(b, _lib.GEMV_MAX_ROWS)


def gemv_rows(m: int, k: int, width: int, K: int = 4, widths: Optional[tuple] = None, ldy: Optional[int] = None,
              hold: bool = False) -> bool:
    """Route of an m-row launch: the fused GEMV (True; every row bitwise equal to its m = 1 call)
    or a GEMM."""
    return m <= gemv_max_rows(k, width, K, widths, ldy, hold)


def fused_rows(m: int, k: int, width: int, K: int = 4, widths: Optional[tuple] = None, ldy: Optional[int] = None,
               hold: bool = False) -> bool:
    """The GEMV route for the fused-epilogue forms (SiLU input, gated, approximate): <= 32 rows."""
    return m <= _lib.GEMV_FUSED_MAX_ROWS and gemv_rows(m, k, width, K, widths, ldy, hold)


# widest non-lm_head layer (17408): the shared reconstruction buffer of the `recon` prefill route
RECON_SLICE_N = int(os.environ.get("EXL3_RECON_SLICE_N", "17408"))
PREFILL_ROUTE = os.environ.get("EXL3_PREFILL", "fused")
# linear_silu_mul on the GEMV route: "unfused" (grouped GEMV + elementwise kernel) or "fused" (one
# gated GEMV launch)
GATED_ROUTE = os.environ.get("EXL3_GATED", "unfused")
def approx_mode(value: Optional[str]) -> str:
    """EXL3_GEMV_APPROX -> the GEMV's approximate mul1 route: "" (faithful, the default; also for
    "0", "off", "none", "faithful"), "affine" (unrounded weights) or "int8" (int8 activations, the
    reference's EXL3_ROCM_GFX1201_INT8 path).  Any other value raises: a misspelt opt-in must not
    silently run (or silently skip) a route with a different numerical budget."""
    v = (value or "").strip().lower()
    if v in ("", "0", "off", "none", "faithful"):
        return ""
    if v not in E.APPROX_MODES:
        raise ValueError(f"exl3rocm: EXL3_GEMV_APPROX={value!r}: expected one of "
                         f"{sorted(E.APPROX_MODES)} or off")
    return v


# opt-in approximate mul1 GEMV, up to 32 rows of the boundary against the prefill GEMM (fused_rows, hold)
GEMV_APPROX = approx_mode(os.environ.get("EXL3_GEMV_APPROX"))


def _approx(m: int, mul1: bool) -> bool:
    return bool(GEMV_APPROX) and mul1 and m <= _lib.GEMV_FUSED_MAX_ROWS


def _hold(x2: torch.Tensor, mul1: bool) -> bool:
    """Whether a launch keeps the GEMV up to the boundary against the prefill GEMM: the approximate form
    that the user asked for, or a stream that captures a graph without the workspace that the
    register-decode GEMM needs (it would record the unsplit prefill GEMM: gate at 16 rows 64 us, on the
    GEMV 28)."""
    return (GEMV_APPROX != "" and _approx(x2.shape[0], mul1)) or (x2.is_cuda and E.captures_without_prefill_workspace(x2))


def _gemv(m: int, x2: torch.Tensor, mul1: bool, k: int, width: int, K: int, widths: Optional[tuple] = None,
          ldy: Optional[int] = None, held: bool = False) -> bool:
    """gemv_rows(..., held or _hold) of a launch over the m rows x2, for the ops: no boundary lies below MID_MR or
    above the GEMV's rows, and _hold only raises one, so it asks for no more than decides the call (an eager
    call's host time: every question at every call took an MLP of 20 rows from 71.3 to 74.7 us, these 72.0)."""
    if MR_MAX is not None:
        return m <= MR_MAX
    if m <= MID_MR:
        return True
    if m > _lib.GEMV_MAX_ROWS:
        return False
    if held or PREFILL_ROUTE == "recon" or GEMM_KERNEL or not _rd_serves(k, widths or (width,), K, ldy or width):
        return m <= PREFILL_CROSSOVER.get((k, width), DEFAULT_MR)
    if m <= _crossover(k, width, K):
        return True
    return m <= PREFILL_CROSSOVER.get((k, width), DEFAULT_MR) and _hold(x2, mul1)


_wbuf: dict = {}


def ext():
    """The loaded HIP library (raises if it is not built)."""
    return _lib.lib()


def reserve_weight_buffer(device, numel):
    """Grow the shared reconstruction buffer (used by the `recon` prefill route) at load time,
    so graph capture never allocates it (reference ops.py:52-57)."""
    device = torch.device(device)
    buf = _wbuf.get(device)
    if buf is None or buf.numel() < numel:
        _wbuf[device] = torch.empty(numel, dtype=torch.float16, device=device)


def _weight_buffer(device, numel):
    reserve_weight_buffer(device, numel)
    return _wbuf[torch.device(device)][:numel]


def reserve_workspace(device, k: int, n: int, K: int, groups: int = 1, m: Optional[int] = None):
    """Reserve the GEMV workspace for up to m rows (load time; default: the most rows that any route
    sends to the GEMV for a module of groups x n columns): the current stream gets it now, and
    every other stream gets at least this much on its first eager call (so a later graph capture on
    that stream never allocates)."""
    if m is None:
        m = MR_MAX if MR_MAX is not None else max(PREFILL_CROSSOVER.get((k, n * groups), DEFAULT_MR),
                                                  gemv_max_rows(k, n * groups, K))
    if m < 1:
        return
    E.workspace(torch.device(device), E.gemv_workspace_bytes(min(m, _lib.GEMV_MAX_ROWS), k, n, K, groups),
                reserve=True)


def _prep(x: torch.Tensor):
    k = x.shape[-1]
    x2 = x if x.dim() == 2 and k else x.reshape(-1, k)
    if x2.dtype != torch.float16:
        x2 = x2.to(torch.float16)
    if not x2.is_contiguous():
        x2 = x2.contiguous()
    return x2, k


def _linear_into(x2, trellis, suh, svh, K, mcg, mul1, y, gemv: bool):
    """One group into y ([M, n] view, unit column stride, any row stride); gemv: the route chosen
    by the caller for the launch this group belongs to."""
    M, k = x2.shape
    n = svh.shape[0]
    if gemv and _approx(M, mul1):
        rc = E.exl3_gemv_mr_approx(x2, trellis, y, suh, None, svh, K, GEMV_APPROX)
        if rc != 0:
            raise RuntimeError(f"exl3rocm: approximate GEMV declined shape m={M} k={k} n={n} K={K}")
    elif gemv:
        rc = E.exl3_gemv_mr(x2, trellis, y, suh, None, svh, K, mcg, mul1)
        if rc != 0:
            raise RuntimeError(f"exl3rocm: GEMV declined shape m={M} k={k} n={n} K={K}")
    elif PREFILL_ROUTE == "recon":
        # the prefill GEMM's float32 transforms (exact=False): this route is bitwise equal to its whole tiles
        xh = torch.empty_like(x2)
        E.had_r_128(x2, xh, suh, None, 1.0, exact=False)
        for n0 in range(0, n, RECON_SLICE_N):
            n1 = min(n0 + RECON_SLICE_N, n)
            w = _weight_buffer(x2.device, k * (n1 - n0)).view(k, n1 - n0)
            if n0 == 0 and n1 == n:
                E.reconstruct(w, trellis, K, mcg, mul1)
            else:
                E.reconstruct_slice(w, trellis, K, mcg, mul1, n0)
            E.hgemm_recon(xh, w, y[:, n0:n1])
        E.had_r_128(y, y, None, svh, 1.0, exact=False)
    else:
        # the grouped entry point with one group: its launch balances the last wave of tiles
        xh = torch.empty_like(x2)
        E.exl3_gemm_trellis_grouped(x2, [trellis], y, [suh], xh, [svh], K, mcg, mul1)


def _shaped(y: torch.Tensor, x: torch.Tensor) -> torch.Tensor:
    """The [M, n] result y in the batch shape of x."""
    return y if x.dim() == 2 else y.view(*x.shape[:-1], y.shape[-1])


# The ops' bodies are plain functions: an op whose body needs another's calls that body, not the op
# (a custom op's way through the dispatcher takes ~7 us of host time, and the outer op has been through it).
def _linear(x: torch.Tensor, trellis: torch.Tensor, suh: torch.Tensor, svh: torch.Tensor,
            K: int, mcg: bool, mul1: bool) -> torch.Tensor:
    x2, k = _prep(x)
    n = svh.shape[0]
    M = x2.shape[0]
    y = torch.empty((M, n), dtype=torch.float16, device=x.device)
    if M:
        _linear_into(x2, trellis, suh, svh, K, mcg, mul1, y, _gemv(M, x2, mul1, k, n, K))
    return _shaped(y, x)


exl3_linear = torch.library.custom_op("exl3rocm::linear", mutates_args=())(_linear)


@exl3_linear.register_fake
def _(x, trellis, suh, svh, K, mcg, mul1):
    return x.new_empty((*x.shape[:-1], svh.shape[0]), dtype=torch.float16)


def _linear_groups(x: torch.Tensor, trellis: list[torch.Tensor], suh: list[torch.Tensor],
                   svh: list[torch.Tensor], K: list[int], mcg: bool, mul1: bool,
                   ptrs_trellis: Optional[torch.Tensor] = None, ptrs_suh: Optional[torch.Tensor] = None,
                   ptrs_svh: Optional[torch.Tensor] = None) -> torch.Tensor:
    """A fused module made of several checkpoint tensors (e.g. gate_proj + up_proj), each with its
    own K / suh / svh; the concatenation happens inside this opaque op (reference ops.py:106-175).

    ptrs_* = int64 device tensors of per-group data pointers, given when all groups share K and
    width (the reference's M == 1 exl3_mgemm route).  They are accepted and not read: the grouped
    launch takes the same pointers as kernel arguments instead (exl3_gemv_mr_grouped, the same
    kernel, split and output bitwise as exl3_mgemm over the tables), which saves every workgroup a
    dependent load of its table entries before its first trellis request (~1.3 us of a 5120 ->
    2 x 17408 launch)."""
    if len(trellis) == 1:
        return _linear(x, trellis[0], suh[0], svh[0], K[0], mcg, mul1)
    widths = [s.shape[0] for s in svh]
    x2, k = _prep(x)
    M = x2.shape[0]
    ng = len(trellis)
    if M == 0:                                        # every route: an empty batch launches nothing
        return x2.new_empty((*x.shape[:-1], sum(widths)), dtype=torch.float16)
    n_all = sum(widths)
    y = torch.empty((M, n_all), dtype=torch.float16, device=x.device)
    # runs of consecutive groups with equal K share one launch, each group written straight into
    # its row-strided column slice; each run takes the route of its own shape (EXL3_GATED=fused: gate and
    # up that of their one-launch form, so that both stay bitwise the same)
    held = GATED_ROUTE == "fused" and ng == 2 and K[0] == K[1] and widths[0] == widths[1] and M <= _lib.GEMV_FUSED_MAX_ROWS
    i, n0 = 0, 0
    while i < ng:
        j = i + 1
        while j < ng and j - i < _lib.MAX_GROUPS and K[j] == K[i]:
            j += 1
        w = sum(widths[i:j])
        gemv = _gemv(M, x2, mul1, k, w, K[i], tuple(widths[i:j]), n_all, held)
        if j == i + 1 or (gemv and _approx(M, mul1)) or \
                (not gemv and PREFILL_ROUTE == "recon"):
            # one group, the approximate GEMV or the recon prefill: each group its own launch
            c = n0
            for g in range(i, j):
                _linear_into(x2, trellis[g], suh[g], svh[g], K[g], mcg, mul1, y[:, c:c + widths[g]], gemv)
                c += widths[g]
        elif gemv and all(wd == widths[i] for wd in widths[i:j]):
            # equal widths (gate/up, k/v): the reference's grouped entry point
            E.exl3_gemv_mr_grouped(x2, list(trellis[i:j]), y[:, n0:], list(suh[i:j]), None, list(svh[i:j]),
                                   K[i], mcg, mul1, j - i)
        elif gemv:
            # mixed widths (q/k/v)
            E.exl3_gemv_mr_grouped_widths(x2, list(trellis[i:j]), y[:, n0:], list(suh[i:j]), list(svh[i:j]),
                                          K[i], mcg, mul1)
        else:
            # one grouped prefill GEMM launch, each group its own rotated input
            xh = torch.empty((j - i, M, k), dtype=torch.float16, device=x.device)
            E.exl3_gemm_trellis_grouped(x2, list(trellis[i:j]), y[:, n0:], list(suh[i:j]), xh, list(svh[i:j]),
                                        K[i], mcg, mul1)
        n0 += w
        i = j
    return _shaped(y, x)


exl3_linear_groups = torch.library.custom_op("exl3rocm::linear_groups", mutates_args=())(_linear_groups)


@exl3_linear_groups.register_fake
def _(x, trellis, suh, svh, K, mcg, mul1, ptrs_trellis=None, ptrs_suh=None, ptrs_svh=None):
    return x.new_empty((*x.shape[:-1], sum(s.shape[0] for s in svh)), dtype=torch.float16)


@torch.library.custom_op("exl3rocm::linear_silu_mul", mutates_args=())
def exl3_linear_silu_mul(x: torch.Tensor, trellis: list[torch.Tensor], suh: list[torch.Tensor],
                         svh: list[torch.Tensor], K: list[int], mcg: bool, mul1: bool) -> torch.Tensor:
    """A gated MLP's input: the gate (group 0) and up (group 1) linears of one module followed by
    SiLU-and-mul, act = fp16(fp16(silu(gate)) * up) with gate / up exactly as linear_groups
    computes them.  No counterpart in the reference plugin, whose MLP runs linear_groups and then
    a separate SiluAndMul (the fusion is proposed in reference docs/EFFICIENCY_INVESTIGATION.md:36-66).

    Routes: linear_groups, then an elementwise SiLU-and-mul kernel (the default: measured faster
    on MI355X); or, with EXL3_GATED=fused up to 32 rows (and the boundary against the prefill GEMM), equal K
    and width, one GEMV launch whose workgroup completing a 128-column block of both groups applies the
    activation: bitwise what linear_groups, on the GEMV at those rows under the knob, and SiLU-and-mul give."""
    if not (len(trellis) == 2 and len(suh) == 2 and len(svh) == 2 and len(K) == 2):
        raise RuntimeError("exl3rocm: linear_silu_mul takes exactly two groups (gate, up)")
    n = svh[0].shape[0]
    if svh[1].shape[0] != n:
        raise RuntimeError("exl3rocm: linear_silu_mul needs gate and up of equal width")
    x2, k = _prep(x)
    M = x2.shape[0]
    act = torch.empty((M, n), dtype=torch.float16, device=x.device)
    if M == 0:
        return act.view(*x.shape[:-1], n)
    if GATED_ROUTE == "fused" and K[0] == K[1] and fused_rows(M, k, 2 * n, K[0], (n, n), hold=True):
        E.exl3_gemv_silu_mul(x2, list(trellis), act, list(suh), list(svh), K[0], mcg, mul1)
    else:
        gu = _linear_groups(x2, trellis, suh, svh, K, mcg, mul1)
        E.silu_mul(gu[:, :n], gu[:, n:], act)
    return act.view(*x.shape[:-1], n)


@exl3_linear_silu_mul.register_fake
def _(x, trellis, suh, svh, K, mcg, mul1):
    return x.new_empty((*x.shape[:-1], svh[0].shape[0]), dtype=torch.float16)


@torch.library.custom_op("exl3rocm::silu_mul_linear", mutates_args=())
def exl3_silu_mul_linear(gu: torch.Tensor, trellis: torch.Tensor, suh: torch.Tensor, svh: torch.Tensor,
                         K: int, mcg: bool, mul1: bool) -> torch.Tensor:
    """A gated MLP's output: SiLU-and-mul of gu = [gate | up] (the [.., 2k] output of the gate/up
    linear_groups), act = fp16(fp16(silu(gate)) * up), then the down linear of act.  No
    counterpart in the reference plugin, whose MLP runs a separate SiluAndMul before the down
    linear (the fusion is proposed in reference docs/EFFICIENCY_INVESTIGATION.md:36-66).

    On the GEMV route one GEMV launch forms act from gate and up as its input rows
    load; on the GEMM routes the input transform forms act as it loads the rows (one transform launch and one
    GEMM launch, no act in memory); on the approximate GEMV routes and the recon prefill route the
    elementwise kernel writes act and linear runs on it.  Every route equals silu_mul followed by
    linear, bitwise."""
    k2 = gu.shape[-1]
    k = suh.shape[0]
    if k2 != 2 * k:
        raise RuntimeError(f"exl3rocm: silu_mul_linear takes [gate | up] of 2 * {k} columns, got {k2}")
    g2, _ = _prep(gu)
    M = g2.shape[0]
    n = svh.shape[0]
    y = torch.empty((M, n), dtype=torch.float16, device=gu.device)
    if M == 0:
        return y.view(*gu.shape[:-1], n)
    approx = _approx(M, mul1)
    gemv = _gemv(M, g2, mul1, k, n, K)
    if gemv and M <= _lib.GEMV_FUSED_MAX_ROWS and not approx:
        rc = E.exl3_gemv_silu_in(g2[:, :k], g2[:, k:], trellis, y, suh, None, svh, K, mcg, mul1)
        if rc != 0:
            raise RuntimeError(f"exl3rocm: GEMV declined shape m={M} k={k} n={n} K={K}")
    elif not gemv and PREFILL_ROUTE != "recon":
        xh = torch.empty((M, k), dtype=torch.float16, device=gu.device)
        E.exl3_gemm_trellis_silu_in(g2[:, :k], g2[:, k:], trellis, y, suh, xh, svh, K, mcg, mul1)
    else:
        act = torch.empty((M, k), dtype=torch.float16, device=gu.device)
        E.silu_mul(g2[:, :k], g2[:, k:], act)
        _linear_into(act, trellis, suh, svh, K, mcg, mul1, y, gemv)
    return y.view(*gu.shape[:-1], n)


@exl3_silu_mul_linear.register_fake
def _(gu, trellis, suh, svh, K, mcg, mul1):
    return gu.new_empty((*gu.shape[:-1], svh.shape[0]), dtype=torch.float16)
