"""The GEMM's launch choice as a caller sees it without a GPU: the workspace its k splits ask for,
and the launches it refuses."""
from __future__ import annotations

import ctypes as C

import pytest
import torch

from violetto import _lib as L

COUNTERS = 65536 * 4           # hand-off counters at the front of a workspace
WINDOW = 1 << 31               # bytes of partial sums the kernels can address


def partials_at_most(nbytes: int) -> int:
    """Bytes of partial sums in a workspace (the rest: the counters and a sum of squares per
    token and split, at most 1/64 of the partials)."""
    return max(0, nbytes - COUNTERS)


@pytest.mark.parametrize("m,k", [(28672, 8192), (28672, 4096), (151552, 4096), (27648, 5120), (16384, 8192),
                                 (2048, 8192), (16384, 2048), (32000, 2048), (1280, 3328), (6656, 1280),
                                 (8256, 8192), (40000, 8192)])
def test_split_partials_stay_addressable(m, k):
    """Partial sums are addressed by 32-bit offsets through a 2 GiB descriptor: no row count asks
    for more of them (past it stores were dropped and the sums read back as zeros)."""
    rows = sorted({int(17 * 1.07 ** i) for i in range(115)} | {513, 1025, 1682, 4609, 4770, 8200, 9345, 16385, 63361})
    for n in rows:
        if n * k * 4 >= WINDOW:
            continue
        got = L.lib().sv_matmul_workspace_bytes(n, m, k)
        assert partials_at_most(got) < WINDOW + WINDOW // 64, f"{n} rows: workspace of {got} bytes"


@pytest.mark.parametrize("m,k", [(3072, 2048), (2048, 2048), (16384, 2048), (2048, 8192), (32000, 2048), (1792, 1280),
                                 (1280, 1280), (6656, 1280), (1280, 3328)])
def test_splits_stay_within_one_round(m, k):
    """A split launch is at most one round of 256 workgroups of 512 x 128 sums (64 MiB) at any
    row count: in several rounds the partial sums cost more than the rounds they save."""
    for n in range(17, 2600):
        got = partials_at_most(L.lib().sv_matmul_workspace_bytes(n, m, k))
        assert got <= (64 << 20) * 65 // 64, f"{n} rows: workspace of {got} bytes"


@pytest.mark.skipif(torch.cuda.is_available(), reason="made-up pointers: the call must not reach a GPU")
def test_launch_past_the_window_is_refused():
    """A forced split (the tests' override) with 2 GiB of partial sums or more is refused before
    any launch; the same shape one step below is not (without a device it fails at the launch)."""
    tune = (C.c_int * 7).in_dll(L.lib(), "_ZN2sv11g_gemm_tuneE")
    m, k = 16384, 2048
    one = C.c_void_p(1 << 20)
    try:
        for i, v in enumerate((1, 1, 4, 4, 33, 8, 2)):
            tune[i] = v
        for n, ok in ((8192, False), (8192 - 32, True)):   # m x n x 4 splits x 4 bytes
            mat = L.Matrix(one, one, m, k, L.FMT_I8, 31)
            a = L.MatArgs(n, k, m, L.EPI_RAW, 0, m, 1.0, 0, 0, 1, k, 31)
            rc = L.lib().sv_matmul(None, C.byref(mat), one, None, one, None, None, C.byref(a), one, 1 << 40)
            assert (rc == 4) == (not ok), L.lib().sv_last_error()
    finally:
        for i in range(7):
            tune[i] = 0


# (format, m, k, rows) -> measured us of launches (row tiles per wave, token tiles, k splits, chunks in
# flight, tile: 16 mm_gemm, 32 mm_gemm32, 33 mm_pipe, waves, chunks per iteration), MI355X, weights cold:
# sizes at which a rule of this choice has taken a launch 5-40 % slower than another one.
MEASURED = [
    ("bf16", 32000, 2048, 161, {(1, 4, 1, 4, 33, 8, 1): 64.8, (4, 4, 1, 2, 16, 4, 1): 77.4, (2, 3, 1, 4, 16, 4, 1): 79.4}),
    ("bf16", 32000, 2048, 192, {(1, 4, 1, 4, 33, 8, 1): 67.6, (4, 4, 1, 2, 16, 4, 1): 79.4, (2, 3, 1, 4, 16, 4, 1): 81.6}),
    ("bf16", 32000, 2048, 448, {(1, 4, 1, 4, 33, 8, 1): 132.6, (4, 4, 1, 2, 16, 4, 1): 148.5}),
    ("bf16", 3072, 2048, 352, {(2, 2, 2, 2, 16, 4, 1): 22.3, (1, 1, 1, 4, 33, 8, 2): 25.5}),
    ("bf16", 3072, 2048, 384, {(2, 2, 2, 2, 16, 4, 1): 22.6, (1, 1, 1, 4, 33, 8, 2): 25.3}),
    ("bf16", 1280, 3328, 832, {(2, 2, 2, 2, 16, 4, 1): 28.7, (1, 2, 2, 4, 33, 8, 2): 32.2}),
    ("bf16", 16384, 2048, 1280, {(4, 4, 1, 2, 16, 4, 1): 173.5, (2, 2, 1, 4, 33, 8, 1): 176.3}),
    ("i8", 16384, 2048, 1152, {(2, 2, 1, 4, 33, 8, 1): 159.5, (2, 4, 4, 4, 33, 8, 1): 330.0}),
    ("i8", 2048, 8192, 896, {(1, 2, 2, 4, 33, 8, 2): 70.6, (2, 2, 4, 4, 33, 8, 1): 75.6, (1, 1, 1, 4, 32, 8, 1): 79.7}),
    ("i8", 2048, 8192, 1536, {(2, 2, 2, 4, 33, 8, 1): 106.5, (1, 1, 1, 4, 32, 8, 1): 143.4, (2, 2, 8, 4, 33, 8, 1): 190.5}),
    ("g64", 16384, 2048, 32, {(1, 2, 4, 2, 16, 4, 1): 20.3, (1, 1, 4, 4, 33, 8, 2): 20.6, (1, 1, 2, 4, 33, 8, 2): 23.6}),
    ("g64", 2048, 2048, 256, {(1, 2, 4, 2, 16, 4, 1): 18.4, (1, 2, 2, 2, 16, 4, 1): 19.3, (1, 1, 2, 4, 33, 8, 2): 21.2}),
    ("g64", 1280, 3328, 176, {(1, 2, 4, 2, 16, 4, 1): 19.0, (1, 1, 4, 4, 33, 8, 2): 20.6}),
]


@pytest.mark.parametrize("fmt,m,k,n,us", MEASURED)
def test_choice_takes_a_fast_launch(fmt, m, k, n, us):
    """Within 3 % (the spread of repeated measurements) of the fastest launch measured there."""
    out = (C.c_int * 7)()
    L.lib()._ZN2sv11gemm_choiceEjbjjjPi(L.FMT_BF16 if fmt == "bf16" else L.FMT_I8, C.c_bool(fmt == "g64"), n, m, k, out)
    assert us.get(tuple(out), 1e9) <= 1.03 * min(us.values()), f"{tuple(out)}: {us}"
