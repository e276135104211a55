"""Which kernels a quantized product runs on, by shape alone (host-only)."""

import pytest

from mi355x import _lib

DECODE, MID, MANY, DEQUANT = range(4)


@pytest.mark.parametrize("fmt,M,K,N,route", [
    (0, 1, 4096, 1792, DECODE), (0, 16, 4096, 14336, DECODE), (1, 16, 4096, 14336, DECODE),
    (0, 100, 4096, 14336, MID), (1, 100, 4096, 14336, MID), (0, 128, 4096, 1792, MID),
    (1, 3, 1216, 2048, MID), (1, 1, 4032, 4096, MID),           # K that keeps the streaming kernels out
    (0, 256, 4096, 14336, MID), (1, 700, 4096, 14336, MID),
    (0, 1000, 4096, 14336, DEQUANT), (0, 4096, 4096, 14336, DEQUANT),
    (0, 1024, 2048, 8192, DEQUANT), (1, 768, 4096, 14336, DEQUANT),  # where the paired SwiGLU form is
    (0, 100, 100, 1024, -1), (2, 16, 4096, 4096, -1),
])
def test_route(fmt, M, K, N, route):
    assert _lib.lib().mk_qmatmul_route(fmt, M, K, N) == route


def test_the_mid_row_kernel_can_be_turned_off_or_forced(monkeypatch):
    r = _lib.lib().mk_qmatmul_route
    monkeypatch.setenv("MK_QMM_QT", "0")
    assert r(0, 100, 4096, 14336) != MID
    monkeypatch.setenv("MK_QMM_QT", "2")
    assert r(0, 1000, 4096, 14336) == MID
