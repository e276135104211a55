"""The GEMM's routes, as the host alone decides them: which of them are worth
timing when a plan is built, and which products fit a launch."""

import ctypes

import pytest

from mi355x import _lib

R = _lib.GEMM_ROUTES


def _timed(batch, M, N, K, out_f32=0):
    routes = (ctypes.c_int32 * 22)()
    n = _lib.lib().mk_gemm_bf16_autotune_routes(batch, M, N, K, _lib.MK_EPI_NONE, out_f32, routes)
    names = {v: k for k, v in R.items()}
    return {names[r] for r in routes[:n]}


@pytest.mark.parametrize("batch,M,N,K,there,absent", [
    (1, 4096, 4096, 4096, {"pipe", "ring", "t256x256", "t128x128"}, {"t16x64", "t32x64", "t64x64"}),
    (1, 16, 14336, 4096, {"t16x64"}, {"t256x256", "t128x128"}),
    (1, 256, 4096, 4096, {"t64x64"}, {"t256x256"}),
    (16, 2048, 2048, 128, {"persist"}, {"t16x64", "t32x64"}),
    (1, 1000, 14336, 4096, {"t256x256", "t128x128"}, {"t16x64", "t32x64", "t64x64"}),
])
def test_only_promising_routes_are_timed(batch, M, N, K, there, absent):
    got = _timed(batch, M, N, K)
    assert there <= got and not absent & got, got
    assert len(got) <= 7
    assert not {"reg256", "generic256", "generic128"} & got  # other names of a tile shape
