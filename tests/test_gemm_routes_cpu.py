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


@pytest.mark.parametrize("M,N,fits,refused", [
    (1 << 24, 8, {"t16x64", "t32x64", "t64x64", "t128x64", "t128x128", "t256x256"}, set()),
    (1 << 24, 4096, {"t128x128", "t256x256"}, {"t16x64", "t32x64", "t64x64"}),
    (16, 1 << 24, {"t16x64", "t256x256"}, set()),
])
def test_a_route_whose_grid_passes_a_launch_is_refused(M, N, fits, refused):
    """A launch has at most 2^32 threads in a grid dimension; 16-row tiles have
    a workgroup of 256 for every 16 x 64 results."""
    def ok(r):
        return _lib.lib().mk_gemm_bf16_route_fits(R[r], M, N, 64, _lib.MK_EPI_NONE, 0)
    assert all(ok(r) for r in fits) and not any(ok(r) for r in refused)
