"""The f32 GEMM (gemm_split.hip): a result's bits depend on its row of A and
its column of B alone, whether it keeps the split's sum or is recomputed: not
on the tile, and not on the other rows and columns of the call."""

import pytest

from _gpu import need_gpu, torch

pytestmark = pytest.mark.gpu

SIZES = [(16, 64, 64), (200, 136, 128), (300, 520, 264)]


def _bits(t):
    return t.cpu().view(torch.int32)


def _operands(kind, M, N, K):
    need_gpu()
    g = torch.Generator(device="cuda:0").manual_seed(M + N + K)
    a = torch.randn(M, K, generator=g, device="cuda:0")
    b = torch.randn(K, N, generator=g, device="cuda:0")
    if kind == "zero rows":  # padding
        a[::5], b[:, 3::7] = 0, 0
    elif kind == "tails":  # a softmax's, with padding beside them
        a = torch.exp(-60 * a.abs())
        a[::5] = 0
    elif kind == "far apart":
        a[::3] *= 1e-30
        b[:, ::4] *= 1e25
        b[:, 1::4] *= 1e-25
    elif kind == "subnormal":
        a[::3] *= 1e-40
        b[:, ::2] *= 1e-5
    elif kind == "infinity":
        a[1, 5], a[M - 2, 7], b[3, N // 2] = float("inf"), float("nan"), float("-inf")
    elif kind == "largest":
        a[::4] *= 3e37
        b[:, 1::3] *= 1e-30
    return a, b


KINDS = ["normal", "zero rows", "tails", "far apart", "subnormal", "infinity", "largest"]


@pytest.mark.parametrize("M,N,K", SIZES)
@pytest.mark.parametrize("kind", KINDS)
def test_every_tile_gives_the_same_bits(monkeypatch, kind, M, N, K):
    from mi355x import ops
    a, b = _operands(kind, M, N, K)
    print(f"[f32 bits] {kind} {M}x{N}x{K}", flush=True)
    outs = []
    for tile in ("16", "64", "128"):
        monkeypatch.setenv("MK_GEMM_F32_TILE", tile)
        outs.append(_bits(ops.gemm_f32(a, b)))
    assert torch.equal(outs[0], outs[1]) and torch.equal(outs[0], outs[2])


@pytest.mark.parametrize("M,N,K", SIZES)
@pytest.mark.parametrize("kind", KINDS)
def test_bits_do_not_depend_on_other_rows_and_columns(kind, M, N, K):
    from mi355x import ops
    a, b = _operands(kind, M, N, K)
    print(f"[f32 bits] parts of {kind} {M}x{N}x{K}", flush=True)
    whole = _bits(ops.gemm_f32(a, b))
    for rows in (slice(0, M, 3), slice(1, M, 2), slice(M // 2, M)):
        assert torch.equal(_bits(ops.gemm_f32(a[rows].contiguous(), b)), whole[rows])
    cols = slice(8, N - N % 16, 2)
    part = b[:, cols].contiguous()
    part = part[:, :part.shape[1] // 8 * 8].contiguous()
    assert torch.equal(_bits(ops.gemm_f32(a, part)), whole[:, cols][:, :part.shape[1]])
