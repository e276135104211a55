"""The tiled GEMM families (gemm_tile.hip, 16-bit; gemm_split.hip, f32) through
mk_dot_general: every storage order of the operands, padded rows, misaligned
bases, and sizes at the edges of their tiles and k steps, against float64; and
what the f32 kernel's split cannot represent, against the plain definition.

Tolerances: an f32 result within gamma_{K-1} * (|A| |B|)_ij of the float64
product (16-bit operands' products are exact in f32; f32 products are rounded
or cut at 2^-24, one operation more: gamma_K); a bf16 / f16 result within that
plus one rounding of the value."""

import ctypes

import numpy as np
import pytest

from _gpu import f32_sum_bound, need_gpu, torch

pytestmark = pytest.mark.gpu

# Type code and unit roundoff: round to nearest in a p-bit significand is off by
# at most 2^-p of the value (bf16: p = 8, f16: p = 11).
TYPES = {"bf16": (13, 2.0 ** -8), "f16": (10, 2.0 ** -11), "f32": (11, 0.0)}
TORCH = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}


def _operand(g, batch, rows, cols, dt, pad, offset):
    """A [batch, rows, cols] view whose rows are cols + pad apart, `offset`
    elements into its memory: (view, row stride, batch stride)."""
    ld = cols + pad
    buf = torch.randn(offset + batch * rows * ld, generator=g, device="cuda:0").to(dt)
    return buf[offset:].view(batch, rows, ld)[:, :, :cols], ld, rows * ld


# (batch, M, N, K): one tile and one past its edge for every tile size, K at
# and around the 32-, 64- and 128-k steps, short and odd sums.
SIZES = [(1, 1, 1, 16), (1, 16, 64, 32), (3, 17, 65, 33), (1, 33, 63, 127), (1, 64, 128, 128), (2, 65, 129, 129),
         (1, 128, 72, 1000), (1, 129, 257, 64), (1, 257, 5, 257), (1, 300, 264, 4104), (1, 256, 1001, 96),
         (1, 1024, 2056, 40), (1, 2000, 3001, 31), (5, 8, 8, 4096)]


@pytest.mark.parametrize("batch,M,N,K", SIZES)
@pytest.mark.parametrize("a_t,b_t", [(0, 0), (0, 1), (1, 0), (1, 1)])
@pytest.mark.parametrize("dt,pad,offset", [("bf16", 0, 0), ("bf16", 8, 8), ("bf16", 1, 3), ("f16", 0, 0),
                                           ("f32", 0, 0), ("f32", 3, 1)])
def test_tile_gemm_matches_float64(batch, M, N, K, a_t, b_t, dt, pad, offset):
    need_gpu()
    from mi355x import _lib
    code, unit = TYPES[dt]
    tdt = TORCH[dt]
    g = torch.Generator(device="cuda:0").manual_seed(batch + 3 * M + 5 * N + 7 * K + 2 * a_t + b_t)
    a, lda, ba = _operand(g, batch, K if a_t else M, M if a_t else K, tdt, pad, offset)
    b, ldb, bb = _operand(g, batch, N if b_t else K, K if b_t else N, tdt, pad, offset)
    sa = (ctypes.c_int64 * 3)(ba, *((1, lda) if a_t else (lda, 1)))
    sb = (ctypes.c_int64 * 3)(bb, *((1, ldb) if b_t else (ldb, 1)))
    am = (a.transpose(1, 2) if a_t else a).double().contiguous()
    bm = (b.transpose(1, 2) if b_t else b).double().contiguous()
    ref, mag = am @ bm, (am.abs() @ bm.abs()).cpu().numpy()
    print(f"[tile] {dt} b={batch} M={M} N={N} K={K} order {a_t}{b_t} pad {pad} offset {offset}", flush=True)
    for out_code, out_dt, u in ((11, torch.float32, 0.0), (code, tdt, unit))[:1 if dt == "f32" else 2]:
        c = torch.full((batch, M, N), float("nan"), device="cuda:0", dtype=out_dt)
        _lib.check(_lib.lib().mk_dot_general(code, code, out_code, a.data_ptr(), b.data_ptr(), c.data_ptr(), batch, M,
                                             N, K, sa, sb, torch.cuda.current_stream().cuda_stream))
        torch.cuda.synchronize()
        err = (c.double() - ref).abs().cpu().numpy()
        bound = f32_sum_bound(mag, K + (dt == "f32")) * (1 + u) + u * ref.abs().cpu().numpy()
        if dt == "f16" and u:
            bound = bound + 2.0 ** -25  # half a subnormal step
        bad = ~(err <= bound)
        assert not bad.any(), f"{int(bad.sum())} of {bad.size} outside the bound, worst {np.nanmax(err - bound):.3e}"


def _f32_gemm(a, b):
    from mi355x import ops
    c = ops.gemm_f32(a, b)
    torch.cuda.synchronize()
    return c


@pytest.mark.parametrize("M,N,K", [(16, 64, 64), (200, 136, 128), (300, 520, 264)])
@pytest.mark.parametrize("scale_a,scale_b", [(1.0, 1.0), (1e-15, 1.0), (1e-17, 1e-12), (1e-30, 1e15), (1e-38, 1e20),
                                             (1e18, 1e15), (2e30, 1e-20)])
def test_f32_gemm_keeps_f32_range(M, N, K, scale_a, scale_b):
    """Operands whose bf16 parts would underflow (or whose magnitudes are far
    apart) keep f32 accuracy; a few zero rows and columns among them."""
    need_gpu()
    g = torch.Generator(device="cuda:0").manual_seed(M + N + K)
    a = torch.randn(M, K, generator=g, device="cuda:0") * scale_a
    b = torch.randn(K, N, generator=g, device="cuda:0") * scale_b
    a[::7] = 0
    b[:, 3::11] = 0
    print(f"[f32 range] {M}x{N}x{K} {scale_a} {scale_b}", flush=True)
    c = _f32_gemm(a, b).double()
    ref, mag = a.double() @ b.double(), a.double().abs() @ b.double().abs()
    # A subnormal operand or result is off by up to 2^-150 of its own.
    bound = f32_sum_bound(mag.cpu().numpy(), K + 1) + K * 2.0 ** -149
    assert ((c - ref).abs().cpu().numpy() <= bound).all()
    assert (c[::7] == 0).all() and (c[:, 3::11] == 0).all()


@pytest.mark.parametrize("M,N,K", [(16, 64, 64), (200, 136, 128), (300, 520, 264)])
def test_f32_gemm_infinities_and_nans(M, N, K):
    """An infinity, a NaN and values next to the largest float go through the
    products that they are in and no others, as the definition has it."""
    need_gpu()
    g = torch.Generator(device="cuda:0").manual_seed(K)
    a = torch.randn(M, K, generator=g, device="cuda:0")
    b = torch.randn(K, N, generator=g, device="cuda:0")
    b[5] = b[5].abs() + 0.5  # what the infinity meets: one zero, one negative
    b[5, 2], b[5, 3] = 0.0, -1.0
    a[1, 5], a[9, 7], a[11, 0] = float("inf"), float("nan"), 3.4e38
    b[0] = 0.0
    b[0, 6] = 1.0
    print(f"[f32 special] {M}x{N}x{K}", flush=True)
    c = _f32_gemm(a, b).cpu()
    fin = torch.ones(M, dtype=torch.bool)
    fin[[1, 9, 11]] = False
    assert torch.isfinite(c[fin]).all() and torch.isnan(c[9]).all()
    assert torch.isnan(c[1, 2]) and c[1, 3] == float("-inf")
    assert (c[1, [0, 1] + list(range(4, N))] == float("inf")).all()
    assert c[11, 6] == torch.tensor(3.4e38) and (c[11, :6].abs() < 1e3).all()
    plain = a.double().cpu()[fin] @ b.double().cpu()
    mag = a.double().cpu().abs()[fin] @ b.double().cpu().abs()
    assert ((c[fin].double() - plain).abs().numpy() <= f32_sum_bound(mag.numpy(), K + 1)).all()
