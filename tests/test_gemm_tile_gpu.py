"""The tiled 16-bit GEMM family (gemm_tile.hip) through mk_dot_general: every
storage order of the operands, padded rows, misaligned bases, f16, and sizes
at the edges of its tiles and k steps, against float64.

Tolerances: an f32 result within gamma_{K-1} * (|A| |B|)_ij of the float64
product (the operands' products are exact in f32); a bf16 / f16 result within
that plus one rounding of the value."""

import ctypes

import numpy as np
import pytest

from _gpu import f32_sum_bound, need_gpu, torch

pytestmark = pytest.mark.gpu

# Type code and unit roundoff: round to nearest in a p-bit significand is off by
# at most 2^-p of the value (bf16: p = 8, f16: p = 11).
TYPES = {"bf16": (13, 2.0 ** -8), "f16": (10, 2.0 ** -11)}


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
@pytest.mark.parametrize("dt,pad,offset", [("bf16", 0, 0), ("bf16", 8, 8), ("bf16", 1, 3), ("f16", 0, 0)])
def test_tile_gemm_matches_float64(batch, M, N, K, a_t, b_t, dt, pad, offset):
    need_gpu()
    from mi355x import _lib
    code, unit = TYPES[dt]
    tdt = torch.bfloat16 if dt == "bf16" else torch.float16
    g = torch.Generator(device="cuda:0").manual_seed(batch + 3 * M + 5 * N + 7 * K + 2 * a_t + b_t)
    a, lda, ba = _operand(g, batch, K if a_t else M, M if a_t else K, tdt, pad, offset)
    b, ldb, bb = _operand(g, batch, N if b_t else K, K if b_t else N, tdt, pad, offset)
    sa = (ctypes.c_int64 * 3)(ba, *((1, lda) if a_t else (lda, 1)))
    sb = (ctypes.c_int64 * 3)(bb, *((1, ldb) if b_t else (ldb, 1)))
    am = (a.transpose(1, 2) if a_t else a).double().contiguous()
    bm = (b.transpose(1, 2) if b_t else b).double().contiguous()
    ref, mag = am @ bm, (am.abs() @ bm.abs()).cpu().numpy()
    print(f"[tile] {dt} b={batch} M={M} N={N} K={K} order {a_t}{b_t} pad {pad} offset {offset}", flush=True)
    for out_code, out_dt, u in ((11, torch.float32, 0.0), (code, tdt, unit)):
        c = torch.full((batch, M, N), float("nan"), device="cuda:0", dtype=out_dt)
        _lib.check(_lib.lib().mk_dot_general(code, code, out_code, a.data_ptr(), b.data_ptr(), c.data_ptr(), batch, M,
                                             N, K, sa, sb, torch.cuda.current_stream().cuda_stream))
        torch.cuda.synchronize()
        err = (c.double() - ref).abs().cpu().numpy()
        bound = f32_sum_bound(mag, K) * (1 + u) + u * ref.abs().cpu().numpy()
        if dt == "f16" and u:
            bound = bound + 2.0 ** -25  # half a subnormal step
        bad = ~(err <= bound)
        assert not bad.any(), f"{int(bad.sum())} of {bad.size} outside the bound, worst {np.nanmax(err - bound):.3e}"
