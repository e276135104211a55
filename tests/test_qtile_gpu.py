"""The mid-row quantized kernel (csrc/kernels/qtile.hip): every tile height
and K split at the edges of its tiles, against the oracle, and the routes that
stay on the older kernels.

Tolerance against the oracle: the kernel sums exact products (integer weights,
bf16 x) in f32 and rounds once to bf16, 2^-8 of the value, far under the
workload's rel 2e-2."""

import numpy as np
import pytest

from _gpu import (BF16_RTOL, assert_rel_close, dev, dev_bf16, f32_sum_bound, host_bf16, host_bf16_bits, need_gpu,
                  torch)
from oracle import cport, quant

pytestmark = pytest.mark.gpu


def _case(fmt, M, K, N):
    need_gpu()
    from mi355x import ops
    rng = np.random.default_rng(M * 5 + K + N)
    if fmt == "int4":
        x, p, s, z = quant.make_int4_case(rng, M, K, N)
        return (dev_bf16(x), dev(p), dev_bf16(s), dev(z)), ops.int4_g64_matmul, cport.int4_g64_matmul(x, p, s, z)
    x, w, s = quant.make_int8_case(rng, M, K, N)
    return (dev_bf16(x), dev(w), dev(s)), ops.int8_pc_matmul, cport.int8_pc_matmul(x, w, s)


# Rows around a tile's edge; one k group, fewer groups than wave groups, an
# odd count, uneven splits; columns in whole chunks, 8-byte rows, one tile
# less a chunk, less than a chunk.
SHAPES = [(1, 64, 8), (17, 64, 128), (32, 192, 136), (33, 1088, 120), (65, 704, 16), (97, 1600, 264),
          (129, 448, 3000), (256, 320, 144)]


@pytest.mark.parametrize("M,K,N,ks", [(*s, ks) for s in SHAPES for ks in (1, 2, 3, 8) if s[1] // 64 >= ks])
@pytest.mark.parametrize("bm", [32, 64, 96, 128])
@pytest.mark.parametrize("fmt", ["int4", "int8"])
def test_every_tile_and_split(monkeypatch, fmt, M, K, N, bm, ks):
    args, run, ref = _case(fmt, M, K, N)
    from mi355x import ops
    monkeypatch.setenv("MK_QMM_QT_BM", str(bm))
    monkeypatch.setenv("MK_QMM_QT_KS", str(ks))
    monkeypatch.setenv("MK_QMM_QT", "2")
    print(f"[qtile] {fmt} M={M} K={K} N={N} bm={bm} ks={ks}", flush=True)
    first = host_bf16_bits(run(*args))
    again = host_bf16_bits(run(*args))
    torch.cuda.synchronize()
    assert np.array_equal(first, again)
    if ks > 1:  # the arrival counters return to zero
        assert int(ops.workspace(1, "cuda:0")[: 64 * 1024].count_nonzero()) == 0
    assert_rel_close(host_bf16(run(*args)), ref, BF16_RTOL, f"{fmt} {M}x{K}x{N} tile {bm} split {ks}")


def _route(fmt, M, K, N):
    from mi355x import _lib
    return _lib.lib().mk_qmatmul_route(_lib.MK_QFMT_INT4_G64 if fmt == "int4" else _lib.MK_QFMT_INT8_PC, M, K, N)


# Shapes that the rule gives to this kernel, or leaves, against the kernels it
# stands in for (which MK_QMM_QT=0 leaves): streaming, 64-column, many-row, GEMM.
@pytest.mark.parametrize("fmt,M,K,N,mid", [(f, *s) for f in ("int4", "int8") for s in (
    (100, 4096, 2048, False), (100, 2112, 2048, True), (20, 1088, 1000, True), (3, 1216, 2048, True),
    (300, 1024, 1024, True), (1000, 1024, 520, f == "int8"))])
def test_agrees_with_the_older_kernels(monkeypatch, fmt, M, K, N, mid):
    """The shape's default route is what MK_QMM_QT=2 forces, bit for bit, if it
    is this kernel, and MK_QMM_QT=0's if it is not; and the two kernels agree.
    Each sums K products in f32 (f32_sum_bound of the terms' magnitudes, a
    scale or two more) and rounds to bf16 (2^-9 of the value, 2^-8 together);
    the older kernels may round each weight to bf16 before (2^-9 of its
    term)."""
    args, run, ref = _case(fmt, M, K, N)
    print(f"[qtile] routes {fmt} M={M} K={K} N={N}", flush=True)
    default = host_bf16_bits(run(*args))
    monkeypatch.setenv("MK_QMM_QT", "2")
    assert _route(fmt, M, K, N) == 1
    forced = run(*args)
    monkeypatch.setenv("MK_QMM_QT", "0")
    assert _route(fmt, M, K, N) != 1
    older = run(*args)
    monkeypatch.delenv("MK_QMM_QT")
    torch.cuda.synchronize()
    assert (_route(fmt, M, K, N) == 1) == mid
    assert np.array_equal(default, host_bf16_bits(forced if mid else older))
    new, old = host_bf16(forced).astype(np.float64), host_bf16(older).astype(np.float64)
    assert_rel_close(new, ref, BF16_RTOL, f"{fmt} {M}x{K}x{N}")
    assert_rel_close(old, ref, BF16_RTOL, f"{fmt} {M}x{K}x{N} older kernel")
    if fmt == "int4":
        x, p, s, z = (t.cpu() for t in args)
        q = torch.stack([p & 15, p >> 4], 1).reshape(K, N).double()
        w = (q - z.double().repeat_interleave(64, 0)) * s.double().repeat_interleave(64, 0)
    else:
        x, w, s = (t.cpu().double() for t in args)
        w = w * s
    terms = (x.double().abs() @ w.abs()).numpy()
    bound = 2.0 ** -8 * np.maximum(np.abs(new), np.abs(old)) + 2.0 ** -9 * terms + 2 * f32_sum_bound(terms, K + 2)
    assert (np.abs(new - old) <= 1.01 * bound).all()


@pytest.mark.parametrize("fmt", ["int4", "int8"])
def test_unaligned_pointer_and_replayed_graph(monkeypatch, fmt):
    """Weights 4 bytes off 16-byte alignment stay on the 64-column kernel,
    whose loads are dwords (its bits, which are not this kernel's); a captured
    call replays to the eager bits with work between the replays."""
    args, run, ref = _case(fmt, 50, 1088, 1008)
    assert _route(fmt, 50, 1088, 1008) == 1
    eager = host_bf16_bits(run(*args))
    flat = torch.empty(args[1].numel() + 16, dtype=args[1].dtype, device="cuda")
    w = flat[4:4 + args[1].numel()].view(args[1].shape)
    w.copy_(args[1])
    offset = run(args[0], w, *args[2:])
    assert_rel_close(host_bf16(offset), ref, BF16_RTOL, f"{fmt} offset weights")
    with monkeypatch.context() as m:
        m.setenv("MK_QMM_QT", "0")
        older = host_bf16_bits(run(*args))
    assert np.array_equal(host_bf16_bits(offset), older) and not np.array_equal(older, eager)
    y = torch.empty((50, 1008), dtype=torch.bfloat16, device="cuda")
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        run(*args, out=y)
    for _ in range(3):
        y.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert np.array_equal(host_bf16_bits(y), eager)
        assert np.array_equal(host_bf16_bits(run(*args)), eager)
