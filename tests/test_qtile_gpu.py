"""The mid-row quantized kernel (csrc/kernels/qtile.hip): every tile height
and K split at the edges of its tiles, against the oracle, and the routes that
stay on the older kernels.

Tolerance: the kernel sums exact products (integer weights, bf16 x) in f32 and
rounds once to bf16, 2^-8 of the value, far under the workload's rel 2e-2; the
older kernels round the dequantised weights to bf16 too, so the two agree to
a few 2^-8."""

import numpy as np
import pytest

from _gpu import (BF16_RTOL, assert_rel_close, dev, dev_bf16, host_bf16, host_bf16_bits, need_gpu,
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


# Shapes the rule gives to this kernel, against the kernels it stands in for
# (which MK_QMM_QT=0 leaves): streaming, 64-column, many-row, GEMM.
@pytest.mark.parametrize("fmt", ["int4", "int8"])
@pytest.mark.parametrize("M,K,N", [(100, 4096, 2048), (20, 1088, 1000), (3, 1216, 2048), (300, 1024, 1024),
                                   (1000, 1024, 520)])
def test_agrees_with_the_older_kernels(monkeypatch, fmt, M, K, N):
    args, run, ref = _case(fmt, M, K, N)
    print(f"[qtile] routes {fmt} M={M} K={K} N={N}", flush=True)
    new = host_bf16(run(*args))
    monkeypatch.setenv("MK_QMM_QT", "0")
    old = host_bf16(run(*args))
    torch.cuda.synchronize()
    assert_rel_close(new, ref, BF16_RTOL, f"{fmt} {M}x{K}x{N}")
    assert_rel_close(old, ref, BF16_RTOL, f"{fmt} {M}x{K}x{N} older kernel")


@pytest.mark.parametrize("fmt", ["int4", "int8"])
def test_unaligned_pointer_and_replayed_graph(fmt):
    """Weights 4 bytes off 16-byte alignment stay on the 64-column kernel,
    whose loads are dwords; a captured call replays to the eager bits with
    work between the replays."""
    args, run, ref = _case(fmt, 50, 1088, 1008)
    eager = host_bf16_bits(run(*args))
    flat = torch.empty(args[1].numel() + 16, dtype=args[1].dtype, device="cuda")
    w = flat[4:4 + args[1].numel()].view(args[1].shape)
    w.copy_(args[1])
    assert_rel_close(host_bf16(run(args[0], w, *args[2:])), ref, BF16_RTOL, f"{fmt} offset weights")
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
