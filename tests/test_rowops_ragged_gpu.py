"""Row kernels on rows that are not 16-byte aligned, on few long rows and on
many short ones: the edges of each kernel's range (one wave a row up to 256
vectors, 256 threads up to 16 vectors each, 1024 threads up to 65536 columns,
the streaming kernel beyond), against the oracle, with rows dense in NaN,
infinities and signed zeros for the exact ones."""

import numpy as np
import pytest

from _gpu import BF16_RTOL, F32_RTOL, assert_rel_close, dev, dev_bf16, f32_sum_bound, host_bf16, need_gpu, torch
from oracle import bf16 as obf
from oracle import rowops
from test_rowops_gpu import _edge

pytestmark = pytest.mark.gpu

SHAPES = [(513, 5), (512, 255), (513, 257), (600, 1023), (600, 1025), (520, 2047), (513, 2049), (511, 1001),
          (3, 8193), (5, 16385), (600, 16387), (2, 32001), (1, 50257), (2, 65536), (2, 65537), (1, 131073)]


def _ops():
    need_gpu()
    from mi355x import ops
    return ops


def _x(shape, seed):
    return (np.random.default_rng(seed).standard_normal(shape) * 2).astype(np.float32)


@pytest.mark.parametrize("shape", SHAPES)
def test_ragged_rows_match_oracle(shape):
    ops = _ops()
    x = _x(shape, shape[1])
    g = np.random.default_rng(4).uniform(0.5, 1.5, shape[-1]).astype(np.float32)
    print(f"[rows] {shape}", flush=True)
    assert_rel_close(ops.softmax(dev(x)).cpu().numpy(), rowops.softmax(x), F32_RTOL, f"softmax f32 {shape}")
    assert_rel_close(ops.rmsnorm(dev(x), dev(g)).cpu().numpy(), rowops.rmsnorm(x, g), F32_RTOL, f"rmsnorm f32 {shape}")
    got = ops.reduce_lastdim(dev(x), "sum").cpu().numpy()
    assert (np.abs(got - x.astype(np.float64).sum(-1)) <= f32_sum_bound(np.abs(x).astype(np.float64).sum(-1),
                                                                         shape[1])).all()
    xb, gb = obf.f32_to_bf16_bits(x), obf.f32_to_bf16_bits(g)
    assert_rel_close(host_bf16(ops.softmax(dev_bf16(xb))), obf.bf16_bits_to_f32(rowops.softmax_bf16(xb)), BF16_RTOL,
                     f"softmax bf16 {shape}")
    assert_rel_close(host_bf16(ops.rmsnorm(dev_bf16(xb), dev_bf16(gb))),
                     rowops.rmsnorm(obf.bf16_bits_to_f32(xb), obf.bf16_bits_to_f32(gb)), BF16_RTOL,
                     f"rmsnorm bf16 {shape}")


@pytest.mark.parametrize("shape", SHAPES)
def test_ragged_rows_special_values(shape):
    """argmax, max and min exactly, and softmax's NaN rows, on rows dense with
    special values, a row of -inf, one of +inf and one of NaN among them."""
    ops = _ops()
    x = _edge(shape, shape[1])
    for r, v in enumerate((-np.inf, np.inf, np.nan)):
        if r < shape[0] - 1:
            x[r] = v
    print(f"[rows special] {shape}", flush=True)
    for dt, d, h in (("f32", dev(x), x), ("bf16", dev_bf16(obf.f32_to_bf16_bits(x)),
                                          obf.bf16_bits_to_f32(obf.f32_to_bf16_bits(x)))):
        np.testing.assert_array_equal(ops.argmax(d).cpu().numpy(), rowops.argmax(h), err_msg=dt)
        for op, f in (("max", np.max), ("min", np.min)):
            got = ops.reduce_lastdim(d, op).float().cpu().numpy()
            np.testing.assert_array_equal(got, f(h, axis=-1), err_msg=f"{dt} {op}")
        y = ops.softmax(d).float().cpu().numpy()
        m = h.max(-1)
        np.testing.assert_array_equal(np.isnan(y).all(-1), ~np.isfinite(m), err_msg=dt)


# Row lengths of each kernel that the number of rows chooses between: a wave or
# 256 threads (up to 256 vectors), 256 or 1024 threads (above 8 vectors each).
@pytest.mark.parametrize("dt,cols", [(dt, c) for dt in ("f32", "bf16") for c in (
    100, 250, 256, 500, 512, 1000, 1024, 1025, 2048, 8200, 9001, 12000, 16384, 16400, 20001, 32000, 32768)])
def test_a_rows_bits_do_not_depend_on_the_number_of_rows(dt, cols):
    """Sums of a row are added in an order that its length alone decides."""
    ops = _ops()
    x, g = _x((600, cols), cols), _x((cols,), 1)
    if dt == "bf16":
        x, g = dev_bf16(obf.f32_to_bf16_bits(x)), dev_bf16(obf.f32_to_bf16_bits(g))
    else:
        x, g = dev(x), dev(g)
    print(f"[rows bits] {dt} {cols}", flush=True)
    for name, f in (("softmax", ops.softmax), ("rmsnorm", lambda v: ops.rmsnorm(v, g)),
                    ("sum", lambda v: ops.reduce_lastdim(v, "sum"))):
        many = f(x)
        for n in (1, 7, 511):
            assert torch.equal(f(x[:n].contiguous()), many[:n]), (name, n)
