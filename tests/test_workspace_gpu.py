"""The quantized wrappers' cached workspace (mi355x/ops.py)."""

import numpy as np
import pytest

from _gpu import dev, dev_bf16, host_bf16_bits, need_gpu, torch
from oracle import quant

pytestmark = pytest.mark.gpu


def test_workspace_is_made_and_grown_on_demand():
    """A stream's first call finds no workspace and makes one, a later call
    that needs more replaces it; the bits are those of the default stream."""
    need_gpu()
    from mi355x import _lib, ops
    rng = np.random.default_rng(77)
    stream = torch.cuda.Stream()
    sizes = []
    for M, K, N in [(16, 4096, 1792), (16, 4096, 14336), (16, 4096, 1792)]:
        x, p, s, z = quant.make_int4_case(rng, M, K, N)
        args = (dev_bf16(x), dev(p), dev_bf16(s), dev(z))
        expect = host_bf16_bits(ops.int4_g64_matmul(*args))
        torch.cuda.synchronize()
        with torch.cuda.stream(stream):
            y = ops.int4_g64_matmul(*args)
            sizes.append(ops.workspace(1, "cuda:0").numel())
        torch.cuda.synchronize()
        assert np.array_equal(host_bf16_bits(y), expect)
        assert sizes[-1] >= _lib.lib().mk_qmatmul_workspace_bytes(_lib.MK_QFMT_INT4_G64, M, K, N)
    assert sizes[0] < sizes[1] == sizes[2]
