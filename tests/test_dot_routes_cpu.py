"""Which products the planner leaves in place for the tiled kernels behind
mk_dot_general, and which it copies for the GEMM: in place only if those
kernels can read BOTH operands (one contiguous dimension each), else
mk_dot_general would run one thread per output."""

import pytest

from mi355x import programs as P
from mi355x import runtime as rt


def _plan(sa, sb, dt, lc, rc, lb=(), rb=()):
    text, _ = rt.compile_check(P.dot_general_dims(sa, sb, dt, lc, rc, lb, rb))
    return text


# One operand readable in place, the other with its batch dimension innermost.
@pytest.mark.parametrize("dt", ["bfloat16", "float32"])
@pytest.mark.parametrize("sa,sb,lc,rc,lb,rb", [
    ((8, 1024, 512), (1024, 512, 8), (1,), (0,), (0,), (2,)),   # lhs [K, M]
    ((8, 512, 1024), (1024, 512, 8), (2,), (0,), (0,), (2,)),
    ((512, 1024, 8), (8, 504, 1024), (1,), (2,), (2,), (0,)),   # rhs [N, K]
    ((512, 1024, 8), (8, 512, 1024), (1,), (2,), (2,), (0,)),
    ((512, 1024, 8), (8, 1024, 512), (1,), (1,), (2,), (0,)),
    ((1024, 512, 8), (1024, 512, 8), (0,), (0,), (2,), (2,)),   # neither
])
def test_one_unreadable_operand_means_copies_and_the_gemm(sa, sb, dt, lc, rc, lb, rb):
    plan = _plan(sa, sb, dt, lc, rc, lb, rb)
    assert "dot_general" not in plan and ("gemm_bf16" in plan or "gemm_f32" in plan), plan


@pytest.mark.parametrize("dt", ["bfloat16", "float32"])
@pytest.mark.parametrize("sa,sb,lc,rc,lb,rb", [
    ((1024, 512), (1024, 504), (0,), (0,), (), ()),                 # x^T dy
    ((8, 1024, 512), (8, 1024, 512), (1,), (1,), (0,), (0,)),
    ((8, 1024, 512), (8, 504, 1024), (1,), (2,), (0,), (0,)),       # both transposed
    ((1000, 1024), (504, 1024), (1,), (1,), (), ()),                # dy W^T, ragged
])
def test_readable_operands_stay_in_place(sa, sb, dt, lc, rc, lb, rb):
    plan = _plan(sa, sb, dt, lc, rc, lb, rb)
    assert "dot_general" in plan and "copy" not in plan and "operand" not in plan, plan
