"""Which kernel and grid a product runs, by its sizes alone: the choices of ``kernels/ops.py``, played on the CPU with tensors
that have sizes and no memory.  The grids named were timed on a device of 256 compute units."""

from __future__ import annotations

import pytest
import torch

from turboserve_amd.kernels.ops import Ops


class Planner(Ops):
    """The library's choices without the library: the products note how they were called."""

    def __init__(self):
        self.compute_units = 256
        self._tiled_plans, self._wide_plans, self._stream_plans, self._block_plans = {}, {}, {}, {}
        self.wide_choices, self.wide_timings = {}, {}

    def gemm_block(self, x, weight, bias=None, *, plan, gated=False, sums=False, rule=None):
        return "block", plan, plan[1] > 1 or sums

    def gemm_wide(self, x, weight, bias=None, *, plan, gated=False, sums=False, rule=None):
        return "wide", plan, plan[1] > 1 or sums


def operands(m: int, n: int, k: int) -> tuple[torch.Tensor, torch.Tensor]:
    return (torch.empty(m, k, dtype=torch.bfloat16, device="meta"), torch.empty(n, k, dtype=torch.bfloat16, device="meta"))


@pytest.mark.parametrize("n,k", [(3584, 18944), (3584, 3584), (5120, 13824), (2048, 2048), (16384, 16384), (8192, 29568)])
def test_an_addend_of_the_residual_stream_keeps_its_32_bits(n, k):
    """Up to ``wide_default_rows`` rows what goes into the residual stream is 32-bit sums, as the wide product's ranges
    leave it, also where the block product's cheapest grid is one range (16,384 x 16,384 from 514 rows); with
    ``library_residual_float32`` at any number of rows."""
    ops = Planner()
    for m in (129, 300, 514, 640):
        own, runs = ops._own_product(*operands(m, n, k), None, "sums")
        assert runs and own()[2], m
    ops.library_residual_float32 = True
    for m in (641, 1000, 2048):
        assert ops._own_product(*operands(m, n, k), None, "sums")[0]()[2], m
        x, w = operands(m, n, k)
        assert ops._own_product(x, w[:, :-8], None, "sums")[0]()[2], "the wide product too"
