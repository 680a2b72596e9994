"""Which kernel and grid a product or an attention runs, by its sizes alone: the choices of ``kernels/ops.py``, played on the CPU,
mostly with tensors that have sizes and no memory.  The grids named were timed on a device of 256 compute units."""

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

    def _block_product(self, x, weight, bias, *, plan, gated, sums, rule):
        return "block", plan, plan[1] > 1 or sums

    def gemm_stream(self, x, weight, bias=None, *, plan, gated=False, rule=None):
        return "stream", plan, gated

    def gemm_tiled(self, x, weight, bias=None, *, max_splits=None, plan=None, gated=False, rule=None):
        return "tiled", plan, gated

    def swiglu(self, gate_up, dtype, paired, rule):
        return ("sums, unit", *gate_up[:2])

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


@pytest.mark.parametrize("n,k,first,last", [(3584, 3584, 1574, 1690), (4608, 3584, 1224, 1314), (3072, 3072, 1601, 1661), (5120, 8192, 1281, 1321),
                                            (6144, 16384, 1921, 2048)])
def test_a_wider_tile_takes_no_bits_from_the_residual_stream(n, k, first, last):
    """Rows at which the tiles of 128, 160 and 256 weight rows are cheapest as several ranges of K, whose sums are 32-bit: the addend stays 32-bit where
    one range of 192 or 224 weight rows is sooner, too.  Beside them one range is rounded once."""
    for m in range(first, last + 1):
        assert Planner()._own_product(*operands(m, n, k), None, "sums")[0]()[2], m
    assert not Planner()._own_product(*operands(2048, 3584, 3584), None, "sums")[0]()[2]


@pytest.mark.parametrize("n,k", [(3584, 18944), (3584, 3584), (5120, 13824), (5120, 5120), (2048, 8192), (2048, 2048), (4096, 14336), (6144, 6144),
                                 (8192, 29568)])
def test_an_addend_is_32_bit_wherever_the_first_tiles_leave_it_so(n, k):
    first = tuple(tile for tile in Ops._BLOCK_TILES if tile[0] in (4, 5, 8))
    for m in range(641, 2049, 32):
        ops = Planner()
        assert ops._own_product(*operands(m, n, k), None, "sums")[0]()[2] >= (ops._block_cheapest(m, n, k, "sums", first)[1] > 1), m


def test_one_result_of_a_narrow_product_is_left_to_the_library():
    """A product as one range of K runs the block kernel only from a grid on that fills enough of the device.
    The shapes on the left were up to 2.4 times as slow with it as with the library, those on the right up to 1.5 times as fast."""
    ops = Planner()

    def runs(m, n, k, kind):
        return ops._own_product(*operands(m, n, k), None, kind)[1]

    for m, n, k in ((160, 1024, 4096), (129, 768, 3072), (512, 2048, 8192), (256, 3584, 3584), (300, 4608, 3584), (300, 3072, 2048), (1024, 1024, 4096)):
        assert not runs(m, n, k, "one"), (m, n, k)
    for m, n, k in ((400, 4608, 3584), (512, 4608, 3584), (2048, 4608, 3584), (2016, 7168, 5120), (300, 10304, 2048), (160, 18944, 3584), (2048, 2048, 8192)):
        assert runs(m, n, k, "one"), (m, n, k)
    for m, n, k in ((160, 1024, 4096), (512, 2048, 8192), (256, 3584, 3584), (300, 2816, 2048), (129, 2816, 2048)):
        assert not runs(m, n, k, "gated"), (m, n, k)
    for m, n, k in ((160, 1024, 1024), (256, 5632, 2048), (700, 3584, 3584), (129, 16384, 2048), (129, 37888, 3584), (129, 27648, 5120)):
        assert runs(m, n, k, "gated"), (m, n, k)
    ops.wide_default_rows = 0
    assert not any(runs(m, 37888, 3584, kind) for m in (200, 2048) for kind in ("one", "gated", "sums"))


def test_short_ranges_of_partial_sums_run_the_wide_product():
    """Up to ``wide_default_rows`` rows and eleven iterations of 64 a range; 32-bit sums either way."""
    ops = Planner()

    def picked(m, n, k):
        own, runs = ops._own_product(*operands(m, n, k), None, "sums")
        kernel, plan, float32 = own()
        assert runs and (float32 or m > 640), (m, n, k)
        return kernel

    for m, n, k in ((512, 2048, 2048), (640, 2048, 2048), (400, 1024, 4096), (256, 1536, 2048), (640, 512, 512), (256, 768, 3072)):
        assert picked(m, n, k) == "wide", (m, n, k)
    for m, n, k in ((129, 3584, 3584), (299, 3584, 18944), (640, 5120, 13824), (700, 2048, 2048), (300, 2048, 8192), (640, 2560, 2560)):
        assert picked(m, n, k) == "block", (m, n, k)


def test_tiles_of_224_weight_rows_take_the_matrices_that_16_of_them_cover():
    """At 2,048 rows they fill their rounds of workgroups; two ranges of them, at 1,729 to 1,792, leave an eighth of the units without one and are the
    cheapest grid there all the same."""
    ops = Planner()
    assert ops._block_plan(2048, 3584, 18944, "sums") == (148, 2, 7, 8) and ops._block_plan(2048, 3584, 3584, "sums") == (56, 1, 7, 4)
    assert ops._block_plan(2048, 7168, 5120, "one") == (80, 1, 7, 8)
    for m in (1729, 1768, 1792):
        assert ops._block_plan(m, 3584, 18944, "sums") == (148, 2, 7, 8), m


def test_a_norm_waits_for_a_product_that_makes_it(monkeypatch):
    """One row up to 6,144 wide and two up to 3,072, as 32-bit sums of up to four ranges, for a matrix that the streaming product takes; every
    other norm runs by itself."""
    monkeypatch.setattr("turboserve_amd.kernels.ops._gpu", lambda *tensors: None)
    ops = Planner()

    def waits(rows, n, k, gated=False, sums=2, dtype=torch.bfloat16, pending=True):
        parts = torch.empty(sums, rows, k, device="meta") if pending else None
        gain, matrix = torch.empty(k, dtype=dtype, device="meta"), torch.empty(n, k, dtype=dtype, device="meta")
        residual = torch.empty(rows, k, device="meta")
        norm = ops.waiting_norm(residual, parts, gain, 1e-6, matrix, gated=gated)
        assert norm is None or (norm.after.shape == residual.shape and norm.after is not residual)
        return norm is not None

    assert waits(1, 4608, 3584) and waits(1, 37888, 3584, gated=True) and waits(2, 16384, 2048, gated=True) and waits(1, 9216, 6144) and waits(2, 6144, 3072)
    assert not waits(2, 4608, 3584) and not waits(3, 3072, 2048) and not waits(1, 8192, 8192) and not waits(1, 4608, 3584, sums=5)
    assert not waits(1, 4608, 3584, pending=False) and not waits(1, 4608, 3584, dtype=torch.float32) and not waits(1, 4608, 3592) and not waits(1, 96, 3584)
    assert not waits(1, 27648, 5120, gated=True) and not waits(1, 3584, 18944, gated=True)  # tiles or several ranges are sooner
    parts = torch.empty(1, 3584, dtype=torch.bfloat16, device="meta")  # one result of the run's type
    gain, matrix = torch.empty(3584, dtype=torch.bfloat16, device="meta"), torch.empty(4608, 3584, dtype=torch.bfloat16, device="meta")
    assert ops.waiting_norm(torch.empty(1, 3584, device="meta"), parts, gain, 1e-6, matrix, gated=False) is None


@pytest.mark.parametrize("n,k,ranges", [(8224, 2048, 1), (10304, 2048, 1), (12288, 2048, 1), (8224, 1792, 3), (10304, 1920, 2), (18944, 1792, 1), (4608, 3584, 3)])
def test_products_that_make_their_rows_have_the_grid_of_their_own_tiles(monkeypatch, n, k, ranges):
    """They run in tiles of 32 weight rows, as many ranges of K as are the cheapest with those; over a K of 2,048, whose halves two ranges read slowly, one,
    where the product of plain rows takes tiles of 16; the norm that waits and the product launch one plan."""
    from turboserve_amd.kernels.ops import WaitingHeads

    monkeypatch.setattr("turboserve_amd.kernels.ops._gpu", lambda *tensors: None)
    ops, seen = Planner(), {}

    class Core:
        def __getattr__(self, name):
            return lambda *operands: seen.update({name: operands}) or 0

    ops.core, ops.stream = Core(), lambda: None
    weight = torch.empty(n, k, dtype=torch.bfloat16)
    cheapest = min(range(1, 9), key=lambda want: ops._stream_cost(n, k, want))
    assert k == 2048 or cheapest == ranges
    norm = ops.waiting_norm(torch.zeros(1, k), torch.zeros(2, 1, k), torch.ones(k, dtype=torch.bfloat16), 1e-6, weight, gated=False)
    assert ops.linear(norm, weight).shape == (ranges, 1, n)
    per_wave = -(-k // 64 // (4 * ranges))
    assert seen["ts_gemm_stream_normed"][-7:-5] == (per_wave, ranges)
    assert ops.linear(WaitingHeads(torch.zeros(k // 128, 4, 128), torch.zeros(k // 128, 4, 2)), weight).shape == (ranges, 1, n)
    assert seen["ts_gemm_stream_heads"][-3:-1] == (per_wave, ranges)
    assert ops._stream_plan(n, k, None) == (per_wave, ranges, 1 if k == 2048 else 2)


@pytest.mark.parametrize("gated", [False, True])
def test_what_waits_is_for_the_matrix_it_was_made_for(monkeypatch, gated):
    """A norm or heads that wait are not multiplied by a matrix that the launch would read past its end or by the wrong type; a step without rows has a
    norm of its own."""
    from turboserve_amd.kernels.ops import KernelError, WaitingHeads

    monkeypatch.setattr("turboserve_amd.kernels.ops._gpu", lambda *tensors: None)
    ops, k = Planner(), 2048
    gain, residual, pending = torch.ones(k, dtype=torch.bfloat16), torch.zeros(1, k), torch.zeros(2, 1, k)
    norm = ops.waiting_norm(residual, pending, gain, 1e-6, torch.zeros(256, k, dtype=torch.bfloat16), gated=gated)
    heads = WaitingHeads(torch.zeros(16, 4, 128), torch.zeros(16, 4, 2))
    refused = [torch.zeros(256, k - 64, dtype=torch.bfloat16), torch.zeros(256, k), torch.zeros(k, 256, dtype=torch.bfloat16).t(),
               torch.zeros(256 * k + 4, dtype=torch.bfloat16)[4:].view(256, k), torch.zeros(256 * k, dtype=torch.bfloat16)]
    assert refused[3].data_ptr() % 16
    for matrix in refused:
        with pytest.raises(KernelError):
            (ops.linear_swiglu if gated else ops.linear)(norm, matrix)
        with pytest.raises(KernelError):
            ops.linear(heads, matrix)
    with pytest.raises(KernelError):  # no workgroup for the last elements of the sum
        (ops.linear_swiglu if gated else ops.linear)(norm, torch.zeros(32, k, dtype=torch.bfloat16))
    assert ops.waiting_norm(residual[:0], pending[:, :0], gain, 1e-6, torch.zeros(256, k, dtype=torch.bfloat16), gated=gated) is None


def test_a_gated_product_of_other_than_rows_is_refused_as_any_product(monkeypatch):
    from turboserve_amd.kernels.ops import KernelError

    monkeypatch.setattr("turboserve_amd.kernels.ops._gpu", lambda *tensors: None)
    for x, w in ((torch.zeros(2, 3, 32), torch.zeros(64, 32)), (torch.zeros(32), torch.zeros(64, 32)), (torch.zeros(3, 32), torch.zeros(2, 64, 32))):
        with pytest.raises(KernelError):
            Planner().linear_swiglu(x, w)


def test_the_store_of_heads_adds_up_what_few_rows_leave():
    """A prompt's q|k|v as two to four 32-bit sums wherever those are the model's cheapest grid (up to ``wide_default_rows`` rows), one result elsewhere."""
    ops = Planner()

    def ranges(m, n, k):
        plan = ops._sums_plan(*operands(m, n, k), None)
        return plan and plan[1]

    for n, k in ((4608, 3584), (7168, 5120), (3072, 2048), (1536, 1024)):
        for m in range(129, 513, 19):
            assert 2 <= ranges(m, n, k) <= 4, (m, n, k)
        assert ranges(128, n, k) is None and ranges(641, n, k) is None and ranges(2048, n, k) is None
    assert ranges(640, 4608, 3584) is None and ranges(509, 12288, 4096) is None and ranges(640, 3072, 2048) == 2


def test_32_bit_attention_is_asked_only_for_what_it_takes():
    """Pages of 24 keys and pages or rows that 16-byte accesses do not fit stay with the kernel that takes any geometry."""
    ops = Planner()

    def asked(page=16, dim=64, value_dim=64, shift=0, stride=256, dtype=torch.float32):
        room = torch.zeros(4 * page * max(dim, value_dim) + 4, dtype=dtype)
        k = room[shift: shift + 2 * page * dim].view(1, 2, page, dim)
        v = room[: 2 * page * value_dim].view(1, 2, value_dim, page)
        return ops.float32_attention_supported(torch.zeros(3, stride, dtype=dtype), stride, k, v)

    assert asked() and asked(page=64) and asked(dim=128, value_dim=128)
    assert not asked(page=24) and not asked(page=8) and not asked(page=48)
    assert not asked(shift=1) and asked(shift=4)
    assert not asked(stride=257) and not asked(dim=72, value_dim=72) and not asked(value_dim=32) and not asked(dtype=torch.bfloat16)


def test_wide_matrices_at_17_to_128_rows():
    """(ranges of K, tile of weight rows) of the block product, ungated: what was fastest of the grids timed, or within a few percent of it.
    A matrix beyond 16,384 rows had run as one range of tiles of 128 whatever its width: 37,888 x 3,584 in two rounds,
    up to 1.3 times as slow as the kernels before."""
    plan = Planner()._block_few_plan
    for m in (17, 24, 32, 64, 100, 128):
        assert plan(m, 18944, 3584, None)[1:3] == (2, 5) and plan(m, 20480, 5120, None)[1:3] == (2, 5)
        assert plan(m, 32768, 4096, None)[1:3] == (1, 4)
        assert plan(m, 34944, 3584, None)[1:3] == (1, 5) and plan(m, 37888, 3584, None)[1:3] == (1, 5)
        assert plan(m, 55296, 5120, None)[1:3] == (1, 8)
        assert plan(m, 3584, 18944, None)[1:3] == (9, 4) and plan(m, 2048, 2048, None)[1:3] == (8, 2)
        assert (plan(m, 24576, 4096, None) is None) == (m == 64)
        for max_splits in (1, None):  # tiles of 256 over a long K
            assert (plan(m, 59136, 8192, max_splits) is None) == (m <= 64)
        assert plan(m, 59136, 7168, 1)[1:3] == (1, 8) and plan(m, 37888, 3584, 1)[1:3] == (1, 5)
    assert plan(64, 8192, 2048, None)[1:3] == (4, 4) and plan(128, 8192, 2048, None)[1:3] == (2, 2)
    assert plan(128, 16384, 2048, None)[1:3] == (1, 2) and plan(64, 16384, 2048, None)[1:3] == (2, 4)
    assert plan(128, 10304, 2048, None)[1:3] == (3, 4)


@pytest.mark.parametrize("m", [17, 32, 64, 65, 128])
def test_grids_of_17_to_128_rows_cover_k(m):
    """Whatever the sizes and the ranges allowed, the ranges cover K without an empty one."""
    ops = Planner()
    for n in (16, 272, 2048, 3584, 8192, 16400, 20480, 20496, 24576, 33000, 40960, 41000, 65536, 65552, 152064):
        for k in (64, 128, 384, 448, 2048, 3584, 4160, 8192, 18944):
            for max_splits in (None, 1, 2, 5):
                plan = ops._block_few_plan(m, n, k, max_splits)
                if plan is not None:
                    per_split, splits, tn, tm = plan
                    assert splits == -(-(k // 64) // per_split) and 1 <= splits <= (max_splits or 12)
                    assert (tn, tm) in {(a, b) for a in (2, 4, 5, 8) for b in (1, 2, 4)} and m <= 32 * tm


def test_gated_products_of_up_to_16_rows(monkeypatch):
    """A gated product runs as one range of K where that costs no more than a launch of the unit's own; over a long K on few
    units it took up to 1.4 times what partial sums and the unit take."""
    monkeypatch.setattr("turboserve_amd.kernels.ops._gpu", lambda *tensors: None)
    ops = Planner()
    for n, k in ((3584, 18944), (5120, 13824), (2048, 8192), (1024, 4096), (768, 3072)):
        kernel, product, plan = ops.linear_swiglu(*operands(16, n, k))
        assert (kernel, product) == ("sums, unit", "stream") and plan[1] > 1, (n, k)
    for n, k in ((37888, 3584), (16384, 2048), (3584, 3584), (4608, 3584), (2816, 2048), (512, 512), (8192, 8192)):
        kernel, plan, gated = ops.linear_swiglu(*operands(1, n, k))
        assert kernel == "stream" and plan[1] == 1 and gated, (n, k)
    assert ops.linear_swiglu(*operands(8, 27648, 5120))[0] == "tiled"


@pytest.mark.parametrize("m", [17, 64, 128, 129, 300, 1000])
@pytest.mark.parametrize("kind", ["sums", "one", "gated"])
def test_a_product_looks_at_its_operands_once(monkeypatch, m, kind):
    """Choosing the block product asks whether it takes the operands; launching it does not ask again, and the choice is worked out
    once for all products of the same sizes: the host's share of a short prompt's step."""
    monkeypatch.setattr("turboserve_amd.kernels.ops._gpu", lambda *tensors: None)
    ops, asked, planned = Planner(), [], []
    ops.time_wide_choices = False
    monkeypatch.setattr(ops, "block_supported", lambda x, w: asked.append(1) or Ops.block_supported(x, w), raising=False)
    for name in ("_block_plan", "_wide_plan"):
        monkeypatch.setattr(ops, name, lambda *a, plan=getattr(ops, name): planned.append(1) or plan(*a), raising=False)
    x, w = operands(m, 37888, 3584)
    product = {"sums": lambda: ops.linear(x, w, for_residual=True), "one": lambda: ops.linear(x, w), "gated": lambda: ops.linear_swiglu(x, w)}[kind]
    assert product()[0] == "block" and len(asked) == 1
    planned.clear()
    assert product()[0] == "block" and len(asked) == 2 and not planned


@pytest.mark.parametrize("m,n,k,kernel", [
    (1, 8192, 2048, "stream"), (8, 2048, 8192, "stream"), (1, 20480, 5120, "tiled"), (40, 37888, 3584, "block"), (64, 8192, 2048, "block"),
    (200, 16384, 2048, "block"), (160, 1024, 4096, "library"), (400, 8192, 1544, "wide"),
])
def test_the_unit_of_a_product_asks_for_the_products_choice_once(monkeypatch, m, n, k, kernel):
    """max(y, 0)^2 in the product's launch where that is one range of the streaming or the block kernel, else behind the product that ``linear`` runs, whose
    choice is not worked out a second time: a prompt of a small model is bound by the host."""
    monkeypatch.setattr("turboserve_amd.kernels.ops._gpu", lambda *tensors: None)
    ran, asked = [], []

    class Squares(Planner):
        def _block_product(self, x, weight, bias, *, plan, gated, sums, rule, squared=False):
            ran.append(("block", squared))
            return "block", plan[1] > 1

        def gemm_stream(self, x, weight, bias=None, *, plan, gated=False, rule=None, squared=False):
            ran.append(("stream", squared))
            return "stream", plan[1] > 1

        def gemm_wide(self, *operands, **more):
            ran.append(("wide", False))
            return "wide", more["plan"][1] > 1

        def gemm_tiled(self, *operands, **more):
            ran.append(("tiled", False))
            return "tiled", True

        def _library_product(self, *operands):
            ran.append(("library", False))
            return "library", False

        def activate(self, product, kind, dtype):
            assert kind == "relu_squared" and dtype == torch.bfloat16
            ran.append("unit")
            return product

    ops = Squares()
    ops.time_wide_choices = False
    for name in ("block_supported", "_own_choice", "_stream_runs", "_block_few_runs", "_wide_runs"):
        monkeypatch.setattr(ops, name, lambda *of, name=name, real=getattr(ops, name): asked.append(name) or real(*of), raising=False)
    x, w = operands(m, n, k)
    _, ranges = ops.linear_relu_squared(x, w)
    alone = kernel in ("stream", "block") and not ranges
    assert ran == ([(kernel, True)] if alone else [(kernel, False), "unit"])
    assert kernel == "tiled" or max(map(asked.count, asked)) == 1
    ran.clear()
    assert ops.linear(x, w)[0] == kernel  # the same product without the unit


@pytest.mark.parametrize("n,k,ranges", [(8320, 3136, 3), (8320, 3584, 3), (8704, 3584, 3), (8320, 4608, 4), (9728, 3584, 3), (12288, 3584, 2), (18944, 3584, 2), (2048, 8192, 3)])
def test_finer_grids_over_a_long_k_leave_a_wavefront_five_slices(n, k, ranges):
    """Five ranges of 8,320 x 3,584, three slices a wavefront, were slower than three."""
    per_wave, splits, tile = Planner()._stream_plan(n, k, None)
    assert (splits, tile) == (ranges, 2) and per_wave == -(-k // 64 // (4 * ranges)) and per_wave >= 5


def test_one_range_with_a_nearly_empty_last_round_is_left_to_the_tiled_product():
    ops = Planner()
    assert ops._stream_plan(20480, 5120, None) is None and ops._stream_plan(27648, 5120, 1) is None and ops._stream_plan(17408, 2048, 1) is None
    for n, k in ((18944, 3584), (37888, 3584), (17408, 2048), (55296, 5120), (8192, 8192), (5120, 5120)):
        assert ops._stream_plan(n, k, None) is not None, (n, k)


def test_a_steps_estimate_holds_what_its_products_and_attention_leave():
    """No plan's partial sums are larger than what the sizing of the cache leaves room for, and a 32-bit model's estimate holds the
    scratch of its single tokens' attention."""
    from turboserve_amd.weights.random_init import describe_model

    ops = Planner()
    for n in (512, 2048, 3584, 5120, 7168, 8192, 16384):
        for k in (512, 2048, 3584, 8192, 18944, 29568, 65536):
            for m in (1, 16, 17, 64, 128, 129, 257, 640, 641, 1024, 1788, 2048, 2500, 4096, 8192, 16384):
                splits = [1]
                if m <= 128:
                    splits += [ops._tiled_plan(m, n, k, None)[1], ops._wide_plan_few_rows(m, n, k, None)[1]]
                    few = ops._block_few_plan(m, n, k, None) if m > 16 else ops._stream_plan(n, k, None)
                    splits += [few[1] if few else 1]
                else:
                    splits += [ops._block_plan(m, n, k, "sums")[1]] + ([ops._wide_plan(m, n, k, False)[1]] if m <= 640 else [])
                assert 4 * max(splits) * m * n <= Ops.partial_sums_bytes(m, n), (m, n, k, splits)
    config = {
        "architectures": ["Qwen2ForCausalLM"], "model_type": "qwen2", "hidden_size": 3584, "num_hidden_layers": 2, "num_attention_heads": 28,
        "num_key_value_heads": 4, "head_dim": 128, "intermediate_size": 18944, "vocab_size": 1000, "rope_theta": 1e6, "rms_norm_eps": 1e-6,
        "tie_word_embeddings": False, "use_sliding_window": False, "max_position_embeddings": 32768,
    }
    _, model = describe_model(config)
    sums = max(4 * ops._block_plan(m, 3584, 18944, "sums")[1] * m * 3584 for m in range(129, 2049))
    assert sums > 4 * 2048 * 3584  # more than one 32-bit result of the largest step: whatever plans are chosen, some are several ranges
    stream = 2 * 2048 * 3584 * 8
    products = 2048 * (3 * 18944 * 2 + 3584 * 4)  # gate|up, its units, what the stream waits for
    assert model.activation_bytes(2048, 64, 2) >= stream + products + sums
    assert model.activation_bytes(64, 64, 4) >= Ops.float32_attention_scratch


def test_only_a_head_is_asked_for_rounds(monkeypatch):
    """A decode-sized product knows its grid; only a matrix of more weight rows than a round of tiles of 256 is looked at for whole rounds
    and a rest (asked for every gated product, with a loop over one launch in each product: 2% of a short prompt of eight layers 2,048 wide)."""
    monkeypatch.setattr("turboserve_amd.kernels.ops._gpu", lambda *tensors: None)
    ops, asked = Planner(), []
    monkeypatch.setattr(ops, "_block_few_rounds", lambda *of: asked.append(of) or Ops._block_few_rounds(ops, *of), raising=False)
    for n, k in ((16384, 2048), (37888, 3584), (65280, 2048)):
        ops._block_few_runs(*operands(31, n, k), None, 1)
    assert not asked
    assert len(ops._block_few_runs(*operands(64, 152064, 3584), None, 1)) == 7 and asked == [(64, 152064, 3584)]
