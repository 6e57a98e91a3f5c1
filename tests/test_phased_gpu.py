"""The phased prefill tiles where they can go wrong: K from the least they take, an odd and an
even number of step pairs, a ragged last row block, one token, several tiles a workgroup (the
next tile's first steps requested in the last two of this one), every output and bias dtype and
scale layout, bit for bit against the CPU oracle."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from helpers import bits, ints, np_, say
from int8_linear import Config, _lib, kernel, tune, w8a8_mm
from oracle import oracle as o

pytestmark = pytest.mark.gpu

TILES = [Config(bm, bn, 128, 4, tune.PHASED, 4) for bm, bn in tune.PHASED_TILES]
ids = lambda c: c.name.replace(" ", "_")


@pytest.mark.parametrize("config", TILES, ids=ids)
@pytest.mark.parametrize("m,k", [(1, 512), (129, 768), (256, 1024), (511, 1280)])
def test_int32_product_is_exact(config, m, k):
    n = 3 * config.bn
    say(f"phased raw {config.name} m={m} k={k} n={n}")
    a, w = ints((m, k), m + k), ints((n, k), n)
    one = torch.ones(1, device="cuda")
    got = w8a8_mm(a, w.t(), one, one, raw=True, config=config)
    assert np.array_equal(np_(got), o.gemm_i32(np_(a), np_(w)))


@pytest.mark.parametrize("config", TILES, ids=ids)
def test_several_tiles_a_workgroup(config):
    """At least two tiles on every workgroup and a ragged third round, called three times."""
    slots = 256 * (2 if config.bm * config.bn == 128 * 128 else 1)
    m, k = 9 * config.bm - 5, 512
    n = config.bn * (-(-(2 * slots + 7) // 9))
    say(f"phased several tiles {config.name} m={m} k={k} n={n}")
    a, w = ints((m, k), 3), ints((n, k), 4)
    one = torch.ones(1, device="cuda")
    ref = o.gemm_i32(np_(a), np_(w))
    for _ in range(3):
        got = w8a8_mm(a, w.t(), one, one, raw=True, config=config)
        assert np.array_equal(np_(got), ref)


@pytest.mark.parametrize("config", TILES, ids=ids)
@pytest.mark.parametrize("tiles_m,tiles_n", [(1, 1), (1, 7), (3, 3), (5, 3), (9, 29), (19, 27)])
def test_tile_counts_that_eight_does_not_divide(config, tiles_m, tiles_n):
    """Every tile is computed once, whatever number of them the 8 XCDs share: fewer than 8, one more
    or less than a multiple, more than the workgroups."""
    m, n, k = tiles_m * config.bm - 3, tiles_n * config.bn, 512
    assert tiles_m * tiles_n % 8
    say(f"phased {config.name} {tiles_m} x {tiles_n} tiles")
    a, w = ints((m, k), tiles_m), ints((n, k), tiles_n)
    one = torch.ones(1, device="cuda")
    got = w8a8_mm(a, w.t(), one, one, raw=True, config=config)
    assert np.array_equal(np_(got), o.gemm_i32(np_(a), np_(w)))


@pytest.mark.parametrize("config", TILES, ids=ids)
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
def test_every_bias_and_scale(config, dtype):
    code = {torch.bfloat16: o.BF16, torch.float16: o.F16, torch.float32: o.F32}
    m, k, n = 300, 512, 2 * config.bn
    a, w = ints((m, k), 31), ints((n, k), 32)
    acc = o.gemm_i32(np_(a), np_(w))
    g = torch.Generator().manual_seed(33)
    for per_row, per_col in ((True, True), (True, False), (False, True)):
        sa = (torch.rand((m, 1) if per_row else (1,), generator=g) * 1e-2 + 1e-3).cuda()
        sb = (torch.rand((n, 1) if per_col else (1,), generator=g) * 1e-2 + 1e-3).cuda()
        for bd in (None, torch.bfloat16, torch.float16, torch.float32):
            say(f"phased {config.name} {dtype} row={per_row} col={per_col} bias={bd}")
            bias = torch.randn(n, generator=g).to(bd).cuda() if bd else None
            got = w8a8_mm(a, w.t(), sa, sb, dtype, bias, config=config)
            b = None if bd is None else np_(bias) if bd == torch.float32 else bits(bias)
            ref = o.epilogue(acc, np_(sa), np_(sb), b, o.NONE if bd is None else code[bd],
                             code[dtype])
            out = np_(got) if dtype == torch.float32 else bits(got)
            assert np.array_equal(out, ref), (per_row, per_col, bd)


def test_wide_strides_leave_the_phased_kernel():
    """Row strides past what 32-bit in-tile offsets hold (256 rows) leave the phased kernel."""
    config, m, k, n = TILES[0], 3, 512, 256
    stride = (2 ** 31 - 1) // 256 + 1 + 15 & ~15
    say(f"phased wide stride {stride}")
    a, w = ints((m, k), 5), ints((n, k), 6)
    wide = torch.zeros((m - 1) * stride + k, dtype=torch.int8, device="cuda")
    view = wide.as_strided((m, k), (stride, 1))
    view.copy_(a)
    one = torch.ones(1, device="cuda")
    got = w8a8_mm(view, w.t(), one, one, raw=True, config=config)
    assert np.array_equal(np_(got), o.gemm_i32(np_(a), np_(w)))


def test_wide_strides_keep_the_plan():
    """A call without a configuration whose token rows lie further apart than the phased tile it
    would launch takes runs the default plan, not the generic kernel, which is nine times slower here
    than packed rows (the plan 1.3 times): three times is allowed."""
    m, k, n = 200, 2560, 9728
    stride = (2 ** 31 - 1) // 256 + 1 + 15 & ~15
    assert kernel.launch_config(m, n, k).stages == tune.PHASED
    say(f"no config, wide stride {stride}")
    a, w = ints((m, k), 7), ints((n, k), 8)
    wide = torch.zeros((m - 1) * stride + k, dtype=torch.int8, device="cuda")
    view = wide.as_strided((m, k), (stride, 1))
    view.copy_(a)
    one = torch.ones(1, device="cuda")
    ref = o.gemm_i32(np_(a), np_(w))

    def us(x):
        best = float("inf")
        for _ in range(10):
            e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            e0.record()
            got = w8a8_mm(x, w.t(), one, one, raw=True)
            e1.record()
            e1.synchronize()
            best = min(best, e0.elapsed_time(e1) * 1e3)
        assert np.array_equal(np_(got), ref)
        return best

    packed, apart = us(a), us(view)
    say(f"{packed:.1f} us packed, {apart:.1f} us apart")
    assert apart < 3 * packed, (packed, apart)


@pytest.mark.parametrize("config", [None, *TILES], ids=lambda c: c.name if c else "none")
@pytest.mark.parametrize("which", ["a", "b", "both"])
def test_rows_in_reverse(config, which):
    """Row strides below 0 through the C entry (a base at the last row): the phased kernel's in-tile
    offsets are unsigned, so such a call leaves it."""
    m, k, n = 300, 512, 2 * (config.bn if config else 192)
    say(f"reversed rows {which} {config.name if config else None}")
    a, w = ints((m, k), 9), ints((n, k), 10)
    one = torch.ones(1, device="cuda")
    out = torch.empty((m, n), dtype=torch.int32, device="cuda")
    ra, rb = which != "b", which != "a"
    lib = _lib.lib()
    status = lib.i8l_w8a8_mm(
        a.data_ptr() + (m - 1) * k * ra, -k if ra else k, 1,
        w.data_ptr() + (n - 1) * k * rb, 1, -k if rb else k, one.data_ptr(), 1, one.data_ptr(), 1,
        None, _lib.DTYPE_NONE, out.data_ptr(), n, _lib.I32, m, n, k,
        kernel._cconfig(config) if config else None, _lib.stream_of(a))
    assert status == _lib.OK, _lib.last_error()
    ref = o.gemm_i32(np_(a)[::-1] if ra else np_(a), np_(w)[::-1] if rb else np_(w))
    assert np.array_equal(np_(out), ref)


@pytest.mark.parametrize("m,k,n", [(129, 512, 640), (300, 2752, 5504), (777, 4096, 1536),
                                   (640, 1920, 768), (200, 448, 320)])
def test_launched_without_a_config(m, k, n):
    """What a call without a configuration launches (the macro tile with the least modelled time, or
    the plan where none divides the shape), against the oracle."""
    say(f"launch_config m={m} k={k} n={n}: {kernel.launch_config(m, n, k).name}")
    a, w = ints((m, k), m), ints((n, k), n)
    sa = torch.rand((m, 1), generator=torch.Generator().manual_seed(1)).cuda() * 1e-2
    sb = torch.rand((n, 1), generator=torch.Generator().manual_seed(2)).cuda() * 1e-2
    got = w8a8_mm(a, w.t(), sa, sb)
    ref = o.epilogue(o.gemm_i32(np_(a), np_(w)), np_(sa), np_(sb), None, o.NONE, o.BF16)
    assert np.array_equal(bits(got), ref)
