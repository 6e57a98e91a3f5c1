"""The shared-ring decode tile where it can go wrong: every row count it is built for, with a
ragged and a full last fragment and a second row block, fewer steps than the ring has slots and
many more, K split into parts of unequal steps, every epilogue, and the workspace rules of a
split; bit for bit against the CPU oracle."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from helpers import bits, ints, np_, say
from int8_linear import Config, _lib, kernel, w8a8_mm
from oracle import oracle as o

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("bm", range(32, 129, 16))
@pytest.mark.parametrize("steps,parts", [(1, 1), (5, 1), (13, 1), (40, 1), (8, 8), (17, 3),
                                         (29, 2), (50, 7)])
def test_int32_product_is_exact(bm, steps, parts):
    config = Config(bm, 64, 128, 8, 6, parts)
    k, n = 128 * steps, 192
    a, w = ints((2 * bm - 3, k), bm + steps), ints((n, k), steps)
    one = torch.ones(1, device="cuda")
    ref = o.gemm_i32(np_(a), np_(w))
    for m in (1, bm - 5, bm, 2 * bm - 3):
        say(f"shared ring {config.name} m={m} k={k}")
        got = w8a8_mm(a[:m], w.t(), one, one, raw=True, config=config)
        assert np.array_equal(np_(got), ref[:m]), m


@pytest.mark.parametrize("parts", [1, 3])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
def test_every_bias_and_scale(parts, dtype):
    code = {torch.bfloat16: o.BF16, torch.float16: o.F16, torch.float32: o.F32}
    m, k, n = 75, 2688, 192
    config = Config(80, 64, 128, 8, 6, parts)
    a, w = ints((m, k), 41), ints((n, k), 42)
    acc = o.gemm_i32(np_(a), np_(w))
    g = torch.Generator().manual_seed(43)
    for per_row, per_col in ((True, True), (True, False), (False, True)):
        sa = (torch.rand((m, 1) if per_row else (1,), generator=g) * 1e-2 + 1e-3).cuda()
        sb = (torch.rand((n, 1) if per_col else (1,), generator=g) * 1e-2 + 1e-3).cuda()
        for bd in (None, torch.bfloat16, torch.float16, torch.float32):
            say(f"shared ring parts={parts} {dtype} row={per_row} col={per_col} bias={bd}")
            bias = torch.randn(n, generator=g).to(bd).cuda() if bd else None
            got = w8a8_mm(a, w.t(), sa, sb, dtype, bias, config=config)
            b = None if bd is None else np_(bias) if bd == torch.float32 else bits(bias)
            ref = o.epilogue(acc, np_(sa), np_(sb), b, o.NONE if bd is None else code[bd],
                             code[dtype])
            out = np_(got) if dtype == torch.float32 else bits(got)
            assert np.array_equal(out, ref), (per_row, per_col, bd)


@pytest.mark.parametrize("m,k,n", [(20, 3584, 4608), (48, 5120, 5120), (75, 1792, 4096),
                                   (100, 13824, 5120), (128, 8192, 10240), (100, 18944, 3584)])
def test_launched_without_a_config(m, k, n):
    """Untuned decode batches: the launched tile's output, repeated and in a HIP graph (its split's
    partial planes come from the graph's pool), against the plan's."""
    c = kernel.launch_config(m, n, k)
    say(f"launch_config m={m} k={k} n={n}: {c.name}")
    a, w = ints((m, k), m), ints((n, k), n)
    sa = torch.rand((m, 1), generator=torch.Generator().manual_seed(1)).cuda() * 1e-2
    sb = torch.rand((n, 1), generator=torch.Generator().manual_seed(2)).cuda() * 1e-2
    ref = w8a8_mm(a, w.t(), sa, sb, config=kernel.default_config(m, n, k))
    for _ in range(3):
        assert torch.equal(w8a8_mm(a, w.t(), sa, sb), ref)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = w8a8_mm(a, w.t(), sa, sb)
    for _ in range(3):
        out.zero_()
        graph.replay()
        assert torch.equal(w8a8_mm(a, w.t(), sa, sb), ref)
        assert torch.equal(out, ref)


def test_no_split_without_a_workspace():
    """A call with no configuration and no workspace never picks a split of K (i8l_w8a8_mm and
    w8a8_mm_noalloc took every shape before there was one to pick)."""
    m, k, n = 100, 13824, 5120
    say(f"noalloc m={m} k={k} n={n}")
    a, w = ints((m, k), 7), ints((n, k), 8)
    sa, sb = torch.rand(m, 1).cuda() * 1e-2, torch.rand(n, 1).cuda() * 1e-2
    assert kernel.launch_config(m, n, k).group_m > 1
    out = torch.empty((m, n), dtype=torch.bfloat16, device="cuda")
    kernel.w8a8_mm_noalloc(a, w.t(), sa, sb, out)
    assert torch.equal(out, w8a8_mm(a, w.t(), sa, sb))
    c = kernel._cconfig(Config(112, 64, 128, 8, 6, 3))
    assert _lib.lib().i8l_w8a8_mm_workspace_bytes(m, n, k, c) == 3 * m * n * 4


@pytest.mark.parametrize("m,k,n", [(48, 13824, 5120), (75, 18944, 3584), (100, 13824, 5120)])
def test_no_config_leaves_a_workspace_alone(m, k, n):
    """i8l_w8a8_mm_ws without a configuration does not split K, however large the workspace it is
    handed: i8l_w8a8_mm_workspace_bytes gives 0 for such a call, so several in flight may share
    one."""
    say(f"ws with no config m={m} k={k} n={n}")
    a, w = ints((m, k), 7), ints((n, k), 8)
    sa, sb = torch.rand(m).cuda() * 1e-2, torch.rand(n).cuda() * 1e-2
    assert kernel.launch_config(m, n, k).group_m > 1      # the pick with a workspace
    lib = _lib.lib()
    assert lib.i8l_w8a8_mm_workspace_bytes(m, n, k, None) == 0
    ws = torch.full((32 * m * n,), 0x5a, dtype=torch.uint8, device="cuda")
    out = torch.empty((m, n), dtype=torch.bfloat16, device="cuda")
    status = lib.i8l_w8a8_mm_ws(a.data_ptr(), k, 1, w.data_ptr(), 1, k, sa.data_ptr(), m,
                                sb.data_ptr(), n, None, _lib.DTYPE_NONE, out.data_ptr(), n,
                                _lib.BF16, m, n, k, ws.data_ptr(), ws.numel(), None,
                                _lib.stream_of(a))
    assert status == _lib.OK, _lib.last_error()
    assert torch.equal(out, w8a8_mm(a, w.t(), sa, sb))
    assert bool((ws == 0x5a).all())
