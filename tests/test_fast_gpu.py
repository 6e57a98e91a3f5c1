"""The C++ eager binding (csrc/i8l_torch.cpp) on the GPU: every call it takes launches the
same kernel as the ctypes path and gives the same bits; every call it declines comes back
to the Python path, with the reference's errors; it honours the caller's stream and graph
capture.  The launch counter shows which path ran."""

from __future__ import annotations

from dataclasses import astuple

import pytest
import torch

from helpers import ints, randn, say
from int8_linear import Config, _lib, kernel
from int8_linear import fused_quant as fq
from int8_linear import vllm_patch
from int8_linear.kernel import NotSupported, choose_config, w8a8_mm

pytestmark = pytest.mark.gpu


@pytest.fixture
def ctypes_only(monkeypatch):
    """Set the binding aside: the wrappers then launch through ctypes."""
    def off():
        monkeypatch.setattr(_lib, "_fast_mod", None)
    return off


def fast():
    f = _lib.fast()
    assert f is not None, "the binding is built with the library"
    return f


@pytest.mark.parametrize("m,k,n", [(1, 2048, 4096), (16, 2048, 2048), (37, 2048, 12288),
                                   (96, 6144, 2048), (300, 2048, 2048), (1024, 4096, 4096),
                                   (96, 14336, 4096)])   # the last: a split of K (workspace)
@pytest.mark.parametrize("bias_dtype", [None, torch.bfloat16, torch.float32])
def test_mm_binding_equals_ctypes_path(m, k, n, bias_dtype, ctypes_only):
    say(f"binding mm m={m} k={k} n={n} bias={bias_dtype}")
    a, w = ints((m, k), m), ints((n, k), n)
    g = torch.Generator().manual_seed(m + n)
    sa = (torch.rand((m, 1), generator=g) * 1e-2 + 1e-3).cuda()
    sb = (torch.rand((n, 1), generator=g) * 1e-2 + 1e-3).cuda()
    bias = torch.randn(n, generator=g).to(bias_dtype).cuda() if bias_dtype else None
    before = fast().launches()
    got = w8a8_mm(a, w.t(), sa, sb, torch.bfloat16, bias)
    assert fast().launches() == before + 1
    cfg = choose_config(m, n, k)
    assert fast().config_for(a.get_device(), m, n, k) == (cfg.bm, cfg.bn, cfg.bk, cfg.warps,
                                                          cfg.stages, cfg.group_m)
    cfg = kernel.launch_config(m, n, k)
    assert fast().launch_config_for(a.get_device(), m, n, k) == astuple(cfg)
    if (m, k, n) == (96, 14336, 4096):
        assert cfg.stages == 6 and cfg.group_m > 1, cfg.name  # the shipped table splits K here
    ctypes_only()
    ref = w8a8_mm(a, w.t(), sa, sb, torch.bfloat16, bias)
    torch.cuda.synchronize()
    assert torch.equal(got.view(torch.int16), ref.view(torch.int16))


def test_binding_launches_what_launch_config_says():
    """The binding's choice is kernel.launch_config's at every tuned bucket, between them and at
    shapes without an entry: the plan, a replaced plan, a split of K."""
    dev, seen = torch.cuda.current_device(), set()
    w8a8_mm(ints((1, 2048), 1), ints((2048, 2048), 2).t(), torch.ones(1, device="cuda"),
            torch.ones(1, device="cuda"))                # the first call hands the table over
    shapes = [tuple(map(int, kn.split("x"))) for kn in kernel._device_table(dev)]
    for k, n in shapes + [(13824, 5120), (2560, 9728), (4096, 5504), (2752, 4096), (64, 48)]:
        for m in (1, 9, 16, 23, 64, 75, 96, 100, 128, 129, 136, 145, 161, 168, 200, 256, 257, 300,
                  512, 513, 768, 777, 1024, 1025, 4096, 5000):
            c, plan = kernel.launch_config(m, n, k), choose_config(m, n, k)
            assert fast().launch_config_for(dev, m, n, k) == astuple(c), (m, n, k)
            seen.add((c == plan, c.stages == 6 and c.group_m > 1))
    assert {(True, False), (False, False), (False, True)} <= seen


def test_binding_launches_a_tuned_split_of_k():
    """A table whose entry is a stages-5 split (the shipped one holds none): the binding launches it
    with a workspace of its own, with the unsplit tile's bits."""
    m, k, n = 96, 14336, 4096
    split = Config(64, 64, 128, 4, 5, 2)
    a, w = ints((m, k), m), ints((n, k), n)
    sa, sb = torch.rand((m, 1)).cuda() * 1e-2, torch.rand((n, 1)).cuda() * 1e-2
    ref = w8a8_mm(a, w.t(), sa, sb, config=kernel.default_config(m, n, k))
    dev = a.get_device()
    say(f"binding mm split {split.name} m={m} k={k} n={n}")
    fast().set_table(dev, [[k, n, m, *astuple(split)]])
    try:
        assert fast().launch_config_for(dev, m, n, k) == astuple(split)
        before = fast().launches()
        got = w8a8_mm(a, w.t(), sa, sb)
        assert fast().launches() == before + 1
    finally:
        fast().set_table(dev, kernel._table_rows(dev))
    assert torch.equal(got, ref)


def test_mm_binding_declines_to_the_python_path():
    a, w = ints((8, 2048), 1), ints((2048, 2048), 2)
    sa2 = torch.rand((8, 2), device="cuda") + 0.5
    sb = torch.rand((2048,), device="cuda") + 0.5
    before = fast().launches()
    # a strided scale view: the Python path copies it, with the same result
    got = w8a8_mm(a, w.t(), sa2[:, :1], sb, torch.bfloat16)
    ref = w8a8_mm(a, w.t(), sa2[:, :1].contiguous(), sb, torch.bfloat16)
    assert fast().launches() == before + 1          # only the contiguous call was taken
    assert torch.equal(got, ref)
    with pytest.raises(NotSupported):                # dtype errors keep their exception
        w8a8_mm(a, w.t(), sa2[:, 0].double(), sb)
    with pytest.raises(ValueError):
        w8a8_mm(a, w.t(), torch.ones(3, device="cuda"), sb)
    with pytest.raises(NotSupported):
        w8a8_mm(a, w.t(), sa2[:, 0].contiguous(), sb, torch.int8)
    with pytest.raises(ValueError):
        w8a8_mm(a, w.t(), sa2[:, 0].contiguous(), sb, torch.bfloat16, torch.ones(7, device="cuda"))


def test_binding_launches_on_the_current_stream_and_under_capture():
    a, w = ints((16, 2048), 3), ints((4096, 2048), 4)
    sa = torch.rand((16, 1), device="cuda") + 0.5
    sb = torch.rand((4096, 1), device="cuda") + 0.5
    ref = w8a8_mm(a, w.t(), sa, sb)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        out = w8a8_mm(a, w.t(), sa, sb)
    side.synchronize()
    assert torch.equal(out, ref)
    graph = torch.cuda.CUDAGraph()
    before = fast().launches()
    with torch.cuda.graph(graph):
        cap = w8a8_mm(a, w.t(), sa, sb)
    assert fast().launches() == before + 1
    for seed in (5, 6, 7):
        a.copy_(ints((16, 2048), seed))
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(cap, w8a8_mm(a, w.t(), sa, sb))


@pytest.mark.parametrize("m", [1, 16, 300])
def test_quantizer_bindings_equal_ctypes_path(m, ctypes_only):
    say(f"binding quantizers m={m}")
    g = torch.Generator().manual_seed(m)
    x = torch.randn((m, 2048), generator=g).to(torch.bfloat16).cuda()
    r = torch.randn((m, 2048), generator=g).to(torch.bfloat16).cuda()
    w = (1 + 0.1 * torch.randn(2048, generator=g)).to(torch.bfloat16).cuda()
    gu = torch.randn((m, 12288), generator=g).to(torch.bfloat16).cuda()
    qkv = torch.randn((m, 4096), generator=g).to(torch.bfloat16).cuda()
    before = fast().launches()
    got = [fq.add_rmsnorm_quant(x, r, w, 1e-6), fq.add_rmsnorm_quant(x, None, w, 1e-6, False),
           fq.silu_mul_quant(gu, True, True), fq.silu_mul_quant(gu, False, False),
           fq.quant_per_token(qkv[:, :2048]), fq.quant_per_token(x, False)]
    assert fast().launches() == before + len(got)
    ctypes_only()
    ref = [fq.add_rmsnorm_quant(x, r, w, 1e-6), fq.add_rmsnorm_quant(x, None, w, 1e-6, False),
           fq.silu_mul_quant(gu, True, True), fq.silu_mul_quant(gu, False, False),
           fq.quant_per_token(qkv[:, :2048]), fq.quant_per_token(x, False)]
    torch.cuda.synchronize()
    for g_, r_ in zip(got, ref):
        assert len(g_) == len(r_)
        for a_, b_ in zip(g_, r_):
            assert (a_ is None and b_ is None) or torch.equal(a_, b_)


def test_vllm_entry_uses_the_binding_and_records_configs():
    a, w = ints((4, 2048), 8), ints((2048, 2048), 9)
    sa = torch.rand((4, 1), device="cuda") + 0.5
    sb = torch.rand((2048, 1), device="cuda") + 0.5
    calls, before = vllm_patch.CALLS, fast().launches()
    out = vllm_patch.scaled_mm(a, w.t(), sa, sb, torch.bfloat16)
    assert vllm_patch.CALLS == calls + 1 and fast().launches() == before + 1
    assert vllm_patch.CONFIGS[(4, 2048, 2048)] == choose_config(4, 2048, 2048).name
    assert torch.equal(out, kernel.w8a8_mm(a, w.t(), sa, sb, config=choose_config(4, 2048, 2048)))


@pytest.mark.parametrize("m,k,n", [(100, 13824, 5120), (600, 2560, 9728)])
def test_vllm_entry_records_what_is_launched(m, k, n):
    """CONFIGS holds the launched configuration where it is not the plan."""
    a, w = ints((m, k), 8), ints((n, k), 9)
    sa, sb = torch.rand((m, 1), device="cuda"), torch.rand((n, 1), device="cuda")
    vllm_patch.CONFIGS.pop((m, k, n), None)
    out = vllm_patch.scaled_mm(a, w.t(), sa, sb, torch.bfloat16)
    launched = kernel.launch_config(m, n, k)
    assert launched != choose_config(m, n, k)
    assert vllm_patch.CONFIGS[(m, k, n)] == launched.name
    assert torch.equal(out, kernel.w8a8_mm(a, w.t(), sa, sb, config=launched))


def test_outputs_under_a_dispatch_mode():
    """The binding allocates its outputs past the dispatcher, except where a dispatch mode or a
    function transform is active: a mode then sees the allocations, and the outputs are the same."""
    from torch.utils._python_dispatch import TorchDispatchMode

    seen = []

    class Watch(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            seen.append(str(func))
            return func(*args, **(kwargs or {}))

    say("binding outputs under a dispatch mode")
    x = randn((5, 2048), 3)
    q0, s0 = fq.quant_per_token(x)
    before = fast().launches()
    with Watch():
        q, s = fq.quant_per_token(x)
    assert fast().launches() == before + 1
    assert sum("empty" in f for f in seen) == 2
    assert torch.equal(q, q0) and torch.equal(s, s0)
    assert q.is_contiguous() and not q.requires_grad and q.device == x.device


def test_outputs_no_kernel_writes_are_filled_in_deterministic_mode():
    """Under deterministic algorithms torch fills new memory: so it does the binding's outputs, which
    shows where no kernel writes them (the scales of rows without columns)."""
    say("binding outputs under deterministic algorithms")
    x = torch.empty((300, 0), dtype=torch.bfloat16, device="cuda")
    stale = torch.ones((300, 1), device="cuda")
    del stale                               # its block is the next one of this size
    torch.use_deterministic_algorithms(True)
    try:
        assert torch.utils.deterministic.fill_uninitialized_memory
        q, s = fq.quant_per_token(x)
        _, s2 = fq.silu_mul_quant(x, True, True)
    finally:
        torch.use_deterministic_algorithms(False)
    assert q.shape == (300, 0) and bool(s.isnan().all()) and bool(s2.isnan().all())


def test_outputs_under_a_tracer_and_inference_mode():
    """torch.jit.trace records the binding's allocations; in inference mode they are inference
    tensors."""
    say("binding outputs under a tracer and in inference mode")
    x = randn((5, 2048), 3)
    q0, s0 = fq.quant_per_token(x)
    graph = str(torch.jit.trace(lambda t: fq.quant_per_token(t), x, check_trace=False).graph)
    assert graph.count("aten::empty") == 2, graph
    with torch.inference_mode():
        q, s = fq.quant_per_token(x)
    assert q.is_inference() and s.is_inference()
    assert torch.equal(q, q0) and torch.equal(s, s0)


def test_tensors_without_memory_are_refused(ctypes_only):
    """vmap's wrapper has no data pointer and raises; functionalize's and a fake tensor's is 0, which
    every entry refuses before it launches: with the binding and without."""
    from torch._subclasses.fake_tensor import FakeTensorMode

    x = randn((3, 5, 2048), 4)
    rows = x[0]
    a, w, one = ints((5, 2048), 5), ints((2048, 2048), 6), torch.ones(1, device="cuda")

    def refused():
        with pytest.raises(RuntimeError):
            torch.func.vmap(lambda t: fq.quant_per_token(t)[0])(x)
        with pytest.raises(ValueError):
            torch.func.functionalize(lambda t: fq.quant_per_token(t)[0])(rows)
        with pytest.raises(ValueError):
            torch.func.functionalize(lambda t: w8a8_mm(t, w.t(), one, one))(a)
        with FakeTensorMode() as mode, pytest.raises(ValueError):
            fq.silu_mul_quant(mode.from_tensor(rows), True, True)

    say("tensors without memory, binding")
    before = fast().launches()
    refused()
    assert fast().launches() == before
    ctypes_only()
    say("tensors without memory, ctypes")
    refused()
