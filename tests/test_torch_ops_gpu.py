"""torch.ops.aiter.* on the GPU: the registered ops and a compiled graph give exactly what the
eager entry points give (the reference's bindings are reachable the same way,
aiter/jit/utils/torch_guard.py:292-300)."""

import pytest
import torch

import aiter_amd
from aiter_amd import dtypes

from tests.test_torch_ops_host import decoder_step, expert_layer

pytestmark = pytest.mark.gpu


def same(a, b):
    return torch.equal(a.view(torch.uint8) if a.dtype == dtypes.fp8 else a, b.view(torch.uint8) if b.dtype == dtypes.fp8 else b)


def operands(dev, M=96, N=512, K=1024):
    g = torch.Generator(device=dev).manual_seed(5)
    x = torch.randn(M, K, generator=g, device=dev).bfloat16()
    w = (torch.randn(N, K, generator=g, device=dev) * 0.05).bfloat16()
    wq, ws = aiter_amd.weight_per_128x128_quant(w)
    return x, wq, ws


def test_ops_equal_entry_points():
    dev = torch.device("cuda:0")
    x, wq, ws = operands(dev)
    q, s = aiter_amd.per_group_quant_hip(x)
    q2, s2 = torch.ops.aiter.per_group_quant_hip(x)
    assert same(q, q2) and torch.equal(s, s2)
    y = aiter_amd.gemm_a8w8_blockscale(q, wq, s, ws)
    assert torch.equal(y, torch.ops.aiter.gemm_a8w8_blockscale(q, wq, s, ws))
    out = torch.empty_like(y)
    assert torch.ops.aiter.gemm_a8w8_blockscale_ck(q, wq, s, ws, out, -1, "") is None
    assert torch.equal(y, out)

    # the three spellings of the pre-shuffled call
    wsh = aiter_amd.shuffle_weight(wq, layout=(16, 16))
    qt, st = aiter_amd.per_group_quant_hip(x, transpose_scale=True)
    ref = aiter_amd.gemm_a8w8_blockscale_bpreshuffle(qt, wsh, st, ws)
    assert torch.equal(ref, aiter_amd.gemm_a8w8_blockscale(qt, wsh, st, ws, isBpreshuffled=True))
    out = torch.empty_like(ref)
    assert aiter_amd.gemm_a8w8_blockscale_bpreshuffle_asm(qt, wsh, out, st, ws) is out
    assert torch.equal(ref, out)
    out2 = torch.empty_like(ref)
    assert torch.ops.aiter.gemm_a8w8_blockscale_bpreshuffle(qt, wsh, st, ws, torch.bfloat16, out2) is out2
    assert torch.equal(ref, out2)
    # a zero bias changes nothing
    aiter_amd.gemm_a8w8_blockscale_bpreshuffle_asm(qt, wsh, out, st, ws, bias=torch.zeros(ref.shape[1], device=dev))
    assert torch.equal(ref, out)


def test_compiled_decoder_step_equals_eager():
    dev = torch.device("cuda:0")
    g = torch.Generator(device=dev).manual_seed(6)
    x = torch.randn(64, 1024, generator=g, device=dev).bfloat16()
    res = torch.randn(64, 1024, generator=g, device=dev).bfloat16()
    w = (torch.rand(1024, generator=g, device=dev) + 0.5).bfloat16()
    wq, ws = aiter_amd.weight_per_128x128_quant((torch.randn(512, 1024, generator=g, device=dev) * 0.05).bfloat16())
    wq2, ws2 = aiter_amd.weight_per_128x128_quant((torch.randn(256, 512, generator=g, device=dev) * 0.05).bfloat16())
    wsh = aiter_amd.shuffle_weight(wq2, layout=(16, 16))
    eager = decoder_step(x, res, w, wq, ws, wsh, ws2, torch.empty(64, 256, dtype=torch.bfloat16, device=dev))
    compiled = torch.compile(decoder_step, backend="aot_eager", fullgraph=True)
    for _ in range(2):
        got = compiled(x, res, w, wq, ws, wsh, ws2, torch.zeros(64, 256, dtype=torch.bfloat16, device=dev))
        for a, b in zip(eager, got):
            assert torch.equal(a, b)


def test_compiled_expert_layer_equals_eager():
    dev = torch.device("cuda:0")
    g = torch.Generator(device=dev).manual_seed(7)
    E, dim, inter, tokens = 8, 512, 256, 16
    x = torch.randn(tokens, dim, generator=g, device=dev).bfloat16()
    w1q, w1s = aiter_amd.weight_per_128x128_quant((torch.randn(E * 2 * inter, dim, generator=g, device=dev) * 0.1).bfloat16())
    w2q, w2s = aiter_amd.weight_per_128x128_quant((torch.randn(E * dim, inter, generator=g, device=dev) * 0.1).bfloat16())
    w1 = aiter_amd.shuffle_weight(w1q.view(E, 2 * inter, dim).view(torch.uint8)).view(dtypes.fp8)
    w2 = aiter_amd.shuffle_weight(w2q.view(E, dim, inter).view(torch.uint8)).view(dtypes.fp8)
    gating = torch.randn(tokens, E, generator=g, device=dev).bfloat16()
    args = (x, w1, w2, w1s.view(E, -1), w2s.view(E, -1), gating)
    eager = expert_layer(*args)
    got = torch.compile(expert_layer, backend="aot_eager", fullgraph=True)(*args)
    assert torch.equal(eager, got)


def test_native_bridge_and_ctypes_route_call_alike():
    # plain tensors go through the bridge; a subclass, which it declines, through ctypes: same call, same errors
    from aiter_amd import _ffi

    assert _ffi._bridge is not None, "aiter_amd/_bridge.so is not built"

    class Sub(torch.Tensor):
        pass

    g = torch.Generator().manual_seed(3)
    x = torch.randn(48, 1024, generator=g).bfloat16().to("cuda:0")
    gain = torch.ones(1024, dtype=torch.bfloat16, device="cuda:0")
    results = []
    for cast, status in ((lambda t: t, 0), (lambda t: t.as_subclass(Sub), None)):  # None: declined, nothing called
        outs = []
        for call in (_ffi._bridge.call, _ffi.call):
            y = torch.full((48, 1024), 7, dtype=torch.uint8, device="cuda:0").view(dtypes.fp8)
            s = torch.full((48, 8), -1.0, device="cuda:0")
            got = call("rmsnorm_quant", cast(y), x, s, gain, 1e-6, 128, False, False)
            assert got == status if call is _ffi._bridge.call else got is None
            outs.append((y.view(torch.uint8).clone(), s.clone()))
        if status is None:
            assert (outs[0][0] == 7).all() and (outs[0][1] == -1).all()
            del outs[0]
        results += outs
        with pytest.raises(RuntimeError, match="rmsnorm_quant failed: .*group"):
            _ffi.call("rmsnorm_quant", cast(y), x, s, gain, 1e-6, 48, False, False)
    assert len(results) == 3
    for y8, scale in results[1:]:
        assert torch.equal(results[0][0], y8) and torch.equal(results[0][1], scale)
    assert not (results[0][0] == 7).all() and (results[0][1] > 0).all()
    # on the current stream: the call waits for what that stream does before it, which takes a while
    for cast in (lambda t: t, lambda t: t.as_subclass(Sub)):
        late = torch.zeros_like(x)
        y = torch.empty(48, 1024, dtype=dtypes.fp8, device="cuda:0")
        s = torch.empty(48, 8, device="cuda:0")
        side = torch.cuda.Stream()
        torch.cuda.synchronize()
        with torch.cuda.stream(side):
            torch.cuda._sleep(50_000_000)
            late.copy_(x)
            _ffi.call("rmsnorm_quant", cast(y), late, s, gain, 1e-6, 128, False, False)
        side.synchronize()
        assert torch.equal(y.view(torch.uint8), results[0][0]) and torch.equal(s, results[0][1])
    import ctypes

    with pytest.raises(ctypes.ArgumentError):
        _ffi.call("rmsnorm_quant", y, x, s, gain, 1e-6, "128", False, False)
    with pytest.raises((ctypes.ArgumentError, TypeError)):
        _ffi.call("rmsnorm_quant", y, x, s, gain, 1e-6, 128, False)
    with pytest.raises(TypeError, match="dtype"):
        _ffi.call("rmsnorm_quant", y, x.double(), s, gain, 1e-6, 128, False, False)
