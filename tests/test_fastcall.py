"""The tensor bindings of the entry points (csrc/fastcall.cpp): what they refuse, and the tensors
and streams they take."""
import ctypes

import numpy as np
import pytest
import torch

from padra_amd import abi, ops


class _OnGpu:
    """What a binding reads of a tensor, for calls that are refused before the library's."""
    is_cuda, dtype = True, torch.bfloat16

    def __init__(self, *shape):
        self.shape = shape

    def data_ptr(self):
        return 4096

    def get_device(self):
        return 0

    def numel(self):
        return 1


def test_cpu_tensors_are_refused():
    x = torch.zeros((2, 1024), dtype=torch.bfloat16)
    bad = torch.zeros(1, dtype=torch.int32)
    with pytest.raises(ValueError, match="GPU tensors"):
        ops.ResidualPostNorm(x, x.clone(), x.clone(), x[0].clone(), bad)
    with pytest.raises(ValueError, match="GPU tensors"):
        ops.SwiGLU(x.double(), x, x, x, bad)
    with pytest.raises(ValueError, match="GPU tensors"):
        ops.RotateRows(torch.nn.Parameter(torch.zeros(4, 128)), bad)
    with pytest.raises(ValueError, match="invalid decode attention"):
        ops.DecodeAttention(x.view(2, 8, 128), abi.KVCache(format=9, cap=1), x,
                            ops.positions_base(0), bad)


def test_argument_errors():
    calls = abi.fast()
    with pytest.raises(TypeError, match="padra_SwiGLU takes 8 arguments"):
        calls["padra_SwiGLU"](None)
    with pytest.raises(TypeError):  # a descriptor that is no structure
        calls["padra_DecodeAttentionSplits"](3, 1, 4, 0, 0)
    with pytest.raises(AttributeError):  # the stream's tensor
        calls["padra_SiluTableBuild"](None, None)
    kv = abi.KVCache(format=abi.KV_Q8_0, k=None, v=None, scales=None, cap=1024, first=0,
                     seq_stride=0)
    lib = abi.lib()
    for args in ((64, 4, 1, -1), (1, 4, 0, 0), (1, 4, 0, 33)):
        assert calls["padra_DecodeAttentionSplits"](kv, *args) == lib.padra_DecodeAttentionSplits(kv, *args)
    assert calls["padra_DecodeAttentionScratch"](2, 1 << 16, 32, 32) == \
        lib.padra_DecodeAttentionScratch(2, 1 << 16, 32, 32) > 1 << 32


def test_descriptors_are_their_own_structures():
    """A structure of the other kind, or bytes of the right size, are refused before any call (a
    KVCache is larger than a Positions: its words would be read as a mode and control records)."""
    calls = abi.fast()
    from padra_amd import _fastcall
    kv = abi.KVCache(format=abi.KV_Q8_0, cap=1024)
    size = ctypes.sizeof(kv)
    assert size >= ctypes.sizeof(abi.Positions)
    for wrong in (ops.positions_base(0), bytes(kv), bytearray(kv), np.zeros(size, np.uint8),
                  (abi.KVCache * 2)(), ctypes.pointer(kv)):
        with pytest.raises(TypeError, match="expected KVCache"):
            calls["padra_DecodeAttentionSplits"](wrong, 1, 4, 0, 0)
    x = _OnGpu()
    for wrong in (kv, bytes(size)):
        with pytest.raises(TypeError, match="expected Positions"):
            calls["padra_Embed"](x, x, 8, 8, None, wrong, 1, x, x, 0)
        with pytest.raises(TypeError, match="expected Positions"):
            ops.DecodeAttention(_OnGpu(1, 8, 128), kv, x, wrong, x, scratch=x)

    class Derived(abi.KVCache):
        pass

    derived = Derived(format=abi.KV_Q8_0, cap=1024)
    assert calls["padra_DecodeAttentionSplits"](derived, 1, 4, 0, 0) == 32
    for classes in ((abi.KVCache, abi.Positions), (abi.Positions, kv), (int, abi.KVCache)):
        with pytest.raises(TypeError):
            _fastcall.bind(abi.library_path, abi.PadraError, *classes)
    assert calls["padra_DecodeAttentionSplits"](kv, 1, 4, 0, 0) == 32


def test_entry_points_by_name():
    """Any other attribute is absent, and asking for it loads nothing."""
    calls = ops._Calls()
    assert not hasattr(calls, "__wrapped__") and not calls.__dict__
    assert calls.padra_DecodeAttentionScratch(2, 2, 32, 32) > 0
    assert not hasattr(calls, "padra_Nothing")


@pytest.mark.parametrize("wrong", [1.9, 2.0, "2", b"2", None, np.float32(2), [2]])
def test_numbers_are_what_ctypes_takes(wrong):
    """Counts are integers (anything with __index__), as through ctypes: nothing is truncated or
    parsed.  eps takes a number, not its text."""
    scratch, lib = abi.fast()["padra_DecodeAttentionScratch"], abi.lib()
    for at in range(4):
        args = [2, 2, 32, 32]
        args[at] = wrong
        with pytest.raises(ctypes.ArgumentError):
            lib.padra_DecodeAttentionScratch(*args)
        with pytest.raises(TypeError):
            scratch(*args)
    for right in (2, True, np.int64(2), (1 << 32) + 2, -1):
        args = (2, right, 32, 32)
        assert scratch(*args) == lib.padra_DecodeAttentionScratch(*args)
    if not isinstance(wrong, (float, np.floating)):
        x = _OnGpu()
        with pytest.raises(TypeError):
            abi.fast()["padra_ResidualPostNorm"](x, x, x, x, x, 1, 128, wrong, 128, None, x, 0)


@pytest.mark.gpu
def test_tensors_streams_and_status():
    class Sub(torch.Tensor):
        pass

    g = torch.randn((64, 1024), device="cuda").bfloat16()
    table = torch.empty(65536, dtype=torch.int16, device="cuda")
    ops.SiluTableBuild(table)
    bad = torch.zeros(1, dtype=torch.int32, device="cuda")
    want = torch.empty_like(g)
    ops.SwiGLU(g, g, want, table, bad)
    with pytest.raises(abi.PadraError) as e:
        ops.SwiGLU(g[:1, :4], g, want, table, bad)  # not a multiple of 8
    assert e.value.status == abi.INVALID_ARGUMENT and "padra_SwiGLU" in str(e.value)
    with pytest.raises(TypeError, match="activation dtype"):
        ops.SwiGLU(g.double(), g, want, table, bad)
    for t in (torch.nn.Parameter(g, requires_grad=True), g.as_subclass(Sub), g.view(torch.int16)):
        out = torch.zeros_like(want)
        ops.SwiGLU(t, g, out, table, bad)
        torch.cuda.synchronize()
        assert torch.equal(out, want)
    # a call goes to the current stream: it waits for what that stream already holds
    side = torch.cuda.Stream()
    late, out = torch.zeros_like(g), torch.zeros_like(g)
    torch.cuda.synchronize()
    with torch.cuda.stream(side):
        torch.cuda._sleep(20_000_000)
        late.copy_(g)
        ops.SwiGLU(late, g, out, table, bad)
    side.synchronize()
    assert torch.equal(out, want) and bad.item() == 0
