"""The tensor bindings of the entry points (csrc/fastcall.cpp): what they refuse, and the tensors
and streams they take."""
import pytest
import torch

from padra_amd import abi, ops


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
    with pytest.raises(TypeError, match="too small"):
        calls["padra_DecodeAttentionSplits"](bytes(8), 1, 4, 0, 0)
    with pytest.raises(AttributeError):  # the stream's tensor
        calls["padra_SiluTableBuild"](None, None)
    kv = abi.KVCache(format=abi.KV_Q8_0, k=None, v=None, scales=None, cap=1024, first=0,
                     seq_stride=0)
    lib = abi.lib()
    for args in ((64, 4, 1, -1), (1, 4, 0, 0), (1, 4, 0, 33)):
        assert calls["padra_DecodeAttentionSplits"](kv, *args) == lib.padra_DecodeAttentionSplits(kv, *args)
    assert calls["padra_DecodeAttentionScratch"](2, 1 << 16, 32, 32) == \
        lib.padra_DecodeAttentionScratch(2, 1 << 16, 32, 32) > 1 << 32


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
