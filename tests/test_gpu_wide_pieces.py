"""SwiGLU and the expert combine + norm where their lane layouts end: element counts around a
wave's 512, waves of ordinary data beside waves with special values, fp32 rows against BF16 rows
of the same values (the fp32 form takes two fours of columns a lane, 256 apart)."""
import numpy as np
import pytest
import torch

from padra_amd import abi, ops, synth

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def gpu():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    abi.lib()
    yield
    torch.cuda.synchronize()


@pytest.mark.parametrize("act", ["bf16", "f32"])
@pytest.mark.parametrize("special", [None, "zero", "tiny", "huge", "overflow", "nan gate", "inf up"])
def test_swiglu_counts_and_special_waves(oracle, act, special):
    rng = np.random.default_rng(3)
    table = torch.empty(65536, dtype=torch.int16, device="cuda")
    ops.SiluTableBuild(table)
    for count in (8, 248, 256, 264, 504, 512, 520, 768, 4096 + 8, 512 * 1024 * 9 + 264):
        gate = (rng.standard_normal(count) * 2).astype(np.float32)
        up = (rng.standard_normal(count) * 2).astype(np.float32)
        for at in {0, count // 2, count - 1} if special else ():
            gate[at] = {"zero": 0., "tiny": 1e-20, "huge": 300., "overflow": 200., "nan gate": np.nan,
                        "inf up": 1.}[special]
            up[at] = {"overflow": 3e38, "inf up": np.inf}.get(special, up[at])
        gb, ub = synth.bf16_bits(gate), synth.bf16_bits(up)
        if special == "nan gate":
            gb[np.isnan(gate)] = 0x7FC0
        want, wbad = oracle.swiglu(gb, ub)
        skipped = ~np.isfinite(gate) | ~np.isfinite(up)  # the gate stays in its place
        want[skipped] = gb[skipped]
        if act == "bf16":
            g, u = (torch.from_numpy(t.view(np.int16)).cuda() for t in (gb, ub))
        else:
            g, u = (torch.from_numpy(synth.bf16_to_f32(t)).cuda() for t in (gb, ub))
        out = torch.full((count + 512,), 7, dtype=g.dtype, device="cuda")
        bad = torch.zeros(1, dtype=torch.int32, device="cuda")
        ops.SwiGLU(g, u, out, table, bad)
        torch.cuda.synchronize()
        got = out[:count].cpu().numpy()
        got = got.view(np.uint16) if act == "bf16" else synth.bf16_bits(got)
        if special == "nan gate":  # (with the payload its type's path gives)
            assert np.isnan(synth.bf16_to_f32(got[np.isnan(gate)])).all()
            got[np.isnan(gate)] = 0x7FC0
        assert np.array_equal(got, want), count
        assert bool(bad.item()) == wbad
        assert bool((out[count:] == 7).all())


def test_swiglu_f32_inexact_gate():
    """An fp32 gate that is no BF16 value: the flag, the gate rounded in its place, the wave's
    other elements as ever."""
    g = torch.randn(1024, device="cuda").bfloat16().float()
    g[700] = 1.0009765625 + 2**-20
    up = torch.randn(1024, device="cuda").bfloat16().float()
    table = torch.empty(65536, dtype=torch.int16, device="cuda")
    ops.SiluTableBuild(table)
    bad = torch.zeros(1, dtype=torch.int32, device="cuda")
    out, want = torch.empty_like(g), torch.empty(1024, dtype=torch.bfloat16, device="cuda")
    ops.SwiGLU(g, up, out, table, bad)
    assert bad.item() == 1
    bad.zero_()
    ops.SwiGLU(g.bfloat16(), up.bfloat16(), want, table, bad)
    assert bad.item() == 0
    want = want.float()
    want[700] = g[700].bfloat16().float()
    assert torch.equal(out, want)


@pytest.mark.parametrize("act", ["bf16", "f32"])
def test_swiglu_nan_in_the_table(act):
    """A product that is NaN raises the flag also where operands and gate are ordinary: with a
    table that holds a NaN (one never built, or overwritten)."""
    table = torch.empty(65536, dtype=torch.int16, device="cuda")
    ops.SiluTableBuild(table)
    table[0x3F80] = 0x7FC0  # silu(1)
    dtype = torch.bfloat16 if act == "bf16" else torch.float32
    g = torch.full((1024,), 2., device="cuda", dtype=dtype)
    up, out = torch.ones_like(g), torch.empty_like(g)
    for at, flag in ((None, 0), (0, 1), (511, 1), (700, 1)):
        g.fill_(2.)
        if at is not None:
            g[at] = 1.
        bad = torch.zeros(1, dtype=torch.int32, device="cuda")
        ops.SwiGLU(g, up, out, table, bad)
        assert bad.item() == flag, at
        assert out.isnan().sum().item() == flag


@pytest.mark.parametrize("hidden", [1024, 1152, 2048, 2304, 4096, 4608])
@pytest.mark.parametrize("rows,fp8", [(37, False), (37, True), (2048, True)])
def test_combine_norm_f32_equals_bf16(hidden, rows, fp8):
    g = torch.Generator(device="cuda").manual_seed(hidden)
    x = torch.randn((rows, hidden), generator=g, device="cuda").bfloat16()
    down = torch.randn((rows, 8, hidden), generator=g, device="cuda").bfloat16()
    x[5] = 0
    down[5] = 0
    down[9, 3, hidden - 1] = float("inf")
    weights = torch.rand((rows, 8), generator=g, device="cuda")
    gamma = torch.randn(hidden, generator=g, device="cuda").bfloat16()
    got = []
    for dtype in (torch.bfloat16, torch.float32):
        a = x.to(dtype, copy=True)
        y = torch.zeros_like(a)
        packed = torch.zeros((rows, hidden), dtype=torch.uint8, device="cuda") if fp8 else None
        scales = torch.zeros(rows, device="cuda") if fp8 else None
        stats = torch.zeros(2, device="cuda")
        bad = torch.zeros(1, dtype=torch.int32, device="cuda")
        ops.CombineNorm(a, down.to(dtype), weights, y, gamma, bad, packed=packed, scales=scales,
                        statistics=stats)
        torch.cuda.synchronize()
        assert bad.item() == 1
        got.append([a.float(), y.float(), stats] + ([packed, scales] if fp8 else []))
    keep = torch.arange(rows, device="cuda") != 9  # row 9 holds infinities and NaNs
    for one, two in zip(*got):
        if one.shape[0] == rows:
            assert torch.equal(one[keep], two[keep])
            assert torch.allclose(one[9].float(), two[9].float(), equal_nan=True)
        else:
            assert torch.equal(one, two)


@pytest.mark.parametrize("hidden", [1024, 1152, 2048, 2304, 4096, 4608])
@pytest.mark.parametrize("act", [torch.bfloat16, torch.float32])
def test_combine_norm_finite_rows_raise_no_flag(hidden, act):
    """Every column of a row finite, up to the largest whose sums stay so: the flag stays down.  One
    value that is not, in any lane of any chunk, raises it."""
    rows = 3
    g = torch.Generator(device="cuda").manual_seed(hidden)
    weights = torch.full((rows, 8), .125, device="cuda")
    gamma = torch.ones(hidden, device="cuda", dtype=torch.bfloat16)
    x = torch.randn((rows, hidden), generator=g, device="cuda").to(torch.bfloat16).to(act)
    down = torch.randn((rows, 8, hidden), generator=g, device="cuda").to(torch.bfloat16).to(act)
    x[1] = 2.**55  # (the sum of its squares stays finite)
    for at in [None, *range(0, hidden, 4)]:
        a, d = x.clone(), down.clone()
        if at is not None:
            d[2, at % 8, at + at // 4 % 4] = float("inf") if at % 8 else float("nan")
        y, bad = torch.empty_like(a), torch.zeros(1, dtype=torch.int32, device="cuda")
        ops.CombineNorm(a, d, weights, y, gamma, bad)
        assert bad.item() == (at is not None), at
