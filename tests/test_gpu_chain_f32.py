"""The chain entry point on fp32 activations in its larger launches (one kernel: norm rows, then
the four-lanes-per-head Q/K waves) against its two halves called one after the other."""
import pytest
import torch

from padra_amd import abi, ops

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def gpu():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    abi.lib()
    yield
    torch.cuda.synchronize()


@pytest.mark.parametrize("fmt", [None, abi.KV_BF16, abi.KV_Q8, abi.KV_Q8_0, abi.KV_Q8_0_NOROT])
@pytest.mark.parametrize("tokens,hidden,heads,tree", [(321, 2048, 16, abi.TREE_128),
                                                      (385, 2304, 32, abi.TREE_256),
                                                      (1201, 2304, 32, abi.TREE_128),
                                                      (2048, 2048, 4, abi.TREE_256),
                                                      (1793, 2048, 16, abi.TREE_128)])
def test_chain_f32_equals_its_halves(fmt, tokens, hidden, heads, tree):
    """Just past the per-head sizes (320 tokens with a quantized cache, 384 without), odd chunk
    sizes, a local ring narrower than the chunk, a NaN row: every output and the flag equal."""
    print(f"[case] chain f32 fmt={fmt} tokens={tokens} hidden={hidden}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(tokens)

    def normal(*shape):
        return torch.randn(shape, generator=g, device="cuda").bfloat16().float()

    x, r = normal(tokens, hidden), normal(tokens, hidden)
    q, k, v = normal(tokens, heads, 128), normal(tokens, 4, 128), normal(tokens, 4, 128)
    gamma, qn, kn = (normal(n).bfloat16() for n in (hidden, 128, 128))
    table = ops.RopeTable(8192, 128).cuda()
    cap = 1024
    state = torch.tensor([700, 0, tokens, 8192, 700, 1, 1, 1], dtype=torch.int32, device="cuda")
    width = {None: 0, abi.KV_BF16: 1024, abi.KV_Q8: 512}.get(fmt, 544)
    results = []
    for fused in (True, False):
        for poison in (False, True):
            a = [t.clone() for t in (x, r, q, k, v)]
            if poison:
                a[0][tokens // 2, 5] = float("nan")
            y = torch.zeros_like(x)
            stats = torch.zeros((tokens, 2), device="cuda")
            kc, vc = (torch.zeros((cap, max(1, width)), dtype=torch.uint8, device="cuda")
                      for _ in range(2))
            sc = torch.zeros((cap, 4, 2), device="cuda")
            kv = None if fmt is None else ops.kv_cache(fmt, kc, vc, cap, scales=sc,
                                                       first=max(0, tokens - cap))
            pos = ops.positions_prefill(state, maximum=8192)
            bad = torch.zeros(1, dtype=torch.int32, device="cuda")
            if fused:
                ops.ResidualNormQKRopeStore(a[0], a[1], y, gamma, a[2], a[3], a[4], qn, kn, table,
                                            pos, kv, bad, tree=tree, statistics=stats)
            else:
                ops.ResidualPostNorm(a[0], a[1], y, gamma, bad, tree=tree, statistics=stats)
                ops.QKNormRopeStore(a[2], a[3], qn, kn, table, pos, bad, v=a[4], kv=kv)
            torch.cuda.synchronize()
            assert bad.item() == int(poison)
            results.append([t.contiguous().view(torch.uint8) for t in (*a, y, stats, kc, vc, sc)])
    for i in range(2):
        for one, two in zip(results[i], results[i + 2]):
            assert torch.equal(one, two)
