"""Decode attention with one to eight waves per split (the launch's size picks the count): the
same sequence gives the same bits in batches of every size, and the oracle's result alone."""
import numpy as np
import pytest
import torch

from padra_amd import abi, ops, synth

from attn_tolerance import attn_close, bound_bf16, bound_q8_0

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def gpu():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    abi.lib()
    yield
    torch.cuda.synchronize()


def _rows(fmt, rng, rows):
    """A cache plane as stored: BF16 bits, or codes."""
    if fmt == abi.KV_BF16:
        return synth.bf16_bits(rng.standard_normal((rows, 512)).astype(np.float32)).view(np.int16)
    if fmt == abi.KV_Q8:
        return rng.integers(-127, 128, (rows, 512)).astype(np.int8)
    out = rng.integers(-127, 128, (rows, 544)).astype(np.int8).view(np.uint8)
    out[:, :32] = rng.uniform(.005, .02, (rows, 16)).astype(np.float16).view(np.uint8)
    return out


@pytest.mark.parametrize("fmt", [abi.KV_BF16, abi.KV_Q8, abi.KV_Q8_0])
@pytest.mark.parametrize("local", [False, True])
def test_decode_attention_workgroup_sizes(oracle, fmt, local):
    """17 sequences of 1 to 4096 keys (tile and round edges; local rings that wrap inside a
    tile), run in batches of 17 (one wave a split), 8 (two), 3 (four) and 1 (eight); 32 query
    heads on 4 KV heads, 32 splits (local: 16, so batches of 17, 12, 6 and 1: one, one, four, eight).
    q8_0: a workgroup per split (batches of 17), or per split and KV head."""
    hq, hkv, capacity = 32, 4, 4096
    cap = 1024 if local else capacity
    windows = [1, 31, 32, 33, 64, 255, 256, 257, 1023, 1024, 1025, 1500, 2047, 2049, 4000, 4095,
               4096]
    seqs = len(windows)
    batches = (17, 12, 6, 1) if local else (17, 8, 3, 1)
    print(f"[case] attention workgroups fmt={fmt} local={local}", flush=True)
    rng = np.random.default_rng(31 + fmt + 2 * local)
    q = synth.bf16_bits((rng.standard_normal((seqs, hq, 128)) * 2).astype(np.float32))
    kc, vc = _rows(fmt, rng, seqs * cap), _rows(fmt, rng, seqs * cap)
    sc = rng.uniform(.005, .02, (seqs * cap, hkv, 2)).astype(np.float32)
    states = np.array([[5, n - 1, capacity, 10, n - 1, min(n - 1, 1024), 0, 0] for n in windows],
                      np.int32)
    kd, vd, sd = (torch.from_numpy(a).cuda() for a in (kc, vc, sc))
    qd = torch.from_numpy(q.view(np.int16)).cuda()
    bad = torch.zeros(1, dtype=torch.int32, device="cuda")
    outs = []
    for size in batches:
        out = torch.empty((seqs, hq, 128), dtype=torch.int16, device="cuda")
        for at in range(0, seqs, size):
            some = slice(at, min(seqs, at + size))
            rows = slice(at * cap, some.stop * cap)
            kv = ops.kv_cache(fmt, kd[rows], vd[rows], cap,
                              scales=sd[rows] if fmt == abi.KV_Q8 else None, seq_stride=cap)
            ops.DecodeAttention(qd[some], kv, out[some],
                                ops.positions_decode(torch.from_numpy(states[some]).cuda(),
                                                     maximum=capacity), bad, kv_heads=hkv,
                                local=local)
        torch.cuda.synchronize()
        outs.append(out.cpu().numpy().view(np.uint16))
    assert bad.item() == 0
    for got in outs[1:]:
        assert np.array_equal(got, outs[0])
    for s in (0, 3, 7, 10, 16):
        k, v = kc[s * cap:(s + 1) * cap], vc[s * cap:(s + 1) * cap]
        if fmt == abi.KV_Q8_0:
            want, used, wbad = oracle.decode_attention_q8_0(q[s], k, v, windows[s] - 1, local=local)
            bound = bound_q8_0(q[s], k, v, windows[s] - 1, local, used)
            close, d = attn_close(outs[0][s], want, bound)
            assert not wbad and close.all(), (windows[s], int(d.max()))
            continue
        if fmt == abi.KV_BF16:
            k, v = k.view(np.uint16), v.view(np.uint16)
        else:
            scale = sc[s * cap:(s + 1) * cap]
            k, v = (synth.bf16_bits(c.reshape(cap, hkv, 128).astype(np.float32) *
                                    scale[..., i:i + 1]).reshape(cap, -1)
                    for i, c in enumerate((k, v)))
        want, used, wbad = oracle.decode_attention(q[s], k, v, windows[s] - 1, local=local)
        assert not wbad
        close, d = attn_close(outs[0][s], want,
                              bound_bf16(q[s], k, v, windows[s] - 1, local, used))
        assert close.all(), (windows[s], int(d.max()))


def test_decode_attention_rows_past_4gib():
    """A cache of 131072 rows of 160 KV heads (5.4 GB a plane): row offsets past 2^32 bytes.
    Heads taken out into a cache of four give the same bits."""
    hkv, cap, n = 160, 131072, 131072
    print("[case] attention rows past 4 GiB", flush=True)
    g = torch.Generator(device="cuda").manual_seed(5)
    kc, vc = (torch.randn((cap, hkv * 128), generator=g, device="cuda", dtype=torch.bfloat16)
              for _ in range(2))
    q = torch.randn((1, hkv, 128), generator=g, device="cuda").bfloat16()
    states = torch.tensor([[5, n - 1, cap, 10, n - 1, 1024, 0, 0]], dtype=torch.int32, device="cuda")
    bad = torch.zeros(1, dtype=torch.int32, device="cuda")
    pos = ops.positions_decode(states, maximum=cap)
    out = torch.empty_like(q)
    ops.DecodeAttention(q, ops.kv_cache(abi.KV_BF16, kc, vc, cap), out, pos, bad, kv_heads=hkv)
    for h in (0, 124, 156):
        k4, v4 = (t[:, h * 128:(h + 4) * 128].contiguous() for t in (kc, vc))
        some, q4 = torch.empty((1, 4, 128), dtype=torch.bfloat16, device="cuda"), q[:, h:h + 4].contiguous()
        ops.DecodeAttention(q4, ops.kv_cache(abi.KV_BF16, k4, v4, cap), some, pos, bad, kv_heads=4)
        torch.cuda.synchronize()
        assert torch.equal(some, out[:, h:h + 4])
    assert bad.item() == 0


@pytest.mark.parametrize("fmt", [abi.KV_BF16, abi.KV_Q8, abi.KV_Q8_0])
@pytest.mark.parametrize("seqs", [2, 16, 17, 65])
def test_decode_attention_units(fmt, seqs):
    """Batches on either side of each way the split kernels find their work (2 to 16 sequences
    ranked by the waves, 17 to 64 and 65 to 512 by a kernel before), with windows from one key to
    the capacity, ties, and two sequences that are not admitted: those raise the flag and their
    rows stay, every other row equals the sequence decoded alone."""
    hq, hkv, cap = 8, 4, 2048
    print(f"[case] attention units fmt={fmt} seqs={seqs}", flush=True)
    rng = np.random.default_rng(7 * seqs + fmt)
    positions = rng.integers(0, cap, seqs)
    positions[:2] = cap - 1, 0
    positions[2::3] = 100
    q = torch.from_numpy(synth.bf16_bits(rng.standard_normal((seqs, hq, 128)).astype(np.float32))
                         .view(np.int16)).cuda()
    g = torch.Generator(device="cuda").manual_seed(seqs)
    if fmt == abi.KV_BF16:
        kc, vc = (torch.randn((seqs * cap, 512), generator=g, device="cuda").bfloat16()
                  for _ in range(2))
    else:
        width = 544 if fmt == abi.KV_Q8_0 else 512
        kc, vc = (torch.randint(-127, 128, (seqs * cap, width), generator=g, device="cuda",
                                dtype=torch.int8) for _ in range(2))
        if fmt == abi.KV_Q8_0:
            for t in (kc, vc):
                t[:, :32].view(torch.int16)[:] = 0x2400
    sc = torch.rand((seqs * cap, hkv, 2), generator=g, device="cuda") * .01 + .01
    states = torch.tensor([[5, p, cap, 10, p, min(p, 1024), 0, 0] for p in positions.tolist()],
                          dtype=torch.int32)

    def run(rows, st, out):
        some = slice(rows.start * cap, rows.stop * cap)
        bad = torch.zeros(1, dtype=torch.int32, device="cuda")
        kv = ops.kv_cache(fmt, kc[some], vc[some], cap, seq_stride=cap,
                          scales=sc[some] if fmt == abi.KV_Q8 else None)
        ops.DecodeAttention(q[rows], kv, out, ops.positions_decode(st.cuda(), maximum=cap), bad,
                            kv_heads=hkv)
        torch.cuda.synchronize()
        return bad.item()

    alone = torch.empty((seqs, hq, 128), dtype=torch.int16, device="cuda")
    for i in range(seqs):
        assert run(slice(i, i + 1), states[i:i + 1], alone[i:i + 1]) == 0
    out = torch.full_like(alone, 77)
    assert run(slice(0, seqs), states, out) == 0
    assert torch.equal(out, alone)
    refused = {seqs - 1} if seqs == 2 else {0, seqs - 1}
    for i in refused:
        states[i, 7] = 1  # stopped
    out.fill_(77)
    assert run(slice(0, seqs), states, out) == 1
    for i in range(seqs):
        assert torch.equal(out[i], torch.full_like(out[i], 77) if i in refused else alone[i]), i


@pytest.mark.parametrize("fmt", [abi.KV_BF16, abi.KV_Q8])
@pytest.mark.parametrize("local", [False, True])
def test_decode_attention_infinity_in_the_last_row(oracle, fmt, local):
    """An infinity in the V row of the window's last key comes out as that infinity in its
    dimension (and raises the flag), also where the last tile has keys past the window: those have
    no V row at all.  Batches of 3 and 40 (several waves a split, one)."""
    hq, hkv, capacity = 32, 4, 1024
    windows = [1, 31, 32, 33, 100, 1000, 1023, 1024]
    print(f"[case] attention infinity fmt={fmt} local={local}", flush=True)
    rng = np.random.default_rng(5)
    n = len(windows)
    q = synth.bf16_bits(rng.standard_normal((n, hq, 128)).astype(np.float32))
    kc, vc = _rows(fmt, rng, n * capacity), _rows(fmt, rng, n * capacity)
    sc = rng.uniform(.005, .02, (n * capacity, hkv, 2)).astype(np.float32)
    for i, w in enumerate(windows):
        last = i * capacity + w - 1
        if fmt == abi.KV_BF16:
            vc[last, 7::128] = np.uint16(0xff80).view(np.int16)
        else:
            vc[last] = 0
            vc[last, 7::128] = -100
            sc[last, :, 1] = 1e37
    dense = kc.view(np.uint16), vc.view(np.uint16)
    if fmt == abi.KV_Q8:
        with np.errstate(over="ignore"):
            dense = [synth.bf16_bits(c.reshape(-1, hkv, 128).astype(np.float32) * sc[..., i:i + 1])
                     .reshape(-1, 512) for i, c in enumerate((kc, vc))]
    for size in (3, 40):
        pick = np.arange(size) % n
        rows = np.concatenate([np.arange(i * capacity, (i + 1) * capacity) for i in pick])
        kd, vd, sd, qd = (torch.from_numpy(np.ascontiguousarray(a)).cuda()
                          for a in (kc[rows], vc[rows], sc[rows], q[pick].view(np.int16)))
        states = torch.tensor([[5, windows[i] - 1, capacity, 10, windows[i] - 1,
                                min(windows[i] - 1, 1024), 0, 0] for i in pick], dtype=torch.int32)
        bad = torch.zeros(1, dtype=torch.int32, device="cuda")
        out = torch.empty_like(qd)
        ops.DecodeAttention(qd, ops.kv_cache(fmt, kd, vd, capacity, scales=sd, seq_stride=capacity),
                            out, ops.positions_decode(states.cuda(), maximum=capacity), bad,
                            kv_heads=hkv, local=local)
        torch.cuda.synchronize()
        assert bad.item() == 1
        got = synth.bf16_to_f32(out.cpu().numpy().view(np.uint16))
        for s, i in enumerate(pick):
            k, v = (p[i * capacity:(i + 1) * capacity] for p in dense)
            want, _, wbad = oracle.decode_attention(q[i], k, v, windows[i] - 1, local=local)
            want = synth.bf16_to_f32(want)
            assert wbad and np.isneginf(want[:, 7]).all()
            assert np.isneginf(got[s][:, 7]).all(), (size, windows[i])
            rest = np.arange(128) != 7
            assert np.isfinite(want[:, rest]).all() and np.isfinite(got[s][:, rest]).all()


def _edge_scales(code):
    """The largest scale at which code * scale stays finite in BF16, and the next one (fp32)."""
    limit, s = np.float32(float.fromhex("0x1.ffp127")), np.float32(float.fromhex("0x1.ffp127") / code)
    s = np.nextafter(s, np.float32(0))
    while np.float32(code) * s < limit:
        s = np.nextafter(s, np.float32(np.inf))
    while not np.float32(code) * s < limit:
        s = np.nextafter(s, np.float32(0))
    return s, np.nextafter(s, np.float32(np.inf))


@pytest.mark.parametrize("act", ["bf16", "f32"])
@pytest.mark.parametrize("window", [1, 40, 1024])
def test_decode_attention_q8_values(act, window):
    """kv_q8::Decode's checks of a cache row's scale and codes, K and V, in launches of 1, 16 and 20
    sequences (8 waves a split, one, one held to fewer registers): the largest scale that leaves
    code * scale finite in BF16 passes, the next one, an invalid scale and code -128 raise the flag.
    What passes has the same bits in every batch."""
    print(f"[case] attention q8 values act={act} window={window}", flush=True)
    hq, hkv, cap, seqs = 8, 4, 1024, 20
    g = torch.Generator(device="cuda").manual_seed(window)
    # small queries: a score of the largest values stays finite
    q = (torch.randn((seqs, hq, 128), generator=g, device="cuda") * 2.**-110).bfloat16()
    q = q.float() if act == "f32" else q
    planes = [torch.randint(-127, 128, (seqs * cap, 512), generator=g, device="cuda",
                            dtype=torch.int8) for _ in range(2)]
    sc = torch.rand((seqs * cap, hkv, 2), generator=g, device="cuda") * .01 + .01
    states = torch.tensor([[5, window - 1, cap, 10, window - 1, window - 1, 0, 0]] * seqs,
                          dtype=torch.int32, device="cuda")
    cases = [(0, float(s), True) for s in (np.nan, np.inf, 0., -1.)] + [(-128, .01, True)]
    for code in (127, 100, 1):
        fits, over = _edge_scales(code)
        cases += [(code, float(fits), False), (-code, float(over), True)]

    def run(n):
        bad = torch.zeros(1, dtype=torch.int32, device="cuda")
        out = torch.empty_like(q[:n])
        at = slice((seqs - n) * cap, None)  # the last n sequences
        kv = ops.kv_cache(abi.KV_Q8, planes[0][at], planes[1][at], cap, scales=sc[at],
                          seq_stride=cap)
        ops.DecodeAttention(q[seqs - n:], kv, out, ops.positions_decode(states[:n], maximum=cap),
                            bad, kv_heads=hkv)
        return bad.item(), out

    for plane in (0, 1):
        for code, scale, flagged in cases:
            row = seqs * cap - cap + window - 1  # the last key of the last sequence
            before = planes[plane][row].clone(), sc[row].clone()
            planes[plane][row] = 0
            planes[plane][row, 5::128] = code
            sc[row, :, plane] = scale
            results = [run(n) for n in (1, 16, 20)]
            planes[plane][row], sc[row] = before
            assert [b for b, _ in results] == [int(flagged)] * 3, (plane, code, scale)
            if not flagged:
                assert torch.equal(results[0][1][-1], results[1][1][-1])
                assert torch.equal(results[0][1][-1], results[2][1][-1])
                assert torch.equal(results[1][1], results[2][1][-16:])
                assert results[0][1].isfinite().all()
    bad, out = run(20)
    assert bad == 0 and out.isfinite().all()


def _q8_0_batch(rng, seqs, hq, cap, positions):
    q = synth.bf16_bits((rng.standard_normal((seqs, hq, 128)) * 2).astype(np.float32))
    kc, vc = _rows(abi.KV_Q8_0, rng, seqs * cap), _rows(abi.KV_Q8_0, rng, seqs * cap)
    states = torch.tensor([[5, p, cap, 10, p, min(p, 1024), 0, 0] for p in positions],
                          dtype=torch.int32)
    kd, vd = torch.from_numpy(kc).cuda(), torch.from_numpy(vc).cuda()
    qd = torch.from_numpy(q.view(np.int16)).cuda()

    def run(some, splits, st=states):
        rows = slice(some.start * cap, some.stop * cap)
        out = torch.full((some.stop - some.start, hq, 128), 77, dtype=torch.int16, device="cuda")
        bad = torch.zeros(1, dtype=torch.int32, device="cuda")
        ops.DecodeAttention(qd[some], ops.kv_cache(abi.KV_Q8_0, kd[rows], vd[rows], cap, seq_stride=cap),
                            out, ops.positions_decode(st[some].cuda(), maximum=cap), bad,
                            splits=splits)
        return out, bad.item()

    return q, kc, vc, states, run


@pytest.mark.parametrize("hq", [4, 8, 16, 32])
def test_decode_attention_q8_0_whole_rows(oracle, hq):
    """The q8_0 split of larger batches (a workgroup per split, its waves the KV heads) for every
    number of query heads on a KV head: 9 sequences of 32 splits against the oracle and, bit for
    bit, against each sequence alone (a workgroup per split and KV head)."""
    print(f"[case] attention q8_0 whole rows hq={hq}", flush=True)
    cap, positions = 2048, [0, 31, 32, 127, 128, 129, 1000, 2046, 2047]
    q, kc, vc, _, run = _q8_0_batch(np.random.default_rng(hq), 9, hq, cap, positions)
    out, bad = run(slice(0, 9), 32)
    assert bad == 0
    for i, p in enumerate(positions):
        one, bad = run(slice(i, i + 1), 32)
        assert bad == 0 and torch.equal(one[0], out[i]), p
        k, v = kc[i * cap:(i + 1) * cap], vc[i * cap:(i + 1) * cap]
        want, used, wbad = oracle.decode_attention_q8_0(q[i], k, v, p, local=False)
        close, d = attn_close(out[i].cpu().numpy().view(np.uint16), want,
                              bound_q8_0(q[i], k, v, p, False, used))
        assert not wbad and close.all(), (p, int(d.max()))


@pytest.mark.parametrize("seqs,splits", [(17, 1), (20, 4), (64, 4), (64, 5)])
def test_decode_attention_q8_0_few_splits(seqs, splits):
    """More than 16 sequences of a global cache in few splits: a workgroup per split and KV head up
    to 64 x 4 (1024 of them), per split above.  Each sequence as alone, bit for bit, also beside
    ones that are not admitted."""
    print(f"[case] attention q8_0 few splits seqs={seqs} splits={splits}", flush=True)
    cap, hq = 1024, 8
    rng = np.random.default_rng(seqs + splits)
    positions = rng.integers(0, cap, seqs).tolist()
    positions[:3] = cap - 1, 0, 127
    _, _, _, states, run = _q8_0_batch(rng, seqs, hq, cap, positions)
    alone = torch.cat([run(slice(i, i + 1), splits)[0] for i in range(seqs)])
    out, bad = run(slice(0, seqs), splits)
    assert bad == 0 and torch.equal(out, alone)
    for refused in ([0], [5, seqs - 1]):
        some = states.clone()
        some[refused, 7] = 1  # stopped
        out, bad = run(slice(0, seqs), splits, some)
        want = alone.clone()
        want[refused] = 77
        assert bad == 1 and torch.equal(out, want)


@pytest.mark.parametrize("fmt", [abi.KV_BF16, abi.KV_Q8])
@pytest.mark.parametrize("hq", [4, 32])
def test_decode_attention_fp8_of_f32(fmt, hq):
    """The FP8 output of fp32 activations: out, codes and scales are those of the BF16 ones, and of
    padra_QuantizeFP8 on that row; a zero row has scale 1."""
    print(f"[case] attention fp8 of f32 fmt={fmt} hq={hq}", flush=True)
    seqs, cap = 5, 512
    rng = np.random.default_rng(hq + fmt)
    kc, vc = _rows(fmt, rng, seqs * cap), _rows(fmt, rng, seqs * cap)
    vc[2 * cap:3 * cap] = 0
    sc = torch.full((seqs * cap, 4, 2), 1 / 64, device="cuda")
    kv = ops.kv_cache(fmt, torch.from_numpy(kc).cuda(), torch.from_numpy(vc).cuda(), cap, scales=sc,
                      seq_stride=cap)
    states = torch.tensor([[5, p, cap, 10, p, p, 0, 0] for p in (0, 33, 100, 510, 511)],
                          dtype=torch.int32, device="cuda")
    pos = ops.positions_decode(states, maximum=cap)
    q = torch.from_numpy(rng.standard_normal((seqs, hq, 128)).astype(np.float32)).cuda().bfloat16()
    got = []
    for dtype in (torch.bfloat16, torch.float32):
        out = torch.empty((seqs, hq, 128), dtype=dtype, device="cuda")
        packed = torch.zeros((seqs, hq * 128), dtype=torch.uint8, device="cuda")
        scales = torch.zeros(seqs, device="cuda")
        bad = torch.zeros(1, dtype=torch.int32, device="cuda")
        ops.DecodeAttention(q.to(dtype), kv, out, pos, bad, packed=packed, scales=scales)
        again, more = torch.zeros_like(packed), torch.zeros_like(scales)
        ops.QuantizeFP8(out.view(seqs, -1), again, more, bad)
        assert bad.item() == 0 and torch.equal(packed, again) and torch.equal(scales, more)
        assert scales[2].item() == 1
        got.append((out.float(), packed, scales))
    assert all(torch.equal(a, b) for a, b in zip(*got))
