"""Decode attention at the edges of its splits and passes (64 positions in four
waves, 128 in eight; one split, several, and longer ones past 2048 or 4096
positions) for every head ratio, in its three entry forms, against float64.

Bar: the output is rounded to fp16 (2^-11 of a value) and, with RoPE, q and the
new k row are too, which moves a score by about 2^-11 |q.k| and the softmax
weights by as much: 2e-3 of the largest output."""
import math

import numpy as np
import pytest

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu

D = 128
TOL = 2e-3


@pytest.fixture(scope="module")
def aexq():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from aiimage_amd import aexq as mod
    return mod


@pytest.fixture(scope="module")
def ctx(aexq):
    c = aexq.Context(0)
    yield c
    torch.cuda.synchronize()
    c.close()


def _inputs(hq, hkv, cap, seed):
    g = np.random.default_rng(seed)
    return [g.standard_normal(s).astype(np.float16) for s in
            ((hq, D), (hkv, D), (hkv, D), (hkv, cap, D), (hkv, cap, D))]


def _attend(q, k, v, scale):
    hkv = k.shape[0]
    out = []
    for g, qg in enumerate(q.astype(np.float64).reshape(hkv, -1, D)):
        s = qg @ k[g].astype(np.float64).T * scale
        p = np.exp(s - s.max(-1, keepdims=True))
        out.append((p / p.sum(-1, keepdims=True)) @ v[g].astype(np.float64))
    return np.concatenate(out)


def _rotate(x, cos, sin):
    x = x.astype(np.float64)
    a, b = x[..., :64], x[..., 64:]
    return np.concatenate([a * cos - b * sin, a * sin + b * cos], -1).astype(np.float16)


CASES = [(hq, hkv, length) for hq, hkv in ((4, 4), (4, 2), (16, 4), (8, 1), (32, 8))
         for length in (1, 17, 63, 64, 65, 129, 2047, 2049, 4096, 4097, 8193)]
# where the number of splits turns with the kv heads
CASES += [(hq, hkv, length) for hq, hkv in ((8, 8), (16, 8), (16, 16), (64, 16), (12, 6))
          for length in (2048, 2049, 4096, 4097, 6144, 6145)]


@pytest.mark.parametrize("hq,hkv,length", CASES)
@pytest.mark.parametrize("form", ["plain", "rope", "rope_at"])
def test_attention_split_edges(ctx, hq, hkv, length, form):
    print(f"[gpu-case] attention {form} {hq}/{hkv} length={length}", flush=True)
    # the device-position form sizes its splits for the capacity
    cap = {"plain": length + 3, "rope": length, "rope_at": max(2 * length, 3000)}[form]
    q, k, v, kc, vc = _inputs(hq, hkv, cap, 7 * length + hq)
    dq, dk, dv, dkc, dvc = (torch.as_tensor(a).cuda() for a in (q, k, v, kc, vc))
    out = torch.zeros_like(dq)
    scale = 1.0 / math.sqrt(D)
    g = np.random.default_rng(1)
    angle = g.uniform(0, 6.28, (cap, 64))
    cos, sin = np.cos(angle).astype(np.float32), np.sin(angle).astype(np.float32)
    if form == "plain":
        ctx.attention_decode(dq, dkc, dvc, hq, hkv, D, cap, length, scale, out)
    else:
        p = length - 1
        if form == "rope":
            dc, ds = torch.as_tensor(cos[p]).cuda(), torch.as_tensor(sin[p]).cuda()
            ctx.attention_decode_rope(dq, dk, dv, dkc, dvc, hq, hkv, D, cap, length, dc, ds,
                                      scale, out)
        else:
            dc, ds = torch.as_tensor(cos).cuda(), torch.as_tensor(sin).cuda()
            pos = torch.tensor([p], dtype=torch.int32, device="cuda")
            ctx.attention_decode_rope_at(dq, dk, dv, dkc, dvc, hq, hkv, D, cap, pos, dc, ds,
                                         scale, out)
        q = _rotate(q, cos[p], sin[p])
        kc[:, p], vc[:, p] = _rotate(k, cos[p], sin[p]), v
    torch.cuda.synchronize()
    ref = _attend(q, kc[:, :length], vc[:, :length], scale)
    got = out.cpu().numpy().astype(np.float64)
    assert np.max(np.abs(got - ref)) / np.max(np.abs(ref)) <= TOL
    if form != "plain":   # the appended rows, and no others
        assert np.array_equal(dvc.cpu().numpy(), vc)
        got_k = dkc.cpu().numpy()
        assert np.max(np.abs(got_k.astype(np.float64) - kc)) <= 4e-3
        assert np.array_equal(np.delete(got_k, p, 1), np.delete(kc, p, 1))


@pytest.mark.parametrize("length,low", [(200, slice(0, 100)), (5000, slice(0, 4100)),
                                        (5000, slice(3000, 5000)), (64, slice(16, 48))])
def test_positions_that_score_minus_infinity(ctx, length, low):
    """Whole waves, passes and splits of -inf scores (an overflowing key) weigh
    nothing next to finite ones."""
    print(f"[gpu-case] attention -inf {length} {low}", flush=True)
    hq, hkv = 4, 1
    q, _, _, kc, vc = _inputs(hq, hkv, length, 5)
    q[:] = np.abs(q) + np.float16(0.5)
    kc[:, low] = np.float16(-np.inf)
    out = torch.zeros((hq, D), dtype=torch.float16, device="cuda")
    ctx.attention_decode(torch.as_tensor(q).cuda(), torch.as_tensor(kc).cuda(),
                         torch.as_tensor(vc).cuda(), hq, hkv, D, length, length, 0.05, out)
    torch.cuda.synchronize()
    keep = np.delete(np.arange(length), low)
    ref = _attend(q, kc[:, keep], vc[:, keep], 0.05)
    got = out.cpu().numpy().astype(np.float64)
    assert np.max(np.abs(got - ref)) / np.max(np.abs(ref)) <= TOL


@pytest.mark.parametrize("hq,hkv", [(4, 4), (16, 8), (16, 4), (8, 1)])
@pytest.mark.parametrize("live", [1, 64, 65, 200, 1000, 2048])
def test_device_position_equals_the_launch_for_its_length(ctx, hq, hkv, live):
    """A device-side position far below the capacity runs the passes that a launch
    for that length runs (64 positions a split), to the last bit."""
    print(f"[gpu-case] attention device position {hq}/{hkv} live={live}", flush=True)
    cap = 9000
    q, k, v, kc, vc = (torch.as_tensor(a).cuda() for a in _inputs(hq, hkv, cap, live + hq))
    angle = torch.rand((cap, 64), device="cuda") * 6.28
    cos, sin = torch.cos(angle), torch.sin(angle)
    pos = torch.tensor([live - 1], dtype=torch.int32, device="cuda")
    want, got = torch.zeros_like(q), torch.zeros_like(q)
    ctx.attention_decode_rope(q, k, v, kc, vc, hq, hkv, D, cap, live, cos[live - 1],
                              sin[live - 1], 0.088, want)
    ctx.attention_decode_rope_at(q, k, v, kc, vc, hq, hkv, D, cap, pos, cos, sin, 0.088, got)
    torch.cuda.synchronize()
    assert torch.equal(got, want)


@pytest.mark.parametrize("hq,hkv", [(16, 8), (8, 8)])
def test_a_run_at_the_longest_length_covers_captures_of_shorter_ones(aexq, hq, hkv):
    """The split scratch never has to grow for a shorter length, also where that
    takes more splits, so its first call may be one under capture."""
    print(f"[gpu-case] attention capture after a longer run {hq}/{hkv}", flush=True)
    own = aexq.Context(0)
    cap, short = 8192, 4096
    q, _, _, kc, vc = _inputs(hq, hkv, cap, 3)
    dq, dk, dv = (torch.as_tensor(a).cuda() for a in (q, kc, vc))
    out = torch.zeros_like(dq)
    own.attention_decode(dq, dk, dv, hq, hkv, D, cap, cap, 0.088, out)
    stream = torch.cuda.Stream()
    stream.wait_stream(torch.cuda.current_stream())
    own.set_stream(stream)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=stream, capture_error_mode="thread_local"):
        own.attention_decode(dq, dk, dv, hq, hkv, D, cap, short, 0.088, out)
    for _ in range(3):
        out.zero_()
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        ref = _attend(q, kc[:, :short], vc[:, :short], 0.088)
        assert np.max(np.abs(out.cpu().numpy() - ref)) / np.max(np.abs(ref)) <= TOL
    del graph
    own.close()
