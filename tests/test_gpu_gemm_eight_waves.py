"""The eight-wave tiles of the LDS-direct GEMM against the float64 oracle: one K
step to more than the ring holds, tails of one and two steps, ragged rows and
columns, pairs, residual, bias and head-packed outputs, every scale format; and
the rule that chooses them.

Bars as in the other GEMM tests: 1e-5 of the largest value for plain fp32
outputs against the weights the plan multiplies, 1e-3 for fp16."""
import sys

import numpy as np
import pytest
from conftest import for_plan, q4_reference

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu

TOL, TOL32 = 1e-3, 1e-5


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


def dev(a):
    return torch.as_tensor(np.ascontiguousarray(a)).cuda()


def normwise(y, r):
    return float(np.max(np.abs(np.asarray(y, np.float64) - r)) / max(np.max(np.abs(r)), 1e-30))


def _weight(ctx, aexq, orc, bits, group, f16, n, k, seed):
    from aiimage_amd import synth
    sdt = np.float16 if f16 else np.float32
    if bits == 8:
        words, scales, _ = synth.q8_weights(n, k, seed, scale_dtype=sdt)
        w = ctx.weight(aexq.QuantizedTensor(n * k, k, words, scales, bits=8), n, k)
        return w, orc.dequant_q8(words, scales, n, k,
                                 scale_dtype=orc.SCALE_F16 if f16 else orc.SCALE_F32)
    words, scales, _ = synth.q4_weights(n, k, seed, group=group, code=1, scale_dtype=sdt)
    w = ctx.weight(aexq.QuantizedTensor(n * k, group, words, scales, bits=4, nibble_code=1), n, k)
    return w, q4_reference(orc, words, scales, n, k, group, 1, f16)


# (bits, group, fp16 scales, m, n, k, epilogue, output columns of a tile)
CASES = [(8, 0, True, 1000, 1601, k, "plain", 128) for k in (64, 128, 192, 256, 320, 1088)]
CASES += [(8, 0, False, 513, 2600, 320, "plain", 128), (8, 0, True, 400, 3001, 256, "swiglu", 64),
          (8, 0, False, 1025, 2047, 192, "residual", 128), (8, 0, True, 700, 2048, 128, "bias", 128),
          (8, 0, True, 390, 3072, 128, "heads", 128)]
CASES += [(4, g, f, 900, 1700, k, "plain", 128) for g, f, k in
          ((32, True, 128), (32, False, 256), (16, True, 384), (16, False, 512), (32, True, 640))]
CASES += [(4, 16, True, 520, 1300, 256, "swiglu", 64), (4, 32, False, 520, 1300, 384, "swiglu", 64),
          (4, 16, False, 1000, 1666, 256, "residual", 128)]


@pytest.mark.parametrize("bits,group,f16,m,n,k,epi,cols", CASES)
def test_eight_wave_tiles(ctx, aexq, orc, bits, group, f16, m, n, k, epi, cols):
    print(f"[gpu-case] eight waves q{bits} g={group} f16={f16} m={m} n={n} k={k} {epi}", flush=True)
    sys.stdout.flush()
    from aiimage_amd import synth
    w, wf = _weight(ctx, aexq, orc, bits, group, f16, n, k, m + k)
    x16 = synth.activations(m, k, 3)
    y32 = epi in ("plain", "bias")
    dt = torch.float32 if y32 else torch.float16
    lay = aexq.LAYOUT_HEAD_PACKED if epi == "heads" else aexq.LAYOUT_PACK4_LINEAR
    hd = 64 if epi == "heads" else 0
    y = aexq.new_activation(m, n, dt, lay, head_dim=hd)
    y.fill_(7.0)
    xd, yd = aexq.describe(dev(x16), m, k), aexq.describe(y, m, n, lay, head_dim=hd)
    kw = {}
    stride = -(-n // 4) * 4
    if epi == "swiglu":
        wu, uf = _weight(ctx, aexq, orc, bits, group, f16, n, k, m + k + 1)
        kw["up"] = wu
    elif epi == "residual":
        rbuf = np.zeros((m, stride), np.float16)
        rbuf[:, :n] = synth.activations(m, n, 9)
        kw["residual"] = aexq.describe(dev(rbuf), m, n, lay)
    elif epi == "bias":
        bias = synth.activations(1, n, 5).astype(np.float32).reshape(-1)
        kw.update(alpha=0.75, beta=1.25, c=dev(bias), broadcast_c=4)
    plan = dict(t.split("=") for t in ctx.plan_check(w, xd, yd, **kw).split())
    assert plan["kernel"] == "qgemm" and plan["waves"] == "8" and plan["splitk"] == "1", plan
    assert int(plan["tiles"]) == -(-(n if epi == "heads" else stride) // cols), plan
    ctx.linear(w, xd, yd, **kw)
    torch.cuda.synchronize()
    text = f"fp16_dequant={plan['fp16_dequant']}"
    # the last rows and every 37th: the oracle is the slow part
    rows = sorted(set(range(0, m, 37)) | set(range(m - 70, m)))
    xr = x16[rows].astype(np.float32)
    ref = orc.gemm_gpu_semantics(xr, for_plan(wf, text))
    if epi == "heads":
        got = orc.head_unpack(y.cpu().numpy().astype(np.float32), m, n // hd, hd)[rows]
    else:
        full = y.cpu().numpy().astype(np.float64).reshape(m, stride)
        assert np.all(full[:, n:] == 0) and np.all(np.isfinite(full))
        got = full[rows][:, :n]
    if epi == "swiglu":
        u = orc.gemm_gpu_semantics(xr, for_plan(uf, text))
        ref = np.stack([orc.swiglu(ref[r].astype(np.float32), u[r].astype(np.float32))
                        for r in range(len(rows))])
    elif epi == "residual":
        ref = ref + rbuf[rows][:, :n].astype(np.float64)
    elif epi == "bias":
        ref = 0.75 * (1.25 * bias[None].astype(np.float64) + ref)
    assert normwise(got, ref) <= (TOL32 if y32 else TOL), plan


@pytest.mark.parametrize("fmt,m,n,k,pair,waves", [
    # 96 tiles and one below; grids padded to eight weight tiles past one per CU
    ((8, 0), 1000, 1536, 1024, False, 8), ((8, 0), 1000, 1408, 1088, False, 4),
    ((4, 32), 1334, 2304, 512, False, 4), ((4, 32), 1334, 2048, 512, False, 8),
    # one and two tiles per CU, weights and pairs
    ((8, 0), 2048, 4096, 1024, False, 8), ((8, 0), 2100, 4096, 1024, False, 4),
    ((4, 16), 2048, 2048, 1024, False, 8), ((4, 16), 2048, 2176, 1024, False, 4),
    ((8, 0), 2048, 1024, 1024, True, 8), ((8, 0), 2048, 1088, 1024, True, 4),
    # long rows on idle CUs; a step or two of one row tile
    ((8, 0), 512, 4096, 2048, False, 8), ((8, 0), 512, 4096, 2112, False, 4),
    ((4, 32), 512, 4096, 2048, False, 8), ((4, 32), 512, 4096, 2176, False, 4),
    ((8, 0), 1024, 4096, 8192, False, 8), ((4, 32), 90, 13312, 256, False, 4),
])
def test_where_eight_waves_are_taken(ctx, aexq, monkeypatch, no_wave, fmt, m, n, k, pair, waves):
    """Both sides of the lines of the rule (planned only)."""
    print(f"[gpu-case] eight waves rule {fmt} m={m} n={n} k={k} pair={pair}", flush=True)
    bits, group = fmt
    w = ctx.weight(aexq.QuantizedTensor(n * k, group or k, np.zeros(n * k * bits // 32, np.uint32),
                                        np.ones(n * k // group if group else n, np.float16),
                                        bits=bits), n, k)
    x = torch.zeros(m * k, dtype=torch.float16, device="cuda")
    lay = aexq.LAYOUT_PACK4_LINEAR
    y = aexq.new_activation(m, n, torch.float16, lay)
    plan = ctx.plan_check(w, aexq.describe(x, m, k), aexq.describe(y, m, n, lay),
                          **({"up": w} if pair else {}))
    assert plan.split()[0] == "kernel=qgemm" and f" waves={waves} " in plan, plan
