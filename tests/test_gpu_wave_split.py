"""The wave-split matmul (aexq_qmmk.hpp) against the float64 oracle at the sizes
where it can go wrong: both sides of its row tiles, one to many K slices, odd
and ragged N and K (half chunks, unaligned scale rows), every scale format,
RMSNorm-in within and past its LDS ring, copies of a stack, and scales of a
neighbouring row that must not leak through a ragged K.

Bars: fp32 outputs of plain products 1e-5 of the largest value (at most 4096
fp32 additions of exact products: 4096 * 2^-24 is 2.4e-4 of the sum of
magnitudes in the worst case and about 1e-6 for random signs); 1e-3 for fp16
outputs and normalised inputs (2^-11 per rounding), as in the other tests."""
import sys

import numpy as np
import pytest
from conftest import for_plan, plan_kernel, q4_reference

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu

TOL, TOL32, EPS = 1e-3, 1e-5, 1e-6


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


# name: (bits, group, fp16 scales, nibble code)
FORMATS = {"q8h": (8, 0, True, 0), "q8s": (8, 0, False, 0), "q4h": (4, 32, True, 1),
           "q4s": (4, 32, False, 0), "q4g16h": (4, 16, True, 0), "q4g16s": (4, 16, False, 0)}


def _weight(ctx, aexq, orc, fmt, n, k, seed, poke=None):
    from aiimage_amd import synth
    bits, group, f16, code = FORMATS[fmt]
    sdt = np.float16 if f16 else np.float32
    if bits == 8:
        words, scales, _ = synth.q8_weights(n, k, seed, scale_dtype=sdt)
    else:
        words, scales, _ = synth.q4_weights(n, k, seed, group=group, code=code, scale_dtype=sdt)
    if poke is not None:
        scales = scales.copy()
        scales[poke] = np.inf
    w = ctx.weight(aexq.QuantizedTensor(n * k, group or k, words, scales, bits=bits,
                                        nibble_code=code), n, k)
    if bits == 8:
        return w, orc.dequant_q8(words, scales, n, k,
                                 scale_dtype=orc.SCALE_F16 if f16 else orc.SCALE_F32)
    return w, q4_reference(orc, words, scales, n, k, group, code, f16)


# (fmt, m, n, k, epilogue, expected kernel)
CASES = [
    # row tiles: 16, 32 and 64 rows and one past; one 128-wide slice and many
    ("q4h", 2, 16, 128, "plain", "wave"), ("q8h", 16, 33, 256, "plain", "wave"),
    ("q4g16s", 17, 1000, 1024, "plain", "wave"), ("q8s", 32, 5137, 512, "plain", "wave"),
    ("q4h", 32, 11000, 1024, "plain", "wave"), ("q4s", 16, 5200, 1152, "plain", "wave"),
    ("q8h", 33, 1001, 1024, "plain", "wave"), ("q4h", 64, 1024, 3584, "plain", "wave"),
    ("q4g16h", 65, 515, 512, "plain", "wave"), ("q4s", 97, 3000, 640, "plain", "wave"),
    ("q8s", 130, 4100, 1024, "plain", "wave"), ("q4g16s", 257, 4096, 1024, "plain", "wave"),
    ("q4h", 500, 1024, 2048, "residual", "wave"), ("q8h", 300, 3072, 1024, "residual", "wave"),
    # SwiGLU pairs; RMSNorm-in: one slice a wave, whole rows in the ring, past it
    ("q4h", 5, 3584, 1024, "swiglu", "wave"), ("q8h", 31, 3000, 2048, "swiglu", "wave"),
    ("q4g16h", 32, 4090, 1024, "swiglu", "wave"), ("q8s", 16, 130, 4096, "rms", "wave"),
    ("q4h", 32, 5200, 1024, "swiglu", "wave"),
    ("q4g16s", 3, 257, 3072, "rms", "wave"), ("q4s", 30, 640, 2048, "rms", "wave"),
    ("q4h", 29, 5201, 2048, "rms", "wave"), ("q4h", 16, 520, 1024, "rms-nogamma", "wave"),
    ("q4s", 64, 200, 1024, "rms", "wave"), ("q8h", 100, 1024, 512, "swiglu", "wave"),
    # K of 16-code halves of a chunk, of odd scale rows, of less than a slice
    ("q8s", 77, 1001, 1008, "plain", "wave"), ("q8h", 9, 50, 16, "plain", "wave"),
    ("q4g16h", 1, 97, 1040, "plain", "wave"), ("q4g16h", 200, 333, 336, "residual", "wave"),
    ("q4g16s", 5, 101, 48, "plain", "wave"), ("q4h", 19, 345, 1120, "plain", "wave"),
    ("q4h", 300, 900, 160, "plain", "wave"), ("q4s", 12, 64, 32, "plain", "wave"),
    ("q4g16s", 40, 70, 2000, "rms", "wave"), ("q4g16h", 700, 640, 208, "rms", "wave"),
    ("q8h", 33, 129, 4080, "rms", "wave"),
]


@pytest.mark.parametrize("fmt,m,n,k,epi,kernel", CASES)
def test_wave_split_against_oracle(ctx, aexq, orc, fmt, m, n, k, epi, kernel):
    print(f"[gpu-case] wave split {fmt} m={m} n={n} k={k} {epi}", flush=True)
    sys.stdout.flush()
    from aiimage_amd import synth
    w, wf = _weight(ctx, aexq, orc, fmt, n, k, n + k + m)
    x16 = synth.activations(m, k, m + 7)
    y32 = epi == "plain"
    dt = torch.float32 if y32 else torch.float16
    lay = aexq.LAYOUT_PACK4_LINEAR
    stride = aexq.storage_elements(lay, m, n)
    xd = aexq.describe(dev(x16), m, k)
    kw, xr = {}, x16.astype(np.float32)
    if epi in ("rms", "rms-nogamma", "swiglu"):
        gamma = synth.rms_gamma(k, 5) if epi != "rms-nogamma" else None
        kw.update(rmsnorm=True, rms_gamma=dev(gamma) if gamma is not None else None, rms_eps=EPS)
        xr = orc.rmsnorm(xr, EPS, gamma).astype(np.float16).astype(np.float32)
    if epi == "swiglu":
        wu, uf = _weight(ctx, aexq, orc, fmt, n, k, n + k + m + 1)
        kw["up"] = wu
    if epi == "residual":
        rbuf = np.zeros((m, stride), np.float16)
        rbuf[:, :n] = synth.activations(m, n, 9)
        kw["residual"] = aexq.describe(dev(rbuf), m, n, lay)
    ys = []
    for _ in range(2):
        y = aexq.new_activation(m, n, dt, lay)
        y.fill_(7.0)   # the padding lanes must be written
        yd = aexq.describe(y, m, n, lay)
        plan = ctx.plan_check(w, xd, yd, **kw)
        assert plan_kernel(plan) == kernel, plan
        ctx.linear(w, xd, yd, **kw)
        ys.append(y)
    torch.cuda.synchronize()
    assert torch.equal(ys[0], ys[1])   # the waves' sums meet in a fixed order
    got = ys[0].cpu().numpy().astype(np.float64).reshape(m, stride)
    assert np.all(got[:, n:] == 0)
    ref = orc.gemm_gpu_semantics(xr, for_plan(wf, plan))
    if epi == "swiglu":
        u = orc.gemm_gpu_semantics(xr, for_plan(uf, plan))
        ref = np.stack([orc.swiglu(ref[r].astype(np.float32), u[r].astype(np.float32))
                        for r in range(m)])
    if epi == "residual":
        ref = ref + rbuf[:, :n].astype(np.float64)
    assert normwise(got[:, :n], ref) <= (TOL32 if y32 else TOL), plan


@pytest.mark.parametrize("fmt,m,k", [("q4h", 16, 1024), ("q8h", 64, 1024), ("q4g16h", 20, 1040)])
def test_wave_split_stack_equals_single(ctx, aexq, orc, fmt, m, k):
    """Every copy of a replicated weight gives the single launch's bits (both
    take the wave-split kernel), with activations of its own."""
    print(f"[gpu-case] wave split stack {fmt} m={m} k={k}", flush=True)
    from aiimage_amd import synth
    n, copies = 200, 3
    w, _ = _weight(ctx, aexq, orc, fmt, n, k, 3)
    st = w.replicate(copies)
    lay = aexq.LAYOUT_PACK4_LINEAR
    xs = dev(np.concatenate([synth.activations(m, k, 20 + c) for c in range(copies)]))
    ys = aexq.new_activation(m, n, torch.float32, lay, batch=copies)
    xd = aexq.describe(xs, m, k, batch=copies, batch_stride=m * k)
    yd = aexq.describe(ys, m, n, lay, batch=copies, batch_stride=m * n)
    assert plan_kernel(ctx.plan_check(st, xd, yd)) == "wave"
    ctx.linear(st, xd, yd)
    for c in range(copies):
        y = aexq.new_activation(m, n, torch.float32, lay)
        ctx.linear(w, aexq.describe(xs[c * m:(c + 1) * m].contiguous(), m, k),
                   aexq.describe(y, m, n, lay))
        torch.cuda.synchronize()
        assert torch.equal(ys[c * m * n:(c + 1) * m * n], y), c


@pytest.mark.parametrize("fmt", ["q4g16h", "q4g16s", "q4h", "q4s", "q8s"])
def test_ragged_k_keeps_to_its_row(ctx, aexq, orc, fmt):
    """An infinite scale in one row reaches that row's outputs only: the last
    slice of a ragged row reads into the next row's codes and scales."""
    print(f"[gpu-case] wave split ragged inf {fmt}", flush=True)
    from aiimage_amd import synth
    bits, group, _, _ = FORMATS[fmt]
    m, n, k = 11, 40, 1056 + (16 if group == 16 else 0)
    bad = 21   # its first scale follows the last one of row 20
    w, wf = _weight(ctx, aexq, orc, fmt, n, k, 8, poke=bad * (k // group) if group else bad)
    x16 = synth.activations(m, k, 4)
    y = aexq.new_activation(m, n, torch.float32, aexq.LAYOUT_LINEAR)
    xd, yd = aexq.describe(dev(x16), m, k), aexq.describe(y, m, n)
    plan = ctx.plan_check(w, xd, yd)
    assert plan.startswith("kernel=wave "), plan
    ctx.linear(w, xd, yd)
    torch.cuda.synchronize()
    got = y.cpu().numpy().reshape(m, n)
    rest = [r for r in range(n) if r != bad]
    assert not np.any(np.isfinite(got[:, bad]))
    wf = wf.exact if hasattr(wf, "exact") else wf
    ref = orc.gemm_gpu_semantics(x16.astype(np.float32), np.ascontiguousarray(wf[rest]))
    assert normwise(got[:, rest], ref) <= TOL32


@pytest.mark.parametrize("fmt,m,k", [("q4g16h", 5, 1024), ("q4g16s", 20, 1024),
                                     ("q4g16h", 20, 1040), ("q4h", 5, 1024), ("q8h", 5, 1024)])
def test_infinite_activation_keeps_its_sign(ctx, aexq, orc, fmt, m, k):
    """An infinite activation gives +-inf by the sign of its code (NaN where the
    code is 0) in its own row, in exact products as in float64, and leaves the
    other rows alone."""
    print(f"[gpu-case] wave split infinite x {fmt} m={m} k={k}", flush=True)
    from aiimage_amd import synth
    n, row = 200, 3
    w, wf = _weight(ctx, aexq, orc, fmt, n, k, 12)
    x16 = synth.activations(m, k, 4)
    x16[row, k - 9] = np.inf
    y = aexq.new_activation(m, n, torch.float32, aexq.LAYOUT_LINEAR)
    xd, yd = aexq.describe(dev(x16), m, k), aexq.describe(y, m, n)
    plan = ctx.plan_check(w, xd, yd)
    assert plan.startswith("kernel=wave "), plan
    ctx.linear(w, xd, yd)
    torch.cuda.synchronize()
    got = y.cpu().numpy().reshape(m, n)
    wx = np.asarray(for_plan(wf, plan), np.float64)[:, k - 9]
    with np.errstate(invalid="ignore"):
        np.testing.assert_array_equal(got[row], np.inf * wx)
    rest = [r for r in range(m) if r != row]
    ref = orc.gemm_gpu_semantics(np.ascontiguousarray(x16[rest]).astype(np.float32),
                                 for_plan(wf, plan))
    assert normwise(got[rest], ref) <= TOL32


def test_rows_too_far_apart_for_its_offsets(ctx, aexq, orc):
    """Row strides whose tile passes 32-bit offsets keep the kernels they had."""
    print("[gpu-case] wave split row strides", flush=True)
    m, n, k = 2, 64, 1024
    w, _ = _weight(ctx, aexq, orc, "q8h", n, k, 2)
    x = torch.zeros(m * k, dtype=torch.float16, device="cuda")
    y = aexq.new_activation(m, n, torch.float16, aexq.LAYOUT_LINEAR)

    def rows_of(t, width, stride):   # tiled storage of one tile row, wider than the matrix
        d = aexq.describe(t, m, width)
        d.layout, d.storage = aexq.LAYOUT_PACK4_TILED, type(d.storage)(3, stride // 4, m, 1, 4)
        return d

    def kernel(xs, rs):   # (planned only: rows that far apart are not there)
        yd = rows_of(y, n, rs)
        return ctx.plan_check(w, rows_of(x, k, xs), yd, residual=yd).split()[0]

    assert kernel(k, n) == "kernel=wave"
    assert kernel((1 << 23) - 8, (1 << 22) - 8) == "kernel=wave"
    assert kernel(1 << 23, n) != "kernel=wave"
    assert kernel(k, 1 << 22) != "kernel=wave"


@pytest.mark.parametrize("m,kernel", [(1 << 19, "wave"), (1 << 20, "generic")])
def test_more_rows_than_one_grid_dimension_holds(ctx, aexq, m, kernel):
    """Ragged launches of 2^32 threads and more stay on the generic kernel, whose
    rows have a grid dimension of their own (planned only: no such rows are there)."""
    print(f"[gpu-case] wave split grid m={m}", flush=True)
    n, k = 16400, 48
    w = ctx.weight(aexq.QuantizedTensor(n * k, k, np.zeros(n * k // 4, np.uint32),
                                        np.ones(n, np.float16), bits=8), n, k)
    x = aexq.describe(torch.zeros(k, dtype=torch.float16, device="cuda"), 1, k)
    y = aexq.describe(torch.zeros(n, dtype=torch.float16, device="cuda"), 1, n)
    for d in (x, y):
        d.logical.h = d.storage.h = m
    assert plan_kernel(ctx.plan_check(w, x, y)) == kernel


def test_other_kernels_where_they_stay(ctx, aexq, orc):
    """Forms the wave-split kernel does not take: one row and short ragged rows
    stream, K of odd 64s is tiled, fp32 rows and other groups go where they went."""
    print("[gpu-case] wave split boundaries", flush=True)
    lay = aexq.LAYOUT_PACK4_LINEAR

    def kernel(fmt, m, n, k, dt=torch.float16, **kw):
        w, _ = _weight(ctx, aexq, orc, fmt, n, k, 2)
        x = torch.zeros(m * k, dtype=dt, device="cuda")
        y = aexq.new_activation(m, n, torch.float16, lay)
        return ctx.plan_check(w, aexq.describe(x, m, k), aexq.describe(y, m, n, lay),
                              **kw).split()[0]

    assert kernel("q4h", 1, 64, 1024) == "kernel=qmv"
    assert kernel("q4h", 5, 64, 1056) == "kernel=qmv"
    assert kernel("q8h", 16, 64, 1088) == "kernel=qgemm"
    assert kernel("q8h", 40, 64, 320) == "kernel=qgemm"
    assert kernel("q8h", 16, 64, 1000) == "kernel=generic"
    assert kernel("q8h", 16, 64, 1008, dt=torch.float32) == "kernel=generic"
    assert kernel("q8h", 512, 8192, 1024) == "kernel=qgemm"
    with pytest.raises(Exception):   # SwiGLU-out off 64-code rows stays refused
        w, _ = _weight(ctx, aexq, orc, "q8h", 64, 1008, 2)
        x = torch.zeros(16 * 1008, dtype=torch.float16, device="cuda")
        y = aexq.new_activation(16, 64, torch.float16, lay)
        ctx.plan_check(w, aexq.describe(x, 16, 1008), aexq.describe(y, 16, 64, lay), up=w)


@pytest.mark.parametrize("fmt,m,n,k,epi,here", [
    # long rows of few tiles, with the norm inside and without; groups of 16 sooner
    ("q8h", 16, 1024, 12288, "plain", True), ("q8h", 16, 1024, 12416, "plain", False),
    ("q8h", 16, 1024, 12416, "rms", True), ("q4g16s", 5, 64, 6272, "plain", False),
    ("q4h", 5, 4200, 1152, "rms", False), ("q4h", 5, 4200, 1024, "rms", True),
    # more than a workgroup per CU: pairs, streamed Q8, the norm over long rows
    ("q8h", 7, 8190, 256, "swiglu", True), ("q8h", 7, 8200, 256, "swiglu", False),
    ("q4h", 7, 8200, 256, "swiglu", True), ("q8h", 7, 16400, 256, "plain", False),
    ("q4h", 7, 16400, 256, "plain", True), ("q4h", 9, 9000, 1664, "rms", False),
    # exact pairs in groups of 16, on tiles of 32 rows by 32
    ("q4g16s", 23, 8192, 1024, "swiglu", False), ("q4h", 23, 8192, 1024, "swiglu", True),
    # tiles of 32 and 64 rows
    ("q4h", 64, 4096, 6144, "plain", True), ("q4h", 64, 4096, 6272, "plain", False),
    ("q8h", 43, 12672, 640, "plain", False), ("q8h", 43, 12160, 640, "plain", True),
    ("q4h", 600, 2048, 1024, "plain", True), ("q4h", 600, 2048, 2176, "plain", False),
    ("q4h", 600, 2048, 768, "plain", False), ("q8h", 45, 24030, 1280, "plain", False),
    # stacked copies, whose odd block fills a tile of its own
    ("q8h", 7, (22, 352), 256, "swiglu", True), ("q8h", 7, (22, 358), 256, "swiglu", False),
    # ragged rows of less than half a slice
    ("q4g16s", 1, 97, 48, "plain", False), ("q4g16s", 1, 97, 80, "plain", True),
])
def test_where_another_kernel_is_faster(ctx, aexq, fmt, m, n, k, epi, here):
    """Both sides of the lines that the rule of the wave-split kernel draws
    (planned only)."""
    print(f"[gpu-case] wave split rule {fmt} m={m} n={n} k={k} {epi}", flush=True)
    bits, group, f16, code = FORMATS[fmt]
    copies, n = n if isinstance(n, tuple) else (1, n)
    sdt = np.float16 if f16 else np.float32
    w = ctx.weight(aexq.QuantizedTensor(n * k, group or k, np.zeros(n * k * bits // 32, np.uint32),
                                        np.ones(n * k // group if group else n, sdt), bits=bits,
                                        nibble_code=code), n, k)
    if copies > 1:
        w = w.replicate(copies)
    lay = aexq.LAYOUT_PACK4_LINEAR
    x = torch.zeros(m * k, dtype=torch.float16, device="cuda")
    y = aexq.new_activation(m, n, torch.float16, lay, batch=copies)
    yd = aexq.describe(y, m, n, lay, batch=copies, batch_stride=y.numel() // copies)
    kw = {}
    if epi in ("rms", "swiglu"):
        kw.update(rmsnorm=True, rms_gamma=None, rms_eps=EPS)
    if epi == "swiglu":
        kw["up"] = w
    plan = ctx.plan_check(w, aexq.describe(x, m, k), yd, **kw)
    assert (plan_kernel(plan) == "wave") == here, plan
