"""aexq_rmsnorm over fp16 rows, both forms, against the oracle: one rounding to
fp16 of each value (2^-11 relative) and the order of the row's sum, 1e-3."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu

TOL = 1e-3


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


@pytest.mark.parametrize("m,k,off,gamma", [(1, 8, 0, True), (5, 1024, 0, True), (64, 1032, 0, False),
                                           (67, 2048, 0, True), (3, 4096, 0, True),
                                           (3, 4104, 0, True), (9, 512, 1, True), (9, 500, 0, True)])
def test_rmsnorm_rows(ctx, aexq, orc, m, k, off, gamma):
    """Rows in a wave's registers (up to 4096, 16-byte aligned) and the other
    form: longer rows, rows at an odd address, K not a multiple of 8."""
    print(f"[gpu-case] rmsnorm m={m} k={k} off={off}", flush=True)
    from aiimage_amd import synth
    x16 = synth.activations(m, k, 4)
    buf = torch.zeros(m * k + 8, dtype=torch.float16, device="cuda")
    x = buf[off:off + m * k]
    x.copy_(dev(x16).reshape(-1))
    g = synth.rms_gamma(k, 6) if gamma else None
    y = torch.full((m * k,), 7.0, dtype=torch.float16, device="cuda")
    ctx.rmsnorm(aexq.describe(x, m, k), aexq.describe(y, m, k), dev(g) if gamma else None, 1e-6)
    torch.cuda.synchronize()
    ref = orc.rmsnorm(x16.astype(np.float32), 1e-6, g).astype(np.float64)
    assert np.max(np.abs(y.cpu().numpy().reshape(m, k) - ref) / np.maximum(np.abs(ref), 1e-2)) <= TOL
