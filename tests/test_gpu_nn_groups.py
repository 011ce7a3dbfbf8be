"""The F16-weight GEMM's tile order (madi_amd/csrc/f16gemm.hip): row tiles are
walked in groups of six, a last group that is not whole among them, where
their A rows do not fit an L2, and column by column elsewhere; every tile is
computed once."""
import numpy as np
import pytest

import oracle as O
from test_gpu_q8 import TOL, dev, dev_f16, host_f16, normwise, say

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


# ungrouped; then in groups: 64 x 128 tiles (13 row tiles, 24, 25), 128 x 128
# (16, 19), 128 x 256 (29, 33); and the last shape of each before its line
@pytest.mark.parametrize("m,n,k", [
    (768, 128, 64), (769, 256, 128), (1153, 384, 64), (1500, 1280, 128),
    (769, 1280, 5120), (1500, 1280, 1280), (1537, 1280, 1280), (1921, 1280, 1280), (2305, 1280, 1280),
    (3585, 2048, 640), (4100, 1536, 1024), (768, 1280, 5120), (1408, 1280, 1280), (1920, 1408, 1280),
    (3584, 2048, 640),
])
def test_groups_of_row_tiles(m, n, k):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import madi_amd.q8 as q
    q.init()
    say(f"nn groups m={m} n={n} k={k}")
    rng = np.random.default_rng(m + n)
    a = rng.standard_normal((m, k)).astype(np.float16)
    b = (rng.standard_normal((k, n)) * 0.05).astype(np.float16)
    bias = rng.standard_normal(n).astype(np.float32)
    out = torch.full((m + 8, n), 0x7E00, dtype=torch.int16, device="cuda")
    q.kM4("m4_gemm_nn", dev_f16(a), dev_f16(b), out, m, n, k)
    q.sync()
    assert np.all(out[m:].cpu().numpy() == 0x7E00)
    got = host_f16(out)[:m].astype(np.float64)
    exact = a.astype(np.float64) @ b.astype(np.float64)
    mag = np.abs(a.astype(np.float64)) @ np.abs(b.astype(np.float64))
    assert np.all(np.abs(got - exact) <= 2.0**-11 * np.abs(exact) + k * 2.0**-24 * mag + 2.0**-25)
    assert normwise(got, O.gemm_f16(a, b, threads=16)) <= TOL
    q.kM4Bias("m4_gemm_bias", dev_f16(a), dev_f16(b), out, dev(bias), m, n, k)
    q.sync()
    want = (exact.astype(np.float16).astype(np.float64) + bias)
    assert normwise(host_f16(out)[:m], want) <= TOL
