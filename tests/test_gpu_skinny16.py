"""The batched projection's kernel with a workgroup per 16 weight rows
(madi_amd/csrc/skinny.hip) at the edges of its ranges: element-wise within
fp32 accumulation of the f16-staged operands, rows and columns past the
result untouched."""
import numpy as np
import pytest

import oracle as O
from madi_amd import synth
from test_gpu_q8 import dev, say

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def q():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import madi_amd.q8 as q8
    q8.init()
    return q8


# activation rows: one, the edges of the 8-, 16- and 32-row forms, a second
# slice of one row and several; weight rows: less than a group, a last panel
# of 1, 9, 17 and 26 rows, one workgroup per CU and one more, wider; K: one chunk, odd
# counts, one window per wave (24 chunks) and the next, the routes' lines at
# 1536 (more than 16 rows), 2048 and 5120 (up to 2048 weight rows), long ones
# (80 and 81 chunks)
@pytest.mark.parametrize("m,n,k", [
    (1, 7, 64), (8, 16, 128), (9, 33, 192), (16, 41, 1536), (17, 49, 1600), (32, 90, 1280), (33, 40, 320),
    (100, 26, 704), (16, 4096, 64), (16, 4097, 64), (9, 3840, 1280), (8, 8192, 128), (8, 1280, 2048),
    (8, 1280, 2112), (5, 1281, 5120), (8, 300, 5184), (9, 300, 5184), (320, 384, 384),
    (17, 49, 1536), (33, 200, 1536), (16, 49, 1600), (16, 49, 2048), (17, 49, 2048), (8, 2048, 5120),
    (8, 2048, 5184), (8, 2049, 5184), (3, 640, 12288),
])
def test_rows_against_exact(q, m, n, k):
    say(f"skinny16 m={m} n={n} k={k}")
    rng = np.random.default_rng(m * 7 + n + k)
    qs, sc = synth.q8_weight(rng, n, k)
    x = rng.standard_normal((m, k)).astype(np.float32)
    w = q.upload_q8(qs, sc)
    big = torch.full((m * n + 4096,), 7.0, dtype=torch.float32, device="cuda")
    q.pproj(dev(x), w, big, m, n, k)
    q.sync()
    out = big.cpu().numpy()
    assert np.all(out[m * n:] == 7.0)
    got = out[:m * n].reshape(m, n).astype(np.float64)
    w16 = O.dequant_q8_f16(qs, sc).astype(np.float64)  # [K][N]
    x16 = x.astype(np.float16).astype(np.float64)
    exact, mag = x16 @ w16, np.abs(x16) @ np.abs(w16)
    assert np.all(np.abs(got - exact) <= k * 2.0**-24 * mag + 1e-30)
    again = torch.empty((m, n), dtype=torch.float32, device="cuda")
    q.pproj(dev(x), w, again, m, n, k)
    q.sync()
    assert np.array_equal(again.cpu().numpy(), out[:m * n].reshape(m, n))
