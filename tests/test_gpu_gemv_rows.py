"""The decoder GEMV's row-group kernel (madi_amd/csrc/gemv.hip: 8 or 16 rows
of all of K per workgroup) at the edges of its ranges, and the sixteen waves
per panel that take 128 to 255 panels of a longer K, against the exact product
within fp32 accumulation."""
import numpy as np
import pytest

from madi_amd import synth
from test_gpu_q8 import dev, dev_f16, gelu_as64, say

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def q():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import madi_amd.q8 as q8
    q8.init()
    return q8


# rows: one, a partial and a whole group, a last panel of one and of nine rows,
# the largest of 8 rows a workgroup and the next, the last narrow width and
# the first wide one; K: one chunk, odd counts, the most of one pair a wave
# (32 chunks) and the next, the most in flight at once (96) and beyond.
# Sixteen waves per panel: the first and last panel count, both sides of K =
# 1536, odd chunk counts, one window per wave (32 chunks) and more.
@pytest.mark.parametrize("n,k", [
    (1, 64), (7, 64), (8, 128), (9, 192), (33, 320), (41, 2048), (26, 2112), (2304, 192), (2305, 192),
    (2311, 2112), (8160, 128), (8161, 128), (40, 6144), (40, 6208), (2344, 6272), (17, 12288),
    (4064, 1600), (4065, 1600), (4065, 1536), (4100, 2048), (5120, 2112), (8160, 3136), (8161, 1600),
    (4096, 12288),
])
def test_rows_against_exact(q, n, k):
    say(f"gemv rows n={n} k={k}")
    x16, qs, sc = synth.gemv_case(n * 3 + k, n, k)
    rng = np.random.default_rng(n + k)
    x = rng.standard_normal(k).astype(np.float32)
    bias, res = (rng.standard_normal(n).astype(np.float32) for _ in range(2))
    w = q.upload_q8(qs, sc)
    w64 = qs.astype(np.float64) * np.repeat(sc.astype(np.float64), 32, axis=1)

    def run(call, v):
        big = dev(np.concatenate([res, np.full(64, 7.0, np.float32)]))  # rows past n stay
        call(big)
        q.sync()
        out = big.cpu().numpy()
        assert np.all(out[n:] == 7.0)
        exact = w64 @ v.astype(np.float64)
        mag = np.abs(w64) @ np.abs(v.astype(np.float64))
        return out[:n].astype(np.float64), exact, (k * 2.0**-24 + 2.0**-21) * mag

    xd, bd = dev(x), dev(bias)
    got, exact, bound = run(lambda o: q.kGemvQ8(o, xd, w, n, k), x)
    assert np.all(np.abs(got - exact) <= bound)
    got, exact, bound = run(lambda o: q.gemv_f16x(o, dev_f16(x16), w, n, k), x16)
    assert np.all(np.abs(got - exact) <= bound)
    got, exact, bound = run(lambda o: q.kGemvQ8Bias(o, xd, w, bd, n, k), x)
    v = exact + bias
    bound = bound + 2.0**-23 * np.abs(v)
    assert np.all(np.abs(got - v) <= bound)
    got, _, _ = run(lambda o: q.kGemvQ8BiasEpi("gemv_q8_bias_gelu", o, xd, w, bd, n, k), x)
    assert np.all(np.abs(got - gelu_as64(v)) <= 1.13 * bound + 4e-7 * (1.0 + np.abs(v)))
    got, _, _ = run(lambda o: q.kGemvQ8BiasEpi("gemv_q8_bias_res", o, xd, w, bd, n, k), x)
    assert np.all(np.abs(got - (res + v)) <= bound + 2.0**-22 * (np.abs(res) + np.abs(v)))


@pytest.mark.parametrize("d", [64, 832])  # 16 rows a workgroup (832: a width of 2496) and 8
def test_rows_qkv(q, d):
    x16, qs, sc = synth.gemv_case(d, 3 * d, d)
    x = x16.astype(np.float32)
    rng = np.random.default_rng(d)
    qb, vb = (rng.standard_normal(d).astype(np.float32) for _ in range(2))
    w = q.upload_q8(qs, sc)
    qo = torch.empty(d, dtype=torch.float32, device="cuda")
    kc, vc = (torch.full((4, d), f, dtype=torch.float32, device="cuda") for f in (5.0, -5.0))
    q.kQkv(qo, dev(x), w, dev(qb), dev(vb), kc, vc, torch.tensor([2], dtype=torch.int32, device="cuda"), d)
    q.sync()
    w64 = qs.astype(np.float64) * np.repeat(sc.astype(np.float64), 32, axis=1)
    y = w64 @ x.astype(np.float64)
    bound = (d * 2.0**-24 + 2.0**-21) * (np.abs(w64) @ np.abs(x.astype(np.float64))) + 2.0**-22
    for got, want, b in ((qo, y[:d] + qb, bound[:d]), (kc[2], y[d:2 * d], bound[d:2 * d]),
                         (vc[2], y[2 * d:] + vb, bound[2 * d:])):
        assert np.all(np.abs(got.cpu().numpy() - want) <= b + 2.0**-23 * np.abs(want))
    for c, f in ((kc, 5.0), (vc, -5.0)):
        assert torch.all(c[[0, 1, 3]] == f)


def test_rows_infinite_x(q):
    """A missing chunk (an odd count, a window's pairs past the range) adds
    nothing even where the activations it stands in for are infinite."""
    for n, k in ((16, 192), (16, 5120), (4096, 1600), (4096, 3136)):
        x16, qs, sc = synth.gemv_case(3, n, k)
        x = x16.astype(np.float32)
        x[-3] = np.inf
        qs[:, -3] = 1 + np.arange(n) % 100
        w = q.upload_q8(qs, sc)
        out = torch.empty(n, dtype=torch.float32, device="cuda")
        q.kGemvQ8(out, dev(x), w, n, k)
        q.sync()
        assert torch.all(out == float("inf")), (n, k)
