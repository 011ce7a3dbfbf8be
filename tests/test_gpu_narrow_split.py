"""64 x 128 tiles of the Q8 GEMM with K split over workgroups (a long K on few
rows, madi_amd/csrc/gemm.hip): against the oracle and element-wise, every
split count and epilogue; and its vmcnt waits (CPU)."""
import numpy as np
import pytest

import oracle as O
from isa_vmcnt import hazards
from madi_amd import _lib, synth
from test_gpu_q8 import TOL, dev, dev_f16, host_f16, normwise, say, tight_epi_ok, tight_ok, tile_rows
from test_isa_vmcnt import gemm_asm  # noqa: F401 (fixture)

torch = pytest.importorskip("torch")


def test_every_instance_is_race_free(gemm_asm):  # noqa: F811
    names = [n for n in gemm_asm if "q8_gemm_narrow_split_kernel" in n]
    assert len(names) == 3, names
    assert not {n: b for n in names if (b := hazards(gemm_asm[n])[:3])}


# four splits (the smallest row count past 64, ragged, the most tiles), three
# (96 chunks), two, and N that ends inside a tile's columns
@pytest.mark.gpu
@pytest.mark.parametrize("m,n,k,epi", [
    (65, 1280, 5120, O.EPI_NONE), (257, 1280, 5120, O.EPI_BIAS_GELU), (384, 1280, 5120, O.EPI_BIAS),
    (500, 1280, 6144, O.EPI_BIAS), (701, 1280, 5120, O.EPI_BIAS_GELU), (130, 1312, 4096, O.EPI_NONE),
    (70, 96, 8192, O.EPI_BIAS),
])
def test_narrow_split(m, n, k, epi):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import madi_amd.q8 as q
    q.init()
    say(f"narrow split m={m} n={n} k={k} epi={epi}")
    a, qs, sc = synth.gemm_case(m + n + k, m, n, k)
    bias = np.random.default_rng(m).standard_normal(n).astype(np.float32)
    w = q.upload_q8(qs, sc)
    a_d, b_d = dev_f16(a), dev(bias)
    big = torch.full((m + 8, n), 0x7E00, dtype=torch.int16, device="cuda")  # rows past M stay
    outs = []
    for name in ("madi_q8_gemm", "madi_q8_gemm", "madi_q8_gemm_noalloc"):
        big.fill_(0x7E00)
        _lib.call(name, a_d.data_ptr(), w.qs, w.scales, big.data_ptr(),
                  None if epi == O.EPI_NONE else b_d.data_ptr(), m, n, k, epi)
        q.sync()
        outs.append(big.cpu().numpy())
        assert np.all(outs[-1][m:] == 0x7E00) and np.array_equal(outs[-1], outs[0]), name
    c, rows = host_f16(big)[:m], tile_rows(m)
    b = None if epi == O.EPI_NONE else bias
    ref = O.q8_gemm_rows(a, qs, sc, rows=rows, bias=b, epilogue=epi, threads=16)
    assert normwise(c[rows], ref) <= TOL
    if epi == O.EPI_NONE:
        assert tight_ok(c[rows], a[rows], qs, sc)
    else:
        assert tight_epi_ok(c[rows], a[rows], qs, sc, bias, epi == O.EPI_BIAS_GELU)
