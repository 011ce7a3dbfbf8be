"""The attention's 32- and 64-row query tiles (short sequences,
madi_amd/csrc/attn.hip): at the lines between the tile heights and ragged
tails, against the fp64 attention and the oracle; in place on q; and their
vmcnt waits (CPU)."""
import numpy as np
import pytest

from isa_vmcnt import hazards
from test_gpu_flash import check, dev_f16, q8, qkv, run, say  # noqa: F401 (fixture)
from test_isa_vmcnt import attn_asm  # noqa: F401 (fixture)

torch = pytest.importorskip("torch")


def test_every_instance_is_race_free(attn_asm):  # noqa: F811
    names = [n for n in attn_asm if "flash_short_kernel" in n]
    assert len(names) == 2, names
    assert not {n: b for n in names if (b := hazards(attn_asm[n])[:3])}


# On 256 CUs: 32-row tiles up to 512 frames of 16 heads and 1024 of 8, 64-row
# ones up to twice that.  Fewer key blocks than the four key groups (1, 31,
# 100), one to three per group, and query tails of 1, 31, 32, 33 and 63 rows.
@pytest.mark.gpu
@pytest.mark.parametrize("seq,nh,scale,dist", [
    (1, 3, 1.0, "normal"), (31, 2, 1.0, "normal"), (33, 20, 2.0, "normal"), (100, 6, 1.0, "uniform"),
    (375, 20, 1.0, "normal"), (512, 16, 2.0, "normal"), (513, 16, 1.0, "normal"), (575, 16, 3.0, "normal"),
    (1024, 16, 1.0, "uniform"), (1025, 16, 1.0, "normal"), (1023, 8, 1.0, "normal"), (1057, 8, 2.0, "normal"),
])
def test_short_tiles(q8, seq, nh, scale, dist):  # noqa: F811
    say(f"flash short seq={seq} nh={nh} {dist}")
    rng = np.random.default_rng(seq * 7 + nh)
    q, k, v = qkv(rng, seq, nh, scale, dist)
    got = run(q8, q, k, v, nh)
    check(got, q, k, v, nh)
    # again, with rows past the sequence left alone, and in place on q
    big = torch.full((seq + 64, nh * 64), 0x7E00, dtype=torch.int16, device="cuda")
    again = run(q8, q, k, v, nh, out=big)
    assert np.array_equal(again[:seq].view(np.uint16), got.view(np.uint16))
    assert np.all(again[seq:].view(np.uint16) == 0x7E00)
    tq = dev_f16(q)
    q8.kFlash("m4_flash_enc", tq, tq, dev_f16(k), dev_f16(v), seq, nh)
    torch.cuda.synchronize()
    assert np.array_equal(tq.cpu().numpy().view(np.uint16), got.view(np.uint16))
