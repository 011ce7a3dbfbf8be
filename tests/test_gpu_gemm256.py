"""The 256 x 256 tiles of the many-row Q8 GEMM (madi_amd/csrc/gemm256.hip)
through the C ABI, against the oracle and element-wise against the exact
product (fp32 accumulation plus one f16 rounding)."""
import numpy as np
import pytest

import oracle as O
from madi_amd import _lib, synth
from test_gpu_q8 import TOL, dev, dev_f16, host_f16, normwise, say, tight_epi_ok, tight_ok

torch = pytest.importorskip("torch")


def takes_256(m, n, k, cus=256):
    """The dispatch of madi_q8_gemm (gemm.hip, gemm256.hip) up to the 256 x 256
    tiles: whether an eager call over m rows takes them."""
    def tiles(mt, pw=2):
        return -(-m // (32 * mt)) * -(-n // (128 * pw))

    chunks = k // 64
    if m <= 64 or (tiles(4) < 160 and chunks >= 64 and 240 // tiles(4) > 1):
        return False  # few rows; K split
    if min(tiles(1), tiles(2), tiles(3)) <= cus:
        return False  # lower tiles, one per CU
    t, fused = -(-m // 256) * (n // 256), -(-m // 128) * (n // 256)
    rounds, fused_rounds = -(-t // cus), -(-fused // cus)
    if n % 256 or n * k * 2 >= 16 << 20 or n * 512 >= 1 << 31:
        return False
    if t * 10 < rounds * cus * 9 or rounds * 30 > fused_rounds * 16:
        return False
    return m >= 5120 if rounds >= 2 else m >= 10240 and k >= 3072


# Streams (the chunks of a workgroup's tiles) of one and two chunks, of two and
# four, three and six, four and eight, of two and three tiles; row tails of
# one, 65, 76 and 112 rows; one tile a workgroup (K from 3072); a fifteenth more
# rounds than the fused kernels.
CASES = [
    (5120, 6144, 64, O.EPI_NONE), (5121, 5888, 64, O.EPI_BIAS), (5185, 5888, 128, O.EPI_BIAS_GELU),
    (7500, 4096, 192, O.EPI_NONE), (6000, 5120, 256, O.EPI_BIAS), (12700, 3840, 128, O.EPI_BIAS_GELU),
    (10241, 1536, 3072, O.EPI_BIAS), (24000, 5120, 64, O.EPI_NONE), (6000, 5120, 1280, O.EPI_BIAS_GELU),
]
# Next to them, on the fused kernels: a row fewer, a K shorter, more rounds than
# a fifteenth more, a round less than nine tenths full; few rows of wide
# weights in one round (one of 256 tiles of 96 rows) and in two and three.
OTHERS = [
    (5119, 6144, 64, O.EPI_NONE), (10240, 1536, 3008, O.EPI_BIAS), (17700, 5120, 64, O.EPI_NONE),
    (5888, 5120, 256, O.EPI_BIAS), (65, 65536, 64, O.EPI_NONE), (256, 59136, 128, O.EPI_BIAS),
    (500, 29696, 192, O.EPI_BIAS_GELU), (600, 20480, 256, O.EPI_NONE),
    (1900, 15872, 192, O.EPI_BIAS_GELU), (2305, 19456, 64, O.EPI_BIAS),
]


def test_cases_take_their_routes():
    assert all(takes_256(*c[:3]) for c in CASES)
    assert not any(takes_256(*c[:3]) for c in OTHERS)
    # the persistent tile loop's own shapes (test_gpu_q8.py)
    assert not any(takes_256(*c) for c in ((21000, 5120, 768), (21000, 5120, 1280), (14600, 5120, 1280),
                                           (5500, 5120, 1280), (7001, 4096, 768), (13300, 1280, 2048)))
    # windows of 1500 rows, the encoder's MLP
    assert [w for w in range(1, 17) if takes_256(1500 * w, 5120, 1280)] == [4, 6, 8, 10, 12, 15, 16]
    assert [w for w in range(1, 17) if takes_256(1500 * w, 1280, 5120)] == [8, 16]


@pytest.fixture(scope="module")
def q():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import madi_amd.q8 as q8
    q8.init()
    return q8


def check(c, a, qs, sc, bias, epi, rows):
    b = None if epi == O.EPI_NONE else bias
    ref = O.q8_gemm_rows(a, qs, sc, rows=rows, bias=b, epilogue=epi, threads=16)
    assert normwise(c[rows], ref) <= TOL
    if epi == O.EPI_NONE:
        assert tight_ok(c[rows], a[rows], qs, sc)
    else:
        assert tight_epi_ok(c[rows], a[rows], qs, sc, bias, epi == O.EPI_BIAS_GELU)
    assert np.all(np.isfinite(c))


@pytest.mark.gpu
@pytest.mark.parametrize("m,n,k,epi", CASES + OTHERS)
def test_tiles_against_oracle(q, m, n, k, epi):
    say(f"gemm256 m={m} n={n} k={k} epi={epi}")
    a, qs, sc = synth.gemm_case(m + k, m, n, k)
    bias = np.random.default_rng(m).standard_normal(n).astype(np.float32)
    w = q.upload_q8(qs, sc)
    big = torch.full((m + 8, n), 0x7E00, dtype=torch.int16, device="cuda")  # rows past M stay
    a_d, b_d = dev_f16(a), dev(bias)
    call = lambda name: _lib.call(name, a_d.data_ptr(), w.qs, w.scales, big.data_ptr(),
                                  None if epi == O.EPI_NONE else b_d.data_ptr(), m, n, k, epi)
    call("madi_q8_gemm")
    q.sync()
    out = big.cpu().numpy()
    assert np.all(out[m:] == 0x7E00)
    edges = np.arange(128, m, 128)
    rows = np.unique(np.r_[0, 15, 16, 63, 64, m // 2, m - 2, m - 1, edges[:8] - 1, edges[:8]])
    check(host_f16(big)[:m], a, qs, sc, bias, epi, rows)
    # again, and through the other entry point: the same bits
    for name in ("madi_q8_gemm", "madi_q8_gemm_noalloc"):
        big.fill_(0x7E00)
        call(name)
        q.sync()
        assert np.array_equal(big.cpu().numpy(), out), name
    # which kernel ran: a captured call takes the fused ones, whose sums are in
    # another order
    assert np.array_equal(captured(q, call, big), out) != takes_256(m, n, k)


def capture(q, call):
    """A graph of `call`, captured on a stream of its own."""
    torch.cuda.synchronize()
    g, side = torch.cuda.CUDAGraph(), torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        with torch.cuda.graph(g, stream=side):
            q.init(side)
            call()
    q.init()
    return g


def captured(q, call, out):
    """The result of a captured madi_q8_gemm, replayed once."""
    g = capture(q, lambda: call("madi_q8_gemm"))
    out.fill_(0x7E00)
    g.replay()
    torch.cuda.synchronize()
    return out.cpu().numpy()


@pytest.mark.gpu
def test_captured_noalloc_is_the_captured_gemm(q):
    """Captured, the two entry points take the same kernels (the fused ones,
    which share no memory with other calls): the same bits, over replays with
    eager calls of another weight through the fixed scratch between them."""
    m, n, k = 6000, 5120, 1280
    say(f"gemm256 noalloc capture m={m} n={n} k={k}")
    a, qs, sc = synth.gemm_case(11, m, n, k)
    bias = np.random.default_rng(12).standard_normal(n).astype(np.float32)
    w, a_d, b_d = q.upload_q8(qs, sc), dev_f16(a), dev(bias)
    a2, qs2, sc2 = synth.gemm_case(13, m, n, k)
    w2, a2_d = q.upload_q8(qs2, sc2), dev_f16(a2)
    outs, graphs = [], []
    for name in ("madi_q8_gemm", "madi_q8_gemm_noalloc"):
        c = torch.empty((m, n), dtype=torch.int16, device="cuda")
        args = (a_d.data_ptr(), w.qs, w.scales, c.data_ptr(), b_d.data_ptr(), m, n, k, O.EPI_BIAS)
        graphs.append(capture(q, lambda: _lib.call(name, *args)))
        outs.append(c)
    eager = torch.empty((m, n), dtype=torch.int16, device="cuda")
    first = None
    for rep in range(3):
        for g, c in zip(graphs, outs):
            c.fill_(-1)
            g.replay()
            torch.cuda.synchronize()
            if first is None:
                first = c.cpu().numpy()
                rows = np.unique(np.r_[0, 127, 128, 255, 256, 3000, m - 1])
                check(host_f16(c), a, qs, sc, bias, O.EPI_BIAS, rows)
            assert np.array_equal(c.cpu().numpy(), first), rep
            _lib.call("madi_q8_gemm_noalloc", a2_d.data_ptr(), w2.qs, w2.scales, eager.data_ptr(),
                      b_d.data_ptr(), m, n, k, O.EPI_BIAS)
            q.sync()
    check(host_f16(eager), a2, qs2, sc2, bias, O.EPI_BIAS, rows)


@pytest.mark.gpu
def test_captured_calls_share_no_scratch(q):
    """A captured call runs the fused kernels, before and after the first
    eager one: the graphs' replays, with eager calls of the same shape and
    another weight between, repeat their bits and are within the bounds."""
    m, n, k = 6000, 5120, 1280
    say(f"gemm256 capture m={m} n={n} k={k}")
    _lib.lib().madi_cleanup()
    q.init()
    a, qs, sc = synth.gemm_case(5, m, n, k)
    bias = np.random.default_rng(6).standard_normal(n).astype(np.float32)
    w = q.upload_q8(qs, sc)
    a_d, b_d = dev_f16(a), dev(bias)
    rows = np.unique(np.r_[0, 127, 128, 255, 256, 3000, m - 1])
    graphs = []
    for _ in range(2):
        c = torch.empty((m, n), dtype=torch.int16, device="cuda")
        torch.cuda.synchronize()
        g = torch.cuda.CUDAGraph()
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            with torch.cuda.graph(g, stream=side):
                q.init(side)
                q.kGemmQ8Bias(a_d, w, c, b_d, m, n, k, gelu=True)
        q.init()
        graphs.append((g, c))
        eager = torch.empty((m, n), dtype=torch.int16, device="cuda")
        q.kGemmQ8Bias(a_d, w, eager, b_d, m, n, k, gelu=True)
        q.sync()
    first = [None, None]
    a2, qs2, sc2 = synth.gemm_case(7, m, n, k)
    w2, a2_d = q.upload_q8(qs2, sc2), dev_f16(a2)
    for rep in range(3):
        for i, (g, c) in enumerate(graphs):
            c.fill_(-1)
            g.replay()
            torch.cuda.synchronize()
            got = host_f16(c)
            if rep == 0:
                first[i] = got.copy()
                check(got, a, qs, sc, bias, O.EPI_BIAS_GELU, rows)
            assert np.array_equal(got.view(np.uint16), first[i].view(np.uint16)), (rep, i)
            q.kGemmQ8Bias(a2_d, w2, eager, b_d, m, n, k, gelu=True)
            q.sync()
    assert np.array_equal(first[0].view(np.uint16), first[1].view(np.uint16))
    check(host_f16(eager), a2, qs2, sc2, bias, O.EPI_BIAS_GELU, rows)


@pytest.mark.gpu
def test_weight_is_not_in_the_workspace(q):
    """An eager many-row call keeps its 13 MB weight out of the split-K
    workspace (4 MiB after madi_init), which captured calls use: it takes no
    device memory."""
    m, n, k = 6000, 5120, 1280
    _lib.lib().madi_cleanup()
    q.init()
    a, qs, sc = synth.gemm_case(5, m, n, k)
    w, a_d = q.upload_q8(qs, sc), dev_f16(a)
    c = torch.empty((m, n), dtype=torch.int16, device="cuda")
    for call in (q.kGemmQ8, lambda *v: _lib.call("madi_q8_gemm_noalloc", v[0].data_ptr(), w.qs, w.scales,
                                                 c.data_ptr(), None, m, n, k, O.EPI_NONE)):
        q.sync()
        before = torch.cuda.mem_get_info()[0]
        call(a_d, w, c, m, n, k)
        q.sync()
        assert torch.cuda.mem_get_info()[0] == before


@pytest.mark.gpu
def test_replayed_split_k_beside_an_eager_call(q):
    """Split-K calls, captured, replay on a stream of their own while eager
    many-row calls run on the library's: each result keeps its bits."""
    say("gemm256 beside a replayed split K")
    m, n, k = 6000, 5120, 1280
    a, qs, sc = synth.gemm_case(21, m, n, k)
    w, a_d = q.upload_q8(qs, sc), dev_f16(a)
    ms, ns, ks = 300, 1280, 5120
    a_s, qs_s, sc_s = synth.gemm_case(22, ms, ns, ks)
    w_s, as_d = q.upload_q8(qs_s, sc_s), dev_f16(a_s)
    x_d = dev(synth.activations(np.random.default_rng(23), 16, ks).astype(np.float32))

    def new():
        return (torch.empty((m, n), dtype=torch.int16, device="cuda"),
                torch.empty((ms, ns), dtype=torch.int16, device="cuda"),
                torch.empty((16, ns), dtype=torch.float32, device="cuda"))

    def many(c):
        q.kGemmQ8(a_d, w, c, m, n, k)

    def split(c, p):
        q.kGemmQ8(as_d, w_s, c, ms, ns, ks)
        q.pproj(x_d, w_s, p, 16, ns, ks)

    want, got = new(), new()
    many(want[0])
    split(*want[1:])
    q.sync()
    g, side = capture(q, lambda: split(*got[1:])), torch.cuda.Stream()
    for rep in range(4):
        for t in got:
            t.fill_(-1)
        torch.cuda.synchronize()
        for _ in range(6):
            many(got[0])
            with torch.cuda.stream(side):
                for _ in range(4):
                    g.replay()
        torch.cuda.synchronize()
        for t, v in zip(got, want):
            assert torch.equal(t, v), rep
