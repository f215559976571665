"""GPU parity: the device encoder behind kq.quantize reproduces the reference's own fixture bytes inside the
reference's x86-vs-Metal band, writes the host encoder's bytes, and what it writes decodes within the codec's bound."""
import os

import numpy as np
import pytest
import torch

import oracle_lib as O

pytestmark = pytest.mark.gpu
DEV_CODECS = ["q8_0", "q4_0", "q4_1", "q5_0", "q5_1", "q2_k", "q3_k", "q4_k", "q5_k", "q6_k"]
# round-trip rel-L2 bounds on N(0, 1) rows: loose sanity limits per bit width
BOUND = {"q8_0": 0.02, "q4_0": 0.2, "q4_1": 0.2, "q5_0": 0.1, "q5_1": 0.1, "q2_k": 0.5, "q3_k": 0.3, "q4_k": 0.15,
         "q5_k": 0.08, "q6_k": 0.05}


@pytest.fixture(scope="module")
def kq():
    import kq as _kq
    return _kq


@pytest.mark.parametrize("codec", DEV_CODECS)
def test_device_encoder_writes_host_bytes(kq, codec):
    rng = np.random.default_rng(100 + O.codec_id(codec))
    rows, K = 37, 1024
    w = rng.standard_normal((rows, K)).astype(np.float32)
    w[3] = 0.0                                 # an all-zero row
    w[5, :256] = 0.0                           # a zero superblock inside a live row
    w[7] *= 1e-6                               # tiny magnitudes
    w[9, ::7] *= 40.0                          # outliers
    im = (np.abs(rng.standard_normal(K)) + 0.1).astype(np.float32)
    wt = torch.from_numpy(w)
    for imat in (None, im):
        it = None if imat is None else torch.from_numpy(imat)
        host, _ = kq.quantize(wt, codec, it)
        dev, scales = kq.quantize(wt.cuda(), codec, None if it is None else it.cuda())
        assert dev.is_cuda and dev.dtype == torch.uint8 and tuple(dev.shape) == tuple(host.shape)
        assert tuple(scales.shape) == (1,)
        assert np.array_equal(dev.cpu().numpy(), host.numpy()), (codec, imat is not None)
    back = O.dequantize(dev.cpu().numpy(), codec).reshape(rows, K)
    live = [r for r in range(rows) if r not in (3, 9)]  # the outlier row is covered by the byte comparison only
    assert np.linalg.norm(back[live] - w[live]) / np.linalg.norm(w[live]) < BOUND[codec]
    assert not back[3].any()


GOLD = os.path.join(os.path.dirname(os.path.abspath(__file__)), "golden")
KCODECS = ["q2_k", "q3_k", "q4_k", "q5_k", "q6_k"]


@pytest.mark.parametrize("codec", KCODECS)
def test_device_encoder_reproduces_reference_fixture_bytes(kq, codec):
    """The device encoder against the reference's own vectors, directly: the committed wire fixtures were minted
    by the reference's encoder from default_rng(1234) (tests/gen_fixtures.py:62-63) on Metal, and the reference's
    x86 encoder lands within a few ULP-tie bytes of them (tests/test_encode.py:203-250).  kq.quantize on cuda:0
    must land in the same band, and what it writes must decode to what the fixture decodes to."""
    gold = np.load(os.path.join(GOLD, f"{codec}.npz"))["wire"]
    w = (np.random.default_rng(1234).standard_normal((256, 512)) * 0.1).astype(np.float32)
    dev, _ = kq.quantize(torch.from_numpy(w).cuda(), codec)
    mine = dev.cpu().numpy()
    assert mine.shape == gold.shape
    frac = np.mean(mine != gold)
    assert frac < 2e-3, (codec, frac)
    a, b = O.dequantize(mine, codec), O.dequantize(gold, codec)
    assert np.linalg.norm(a - b) / np.linalg.norm(b) < 2e-2
    # the fixture's bytes, decoded on the device, are the oracle's decode bit for bit
    got = kq.dequantize(torch.from_numpy(gold).cuda(), None, codec, dtype=torch.float32).cpu().numpy()
    assert np.array_equal(got.view(np.uint32).ravel(), b.view(np.uint32).ravel())


def test_device_encoder_reproduces_reference_moe_fixture_bytes(kq):
    """Same for the expert-stack fixtures (default_rng(4321), four experts of 128 x 512, tests/gen_fixtures.py:80-89)."""
    rng = np.random.default_rng(4321)
    ws = [(rng.standard_normal((128, 512)) * 0.1).astype(np.float32) for _ in range(4 * len(KCODECS))]
    for ci, codec in enumerate(KCODECS):
        gold = np.load(os.path.join(GOLD, f"{codec}_moe.npz"))["wire"]
        stack = np.stack(ws[4 * ci:4 * ci + 4])
        dev, _ = kq.quantize(torch.from_numpy(stack).cuda(), codec)   # leading (expert) dimension kept
        mine = dev.cpu().numpy()
        assert mine.shape == gold.shape
        for e in range(4):
            assert np.mean(mine[e] != gold[e]) < 3e-3, (codec, e)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_device_encoder_half_inputs_and_stacks(kq, dtype):
    """16-bit inputs are widened exactly as the host path widens them; leading dimensions are kept."""
    rng = np.random.default_rng(7)
    w = torch.from_numpy(rng.standard_normal((3, 5, 512)).astype(np.float32) * 0.05).to(dtype)
    for codec in ("q4_k", "q6_k", "q8_0"):
        host, _ = kq.quantize(w, codec)
        dev, _ = kq.quantize(w.cuda(), codec)
        assert tuple(dev.shape) == tuple(host.shape) and dev.shape[:2] == (3, 5)
        assert torch.equal(dev.cpu(), host)


def test_host_encoder_still_reachable_and_iq_stays_on_host(kq):
    rng = np.random.default_rng(8)
    w = torch.from_numpy(rng.standard_normal((4, 512)).astype(np.float32)).cuda()
    a, _ = kq.quantize(w, "q4_k", stream="cpu")          # forced host encoder, result back on the GPU
    b, _ = kq.quantize(w, "q4_k")
    assert a.is_cuda and torch.equal(a, b)
    lib = kq._load()
    assert lib.kq_quantize_dev_supported(lib.kq_codec_id(b"q4_k")) == 1
    assert lib.kq_quantize_dev_supported(lib.kq_codec_id(b"iq4_xs")) == 0
    c, _ = kq.quantize(w, "iq4_xs")                      # host encoder behind the same call
    assert c.is_cuda and tuple(c.shape) == (4, 272)
    assert lib.kq_quantize_dev(w.data_ptr(), 0, None, c.data_ptr(), 4, 512, lib.kq_codec_id(b"iq4_xs"), None) == -2


def test_device_encoder_large_matrix_speed_sanity(kq):
    """A Llama gate/up sized matrix: bytes equal the host's on a sample of rows; prints both times."""
    import time
    rng = np.random.default_rng(9)
    w = torch.from_numpy((rng.standard_normal((2048, 4096)) * 0.02).astype(np.float32))
    wd = w.cuda()
    kq.quantize(wd[:8], "q4_k")
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    dev, _ = kq.quantize(wd, "q4_k")
    torch.cuda.synchronize()
    t_dev = time.perf_counter() - t0
    t0 = time.perf_counter()
    host, _ = kq.quantize(w, "q4_k")
    t_host = time.perf_counter() - t0
    print(f"q4_k 2048 x 4096: device {t_dev * 1e3:.1f} ms, host {t_host * 1e3:.1f} ms")
    assert torch.equal(dev.cpu(), host)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("codec", DEV_CODECS)
def test_device_encoder_both_lane_splits_and_ragged_ends(kq, codec, dtype):
    """Bytes equal the host's on a matrix large enough for one lane per sub-block and on ones that end inside a
    workgroup, from aligned and unaligned addresses, with signed zeros, constant blocks and one-sided ones."""
    gen = torch.Generator().manual_seed(11)
    wpb = kq.CODEC_GEOMETRY[codec][3]
    for rows, K in ((2051, 1024), (1, wpb), (3, 3 * wpb)):
        w = torch.randn((rows, K), generator=gen) * 0.05
        w[0, : wpb // 2] = 0.0
        w[0, 1] = -0.0
        w[rows // 2] = w[rows // 2].abs()
        w[rows - 1, -wpb:] = -0.25
        w = w.to(dtype)
        im = torch.rand(K, generator=gen) + 0.1 if codec in kq.codec_geometry.IMATRIX_CODECS else None
        host = kq.quantize(w, codec, im)[0]
        flat = torch.empty(rows * K + 1, dtype=dtype, device="cuda")
        for off in (0, 1):  # an odd element offset: no four-element loads
            wd = flat[off:off + rows * K].copy_(w.reshape(-1)).reshape(rows, K)
            dev = kq.quantize(wd, codec, None if im is None else im.cuda())[0]
            assert torch.equal(dev.cpu(), host), (codec, rows, K, off)


def _device_bytes(kq, w, codec, im):
    """w encoded as it is (a small matrix: four lanes share a sub-block's candidates) and, repeated until it is no small one, by the
    kernel that rules candidates out: the bytes of both, rows of w by bytes."""
    w, im = w.cuda(), None if im is None else im.cuda()
    times = 2049 * 256 // w.numel() + 1
    yield kq.quantize(w, codec, im)[0].cpu().numpy()
    many = kq.quantize(w.repeat(times, 1), codec, im)[0].reshape(times, len(w), -1)
    assert torch.equal(many, many[:1].expand_as(many))
    yield many[0].cpu().numpy()


@pytest.mark.parametrize("codec", DEV_CODECS)
def test_device_encoder_nonfinite_weights_keep_their_bytes(kq, codec):
    """NaN, infinite and f16-overflowing weights: the bytes that the sequential block encoders write when compiled for the
    device, where a NaN level converts to 0 (tests/golden/encode_nonfinite.npz, made by them on gfx950; the host build
    converts a NaN to the lowest int, so kq_quantize is no reference here).  Rows: a NaN as each lane's first weight of the
    legacy blocks, infinities, whole NaN blocks, scales past the f16 range."""
    gold = np.load(os.path.join(GOLD, "encode_nonfinite.npz"))
    w, im = torch.from_numpy(gold["w"]).cuda(), torch.from_numpy(gold["imatrix"]).cuda()
    for key, imat in ((codec, None), (codec + "_im", im)):
        if key in gold:
            for got in _device_bytes(kq, w, codec, imat):
                bad = np.argwhere((got != gold[key]).any(axis=1)).ravel().tolist()
                assert not bad, (key, bad)


# rows of each kind for the encoders that rule out candidates by a bound: lattices whose levels sit on ties, one-sided and
# narrow blocks (the least-squares system near singular, the minimum held at zero), blocks that few levels fit exactly, a
# few outliers, scales near the ends of the float range and outside those for which the bound is derived
_FIT_ROWS = {
    "normal": lambda r, n: r.standard_normal(n) * 0.02,
    "bytes": lambda r, n: r.integers(-127, 128, n) * 0.0007,
    "few levels": lambda r, n: r.integers(-3, 4, n) * 0.01,
    "two values": lambda r, n: r.choice([-0.5, 0.25], n),
    "16 levels": lambda r, n: r.integers(0, 16, n) * 0.125 - 1.0,
    "one-sided": lambda r, n: np.abs(r.standard_normal(n)),
    "narrow": lambda r, n: 1.0 + r.standard_normal(n) * 0.02,
    "narrow below": lambda r, n: -1.0 + r.standard_normal(n) * 1e-4,
    "outliers": lambda r, n: r.standard_normal(n) * np.where(r.random(n) < 0.03, 50.0, 0.01),
    "peaked": lambda r, n: r.random(n) ** 8 * r.standard_normal(n),
    "sparse": lambda r, n: r.standard_normal(n) * (r.random(n) < 0.1),
    "tiny": lambda r, n: r.standard_normal(n) * 1e-8,
    "vanishing": lambda r, n: r.standard_normal(n) * 1e-22,
    "huge": lambda r, n: r.standard_normal(n) * 3e9,
}
_FIT_WEIGHTS = {
    "none": None,
    "squares": lambda r, n: r.standard_normal(n) ** 2 + 0.05,
    "wide": lambda r, n: 10.0 ** r.uniform(-9, 3, n),
    "zeros": lambda r, n: r.random(n) * (r.random(n) < 0.5),
    "negative": lambda r, n: r.standard_normal(n),
    "tiny": lambda r, n: r.random(n) * 1e-20,
}


@pytest.mark.parametrize("weights", sorted(_FIT_WEIGHTS))
@pytest.mark.parametrize("codec", KCODECS)
def test_device_encoder_fit_bytes_over_kinds_of_rows(kq, codec, weights):
    """Bytes equal the host's for every kind of row, kinds alternating by row and, in the last rows, by sub-block."""
    rng = np.random.default_rng(31 + O.codec_id(codec))
    K = 1024
    w = np.stack([f(rng, K) for f in _FIT_ROWS.values() for _ in range(8)])
    mixed = np.stack([np.concatenate([w[rng.integers(len(w)), 16 * j:16 * j + 16] for j in range(K // 16)])
                      for _ in range(16)])
    w = torch.from_numpy(np.concatenate([w, mixed]).astype(np.float32))
    make = _FIT_WEIGHTS[weights]
    im = None if make is None else torch.from_numpy(make(rng, K).astype(np.float32))
    host = kq.quantize(w, codec, im)[0].numpy()
    kinds = list(_FIT_ROWS)
    for dev in _device_bytes(kq, w, codec, im):
        bad = np.argwhere((dev != host).any(axis=1)).ravel().tolist()
        assert not bad, sorted({kinds[b // 8] if b < 8 * len(kinds) else "mixed" for b in bad})


@pytest.mark.parametrize("codec", ["q2_k", "q4_k", "q5_k"])
def test_device_encoder_fit_of_blocks_far_above_zero(kq, codec):
    """Waves of nothing but blocks without a bound, of some, and of none; weights of one size and of many."""
    rng = np.random.default_rng(91 + O.codec_id(codec))
    K = 1024
    w = np.concatenate([c + rng.standard_normal((16, K)) for c in (1000.0, 300.0, 100.0, 30.0, 5.0)] +
                       [np.where(np.arange(K) // 64 % 2, 1000.0, 0.0) + rng.standard_normal((16, K))])
    w = torch.from_numpy(w.astype(np.float32))
    for im in (None, torch.ones(K), torch.from_numpy((10.0 ** rng.uniform(-6, 0, K)).astype(np.float32))):
        host = kq.quantize(w, codec, im)[0].numpy()
        for dev in _device_bytes(kq, w, codec, im):
            bad = np.argwhere((dev != host).any(axis=1)).ravel().tolist()
            assert not bad, bad


@pytest.mark.parametrize("codec", ["q2_k", "q4_k", "q5_k"])
def test_device_encoder_fit_up_to_the_ends_of_the_bound(kq, codec):
    """Rows whose ranges run up to the largest and down to the smallest for which candidates are ruled out by a bound: the
    bound's own products must hold them.  Weights times 2^s with importance times 2^(-5 s / 3), which keeps every product of the
    scales' own fit in range, have the same scale bytes: the host's at s = 0 (where the f16 factors behind them overflow, the
    quotients that give the levels are not finite, and host and device convert those differently).  And without importance all
    bytes are the host's as far as the factors stay finite."""
    rng = np.random.default_rng(61 + O.codec_id(codec))
    K, bpb = 1024, O.geometry(codec)[1]
    scales = slice(0, 16) if codec == "q2_k" else slice(4, 16)
    w = torch.from_numpy(np.concatenate([rng.random((12, K)), 2 * rng.random((12, K)) - 1, np.clip(rng.standard_normal((8, K)) / 4, -1, 1),
                                         rng.integers(0, 9, (4, K)) / 8]).astype(np.float32))
    for im in (np.ones(K), rng.random(K), 10.0 ** rng.uniform(-6, 0, K)):
        im = torch.from_numpy(im.astype(np.float32))
        host = kq.quantize(w, codec, im)[0].numpy().reshape(len(w), -1, bpb)
        for s in (-27, -12, 15, 18, 21, 24, 27, 30):
            for dev in _device_bytes(kq, w * 2.0 ** s, codec, im * 2.0 ** (-5 * s // 3)):
                bad = np.argwhere((dev.reshape(host.shape)[:, :, scales] != host[:, :, scales]).any(axis=(1, 2))).ravel().tolist()
                assert not bad, (s, bad)
    for s in range(14, {"q2_k": 21, "q4_k": 25, "q5_k": 26}[codec] + 1):  # rows from 0: the minima stay finite
        big = w[:12] * 2.0 ** s
        for dev in _device_bytes(kq, big, codec, None):
            assert np.array_equal(dev, kq.quantize(big, codec)[0].numpy()), s
