"""GPU parity of the matmul between the skinny kernels and the tile GEMMs (9 ... 512 activation rows) at the places where
its tiling can go wrong: one weight row and one step, a ragged last tile, K ending inside a step, several rounds of
persistent workgroups, steps cut over workgroups (also under graph replay), one to four blocks of activation rows."""
import pytest
import torch

import oracle_lib as O
from gpu_util import dev_to_bits, make_x, rel_l2, wire_to_dev

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def kq():
    import kq as _kq
    return _kq


@pytest.fixture
def mid(kq):
    import ctypes
    f = kq._load().kq_set_gemm_tile_rows
    f.argtypes = [ctypes.c_int]
    f(32)
    yield kq
    f(0)


def all_codecs():
    from kq.codec_geometry import CODEC_GEOMETRY
    return sorted(CODEC_GEOMETRY)


@pytest.mark.parametrize("codec", all_codecs())
def test_mid_rows_edges(mid, codec):
    wpb = mid.CODEC_GEOMETRY[codec][3]
    # (rows, N, K): the least of everything; ragged tile, two row blocks and a K tail; cut steps; several rounds
    shapes = [(9, 8, 256), (33, 1003, 2048 + (wpb if wpb < 256 else 256)), (32, 96, 8192), (12, 8205, 512)]
    for i, (M, N, K) in enumerate(shapes):
        dtype = "bfloat16" if i % 2 == 0 else "float16"
        wire = O.synth_wire(codec, N * K // wpb, seed=40 + i).reshape(N, -1)
        xb, xt = make_x((M, K), dtype, seed=50 + i)
        got = dev_to_bits(mid.quantized_matmul(xt, wire_to_dev(wire), None, codec))
        err = rel_l2(got, O.qmm(xb, wire, codec, True, dtype), dtype)
        assert err <= 1e-3, (codec, M, N, K, err)


@pytest.mark.parametrize("M", [31, 64, 65, 128])
def test_mid_row_blocks(mid, M):
    N, K = 264, 1024
    wire = O.synth_wire("q4_k", N * K // 256, seed=3).reshape(N, -1)
    xb, xt = make_x((M, K), "bfloat16", seed=4)
    got = dev_to_bits(mid.quantized_matmul(xt, wire_to_dev(wire), None, "q4_k"))
    assert rel_l2(got, O.qmm(xb, wire, "q4_k", True, "bfloat16"), "bfloat16") <= 1e-3


@pytest.mark.parametrize("codec,M", [("iq4_xs", 129), ("q2_k", 333), ("q8_0", 333), ("mxfp4", 512), ("iq3_s", 511),
                                     ("q6_k", 192), ("q4_k", 129)])
def test_mid_many_row_blocks_as_routed(kq, codec, M):
    """Five to sixteen blocks of activation rows on a narrow matrix, by the dispatch's own rule: a ragged tile, cut steps."""
    N, K = 136, 8192
    wpb = kq.CODEC_GEOMETRY[codec][3]
    wire = O.synth_wire(codec, N * K // wpb, seed=6).reshape(N, -1)
    xb, xt = make_x((M, K), "bfloat16", seed=7)
    got = dev_to_bits(kq.quantized_matmul(xt, wire_to_dev(wire), None, codec))
    assert rel_l2(got, O.qmm(xb, wire, codec, True, "bfloat16"), "bfloat16") <= 1e-3


def test_mid_cut_steps_replay(mid):
    """The arrival counters are set anew by every call: replays of a captured call on changing inputs equal eager calls."""
    N, K, M = 512, 12288, 17
    w = wire_to_dev(O.synth_wire("q6_k", N * K // 256, seed=5).reshape(N, -1))
    xs = [make_x((M, K), "bfloat16", seed=60 + i)[1] for i in range(4)]
    want = [mid.quantized_matmul(x, w, None, "q6_k") for x in xs]
    buf = xs[0].clone()
    side = torch.cuda.Stream()
    with torch.cuda.stream(side):
        mid.quantized_matmul(buf, w, None, "q6_k")
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        out = mid.quantized_matmul(buf, w, None, "q6_k")
    for r in range(8):
        buf.copy_(xs[r % 4])
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want[r % 4]), r


@pytest.mark.parametrize("codec", ["q4_1", "q5_1", "q2_k"])
def test_mid_small_f16_rows_keep_their_sums(mid, codec):
    """f16 activations of about 2^-14 under weights with a large block minimum: the sums that multiply the minimum are two
    f16 terms and need the row's power of two.  One rounding of the result to f16 is at most 2^-11 of it; unscaled sums
    (granularity 2^-24) put q4_1 1.8e-3 and q5_1 0.9e-3 off here."""
    import numpy as np
    M, N, K = 16, 64, 1024
    wpb = mid.CODEC_GEOMETRY[codec][3]
    blocks = O.synth_wire(codec, N * K // wpb, seed=8).reshape(N * K // wpb, -1)
    # codes and minima that nearly cancel
    d, m = (np.array([v], np.float16).view(np.uint8) for v in {"q4_1": (16, -128), "q5_1": (16, -256), "q2_k": (64, 96)}[codec])
    if codec == "q2_k":  # d and dmin end the block; 4-bit scales and minima of their own
        blocks[:, -4:-2], blocks[:, -2:] = d, m
    else:
        blocks[:, 0:2], blocks[:, 2:4] = d, m
    wire = blocks.reshape(N, -1)
    xb, xt = make_x((M, K), "float16", seed=9, scale=2.0**-14)
    got = dev_to_bits(mid.quantized_matmul(xt, wire_to_dev(wire), None, codec))
    assert rel_l2(got, O.qmm(xb, wire, codec, True, "float16"), "float16") <= 2.0**-11


def wide_rows_case(codec, M, K, N, seed):
    """Weights whose first block is zero in every row, and bf16 activations with rows of a range beyond f16's: a mask's value
    over the zero block beside ordinary ones, one large value beside tiny ones, half of the row large."""
    wpb = O.geometry(codec)[0]
    wire = O.synth_wire(codec, N * K // wpb, seed=seed).reshape(N, K // wpb, -1)
    wire[:, 0] = 0
    x = torch.randn((M, K), generator=torch.Generator().manual_seed(seed + 1))
    x[3 % M, 1] = -3.0e38
    x[M - 1, :wpb] = 1e30
    x[M - 1, wpb:] *= 1e-12
    x[M // 2, wpb - 1] = 7e9
    x[M // 2, wpb:] *= 1e-3
    xt = x.to(torch.bfloat16)
    return wire.reshape(N, -1), xt.view(torch.int16).numpy().view("uint16"), xt.cuda()


def row_errors(got, want):
    """Largest relative 2-norm error of a row, bf16 bit patterns."""
    import numpy as np
    f = [(b.astype(np.uint32) << 16).view(np.float32).astype(np.float64) for b in (got, want)]
    return np.max(np.linalg.norm(f[0] - f[1], axis=1) / np.linalg.norm(f[1], axis=1))


@pytest.mark.parametrize("codec", all_codecs())
def test_mid_rows_of_wide_range(mid, codec):
    """Both blocks of rows, K with a tail where the codec has one, steps cut over workgroups: every row on its own within two
    roundings to bf16 (2^-9 each, the reference's and the kernel's)."""
    wpb = mid.CODEC_GEOMETRY[codec][3]
    for M, N, K in ((9, 40, 512), (40, 72, 1024 + wpb), (33, 64, 8192)):
        wire, xb, xt = wide_rows_case(codec, M, K, N, seed=70 + M)
        got = dev_to_bits(mid.quantized_matmul(xt, wire_to_dev(wire), None, codec))
        err = row_errors(got, O.qmm(xb, wire, codec, True, "bfloat16"))
        assert err <= 2.0**-8, (codec, M, N, K, err)


TALL = ["q8_0", "q4_0", "iq4_nl", "q5_0", "q4_1", "q5_1", "mxfp4", "nvfp4", "iq2_xxs", "iq2_xs", "iq2_s", "iq3_xxs", "iq3_s",
        "iq1_s", "iq1_m"]


@pytest.fixture(params=[1024, 1025])
def tall(request):
    import ctypes
    import kq
    f = kq._load().kq_set_gemm_tile_rows
    f.argtypes = [ctypes.c_int]
    f(request.param)
    yield kq
    f(0)


@pytest.mark.parametrize("codec", TALL)
def test_tall_tiles_rows_of_wide_range(tall, codec):
    """Tall-tile calls that fill less than three quarters of the chip: rows beyond f16's range are done again."""
    M, N, K = 160, 264, 1024
    wire, xb, xt = wide_rows_case(codec, M, K, N, seed=90)
    got = dev_to_bits(tall.quantized_matmul(xt, wire_to_dev(wire), None, codec))
    err = row_errors(got, O.qmm(xb, wire, codec, True, "bfloat16"))
    assert err <= 2.0**-8, (codec, err)


@pytest.mark.parametrize("dtype", ["bfloat16", "float16"])
@pytest.mark.parametrize("codec,scale", [("q8_0", 600), ("iq4_nl", 600), ("q4_0", 9000), ("q5_0", 5000), ("q4_1", 5000),
                                         ("q5_1", 3000)])
def test_tall_tiles_weights_beyond_f16(tall, codec, scale, dtype):
    """Block scales whose products with the codes pass 65504, in two weight rows: those columns are done again."""
    import numpy as np
    M, N, K = 130, 264, 512
    wire = O.synth_wire(codec, N * K // 32, seed=95).reshape(N, K // 32, -1)
    wire[[37, 263], :, 0:2] = np.array([scale], np.float16).view(np.uint8)
    wire = wire.reshape(N, -1)
    xb, xt = make_x((M, K), dtype, seed=96, scale=2.0**-6)
    got, want = dev_to_bits(tall.quantized_matmul(xt, wire_to_dev(wire), None, codec)), O.qmm(xb, wire, codec, True, dtype)
    for cols in ([37, 263], [i for i in range(N) if i not in (37, 263)]):
        assert rel_l2(got[:, cols], want[:, cols], dtype) <= 1e-3, (codec, cols[:2])


@pytest.mark.parametrize("dtype", ["bfloat16", "float16"])
def test_tall_tiles_fp4_blocks_far_apart(tall, dtype):
    """mxfp4 blocks of one 64-weight step whose exponents differ by 40, under activations that are zero over the large one; a
    weight row with empty blocks of the smallest exponent beside it."""
    M, N, K = 130, 264, 512
    wire = O.synth_wire("mxfp4", N * K // 32, seed=97).reshape(N, K // 32, 17)
    wire[5, 0::2, 0], wire[5, 1::2, 0] = 150, 110
    wire[6, 0::2] = 0
    xb, xt = make_x((M, K), dtype, seed=98)
    xt = xt.clone()
    xt.view(M, K // 32, 32)[:, 0::2] = 0
    xb = dev_to_bits(xt)
    wire = wire.reshape(N, -1)
    got, want = dev_to_bits(tall.quantized_matmul(xt, wire_to_dev(wire), None, "mxfp4")), O.qmm(xb, wire, "mxfp4", True, dtype)
    for cols in ([5], [6], [i for i in range(N) if i not in (5, 6)]):
        assert rel_l2(got[:, cols], want[:, cols], dtype) <= 1e-3, cols[:2]


@pytest.mark.parametrize("codec,M,N,K", [("iq4_xs", 140, 32776, 256), ("q3_k", 129, 32768, 256), ("q8_0", 333, 13320, 288)])
def test_streamed_where_the_tall_tiles_cannot(kq, codec, M, N, K):
    """As routed: as many tiles as the tall-tile GEMMs want, but fewer rows or another K than theirs accept."""
    wire = O.synth_wire(codec, N * K // kq.CODEC_GEOMETRY[codec][3], seed=11).reshape(N, -1)
    xb, xt = make_x((M, K), "bfloat16", seed=12)
    got = dev_to_bits(kq.quantized_matmul(xt, wire_to_dev(wire), None, codec))
    assert rel_l2(got, O.qmm(xb, wire, codec, True, "bfloat16"), "bfloat16") <= 1e-3


@pytest.mark.parametrize("codec,M,tile", [("q8_0", 40, 32), ("mxfp4", 160, 1025), ("iq3_s", 160, 1024)])
def test_wide_rows_under_replay(kq, codec, M, tile):
    """The flags belong to the call's own rows: replays on ordinary and wide rows in turn equal eager calls."""
    import ctypes
    f = kq._load().kq_set_gemm_tile_rows
    f.argtypes = [ctypes.c_int]
    f(tile)
    try:
        wire, _, wide = wide_rows_case(codec, M, 1024, 264, seed=13)
        w = wire_to_dev(wire)
        xs = [make_x((M, 1024), "bfloat16", seed=14)[1], wide, make_x((M, 1024), "bfloat16", seed=15)[1], wide.flip(0).contiguous()]
        want = [kq.quantized_matmul(x, w, None, codec) for x in xs]
        buf = xs[0].clone()
        torch.cuda.synchronize()
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g):
            out = kq.quantized_matmul(buf, w, None, codec)
        for r in range(8):
            buf.copy_(xs[r % 4])
            g.replay()
            torch.cuda.synchronize()
            assert torch.equal(out, want[r % 4]), r
    finally:
        f(0)
