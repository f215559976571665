"""GPU parity of the one-launch gather_qmm of short contractions (K of one or two 256-weight steps, few rows per expert):
every codec, tiles of weight rows that end inside the matrix, experts without entries, with one row, with more than the 32 rows
of a round and more rounds than workgroups, ids outside the stack, rows of very different size, rows of wide range, infinities,
strided stacks."""
import numpy as np
import pytest
import torch

import kq
import oracle_lib as O
from gpu_util import bits_to_dev, dev_to_bits, rel_l2, wire_to_dev
from test_gpu_moe import TOL, _idx_dev, _stack

pytestmark = pytest.mark.gpu
CODECS = sorted(kq.CODEC_GEOMETRY)


def _case(codec, E, N, K, B, M, L, dtype, ids, seed):
    w = _stack(codec, E, N, K, seed=seed)
    rng = np.random.default_rng(seed + 1)
    lhs = rng.integers(0, L, B)
    x = rng.standard_normal((L, M, K)) * 10.0 ** rng.uniform(-3, 3 if dtype == "bfloat16" else 0, (L, M, 1))
    xb = O.f32_to_bits(x.astype(np.float32), dtype)
    return w, lhs, xb, bits_to_dev(xb, dtype)


def _per_row(got, want, dtype):
    """Largest relative error of a row: rows differ in size by powers of ten."""
    g, w = got.reshape(-1, got.shape[-1]), want.reshape(-1, want.shape[-1])
    return max(rel_l2(a, b, dtype) for a, b in zip(g, w))


# a row of 24 ... 300 bf16 / f16 results: each off by half a unit in the last place at most beside sums in another order
ROW_TOL = {"bfloat16": 2.0 ** -8, "float16": 2.0 ** -11}


@pytest.mark.parametrize("codec", CODECS)
@pytest.mark.parametrize("N,K,B,M,dtype", [(24, 256, 23, 1, "bfloat16"), (72, 512, 30, 3, "float16"), (136, 512, 9, 2, "bfloat16"),
                                           (296, 256, 40, 5, "bfloat16"), (40, 512, 22, 70, "float16")])
def test_few_rows_per_expert(codec, N, K, B, M, dtype):
    E = 11
    rng = np.random.default_rng(77)
    rhs = rng.integers(0, E - 2, B)  # two experts without entries
    rhs[0] = E - 1
    w, lhs, xb, xt = _case(codec, E, N, K, B, M, 7, dtype, rhs, 501)
    got = dev_to_bits(kq.gather_qmm(xt, wire_to_dev(w), None, codec, lhs_indices=_idx_dev(lhs), rhs_indices=_idx_dev(rhs)))
    want = O.gather_qmm(xb, w, codec, lhs, rhs, True, dtype)
    assert rel_l2(got, want, dtype) <= TOL, codec
    assert _per_row(got, want, dtype) <= ROW_TOL[dtype], codec


@pytest.mark.parametrize("codec", ["q4_k", "q8_0", "iq4_xs", "iq2_xs"])
@pytest.mark.parametrize("B,M", [(1024, 1), (200, 7), (33, 1)])
def test_most_entries_on_one_expert(codec, B, M):
    E, N, K, dtype = 64, 40, 512, "bfloat16"
    rng = np.random.default_rng(78)
    rhs = np.where(rng.random(B) < 0.95, 5, rng.integers(0, E, B))
    w, lhs, xb, xt = _case(codec, E, N, K, B, M, 9, dtype, rhs, 511)
    got = dev_to_bits(kq.gather_qmm(xt, wire_to_dev(w), None, codec, lhs_indices=_idx_dev(lhs), rhs_indices=_idx_dev(rhs)))
    want = O.gather_qmm(xb, w, codec, lhs, rhs, True, dtype)
    assert _per_row(got, want, dtype) <= ROW_TOL[dtype], codec


@pytest.mark.parametrize("transpose", [True, False])
@pytest.mark.parametrize("E,B,M", [(1, 256, 1), (3, 96, 8), (64, 1024, 8), (300, 1000, 1), (511, 1024, 5), (700, 1024, 7), (8, 17, 120)])
@pytest.mark.parametrize("spread", ["one", "two", "half", "ramp", "all but one", "outside"])
def test_rounds_that_experts_leave_over(E, B, M, spread, transpose):
    """Experts with more rows than their workgroups do: every row is done, once (the output starts as NaN), whoever takes it."""
    N, K = (64, 256) if transpose else (128, 32)
    rng = np.random.default_rng(E + B)
    rhs = {"one": np.full(B, E // 2), "two": np.where(np.arange(B) % 3 == 0, 0, E - 1),
           "half": np.where(np.arange(B) % 2 == 0, E // 3, rng.integers(0, E, B)),
           "ramp": np.sort((rng.random(B) ** 3 * E).astype(np.int64)), "all but one": np.arange(B) % max(E - 1, 1),
           "outside": np.where(rng.random(B) < 0.5, E + 5, E - 1)}[spread]
    w = _stack("q8_0", E, *((N, K) if transpose else (K, N)), seed=541)
    lhs = rng.integers(0, 9, B)
    xb = O.f32_to_bits(rng.standard_normal((9, M, K)).astype(np.float32), "bfloat16")
    xt, wd, li, ri = bits_to_dev(xb, "bfloat16"), wire_to_dev(w), _idx_dev(lhs).to(torch.int32), _idx_dev(rhs).to(torch.int32)
    out = torch.full((B, M, N), float("nan"), dtype=torch.bfloat16, device="cuda")
    assert kq._load().kq_gather_qmm(xt.data_ptr(), wd.data_ptr(), li.data_ptr(), ri.data_ptr(), out.data_ptr(), B, M, E, N, K, M * K,
                                    wd.stride(0), int(transpose), 0, O.codec_id("q8_0"), kq._DT[torch.bfloat16], None, 0, None) == 0
    torch.cuda.synchronize()
    inside = rhs < E
    assert bool(out[torch.from_numpy(~inside).cuda()].isnan().all())
    want = O.bits_to_f32(xb, "bfloat16").astype(np.float64)[lhs[inside]]
    mats = O.dequantize(w.reshape(-1, w.shape[-1]), "q8_0").reshape(E, -1, K if transpose else N).astype(np.float64)
    mats = mats.transpose(0, 2, 1) if transpose else mats
    want = np.stack([x @ mats[e] for x, e in zip(want, rhs[inside])])
    got = out[torch.from_numpy(inside).cuda()].float().cpu().numpy().astype(np.float64)
    err = np.linalg.norm(got - want, axis=-1) / np.linalg.norm(want, axis=-1)
    assert err.max() <= ROW_TOL["bfloat16"]


@pytest.mark.parametrize("codec", ["q6_k", "q8_0"])
def test_strided_stack_and_repeated_replays(codec):
    """Every second expert of a larger stack; the same call captured and replayed with other activations."""
    E, N, K, B, dtype = 6, 48, 512, 24, "bfloat16"
    rhs = np.arange(B) % E
    w, lhs, xb, xt = _case(codec, 2 * E, N, K, B, 2, 5, dtype, rhs, 521)
    wd, li, ri = wire_to_dev(w)[::2], _idx_dev(lhs), _idx_dev(rhs)
    kq.gather_qmm(xt, wd, None, codec, lhs_indices=li, rhs_indices=ri)
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        y = kq.gather_qmm(xt, wd, None, codec, lhs_indices=li, rhs_indices=ri)
    for k in range(3):
        bits = O.f32_to_bits(np.random.default_rng(530 + k).standard_normal((5, 2, K)).astype(np.float32), dtype)
        xt.copy_(bits_to_dev(bits, dtype))
        g.replay()
        torch.cuda.synchronize()
        assert rel_l2(dev_to_bits(y), O.gather_qmm(bits, w[::2], codec, lhs, rhs, True, dtype), dtype) <= TOL


def _zero_first_weights(w, codec):
    """The first weights of every row made zero: the sub-block's scale (and minimum) inside the first block, or the whole of it."""
    wpb, bpb = O.geometry(codec)
    b = w.reshape(-1, w.shape[-1] // bpb, bpb)[:, 0]
    if codec == "q2_k":
        b[:, 0] = 0
    elif codec == "q3_k":  # six bits less 32
        b[:, 96] &= 0xf0
        b[:, 104] = (b[:, 104] & 0xfc) | 2
    elif codec in ("q4_k", "q5_k"):
        b[:, [4, 8]] &= 0xc0
    elif codec == "q6_k":
        b[:, 192] = 0
    elif codec == "nvfp4":
        b[:, 0] = 0
    elif codec == "iq4_xs":  # six bits less 32
        b[:, 4] &= 0xf0
        b[:, 2] = (b[:, 2] & 0xfc) | 2
    else:
        b[:] = 0
    rows = O.dequantize(w.reshape(-1, w.shape[-1]), codec).reshape(-1, w.shape[-1] // bpb * wpb)
    assert not rows[:, :16].any()


@pytest.mark.parametrize("codec", CODECS)
@pytest.mark.parametrize("K,B,M", [(256, 30, 1), (512, 12, 9)])
def test_rows_of_wide_range(codec, K, B, M):
    """Large values on zero weights beside small ones that are the result: every row on its own; with and without a workspace."""
    if O.geometry(codec)[0] == 256 and K == 256 and codec.startswith("iq") and codec != "iq4_xs":
        pytest.skip("zero weights of this codec fill a step")
    E, N, L, dtype = 5, 136, 6, "bfloat16"
    w = _stack(codec, E, N, K, seed=561)
    _zero_first_weights(w, codec)
    rng = np.random.default_rng(562)
    x = rng.standard_normal((L, M, K)).astype(np.float32)
    x[0, :, 3], x[1, 0, 0], x[2, :, 1] = -3e38, 7e12, 1e30
    x[2, :, 16:] *= 1e-12
    x[3, M - 1] *= 1e-35
    xb = O.f32_to_bits(x, dtype)
    lhs, rhs = rng.integers(0, L, B), rng.integers(0, E, B)
    xt, wd, li, ri = bits_to_dev(xb, dtype), wire_to_dev(w), _idx_dev(lhs).to(torch.int32), _idx_dev(rhs).to(torch.int32)
    want = O.gather_qmm(xb, w, codec, lhs, rhs, True, dtype)
    got = dev_to_bits(kq.gather_qmm(xt, wd, None, codec, lhs_indices=li, rhs_indices=ri))
    assert _per_row(got, want, dtype) <= ROW_TOL[dtype], codec
    out = torch.zeros((B, M, N), dtype=torch.bfloat16, device="cuda")
    assert kq._load().kq_gather_qmm(xt.data_ptr(), wd.data_ptr(), li.data_ptr(), ri.data_ptr(), out.data_ptr(), B, M, E, N, K, M * K,
                                    wd.stride(0), 1, 0, O.codec_id(codec), kq._DT[torch.bfloat16], None, 0, None) == 0
    torch.cuda.synchronize()
    assert _per_row(dev_to_bits(out), want, dtype) <= ROW_TOL[dtype], codec


@pytest.mark.parametrize("dtype", ["bfloat16", "float16"])
@pytest.mark.parametrize("codec", ["q2_k", "q3_k", "q4_k", "q8_0", "nvfp4", "iq2_xs"])
def test_rows_with_an_infinity(codec, dtype):
    """Infinite where the products say so; the other rows of the round are the ordinary ones."""
    E, N, K, B, M, L = 5, 72, 512, 20, 2, 6
    w, lhs, xb, _ = _case(codec, E, N, K, B, M, L, dtype, None, 571)
    rhs = np.arange(B) % E
    xb = xb.copy()
    xb[2, 1, 300] = 0x7f80 if dtype == "bfloat16" else 0x7c00
    xb[4, 0, 7] = 0xff80 if dtype == "bfloat16" else 0xfc00
    got, want = (O.bits_to_f32(b, dtype) for b in (
        dev_to_bits(kq.gather_qmm(bits_to_dev(xb, dtype), wire_to_dev(w), None, codec, lhs_indices=_idx_dev(lhs), rhs_indices=_idx_dev(rhs))),
        O.gather_qmm(xb, w, codec, lhs, rhs, True, dtype)))
    fin = np.isfinite(want)
    assert np.array_equal(got[~fin], want[~fin], equal_nan=True) and np.isfinite(got[fin]).all()
    assert np.linalg.norm(got[fin] - want[fin]) <= ROW_TOL[dtype] * np.linalg.norm(want[fin])


def test_ids_outside_the_stack_write_nothing():
    E, N, K, B, codec, dtype = 5, 40, 256, 20, "q8_0", "bfloat16"
    rhs = np.arange(B) % E
    w, lhs, xb, xt = _case(codec, E, N, K, B, 1, 5, dtype, rhs, 541)
    bad = rhs.copy()
    bad[[3, 17]] = [E, 2 ** 31 - 1]
    out = torch.full((B, 1, N), 7.0, dtype=torch.bfloat16, device="cuda")
    wd, li, ri = wire_to_dev(w), _idx_dev(lhs).to(torch.int32), _idx_dev(bad).to(torch.int32)
    lib = kq._load()
    rc = lib.kq_gather_qmm(xt.data_ptr(), wd.data_ptr(), li.data_ptr(), ri.data_ptr(), out.data_ptr(), B, 1, E, N, K, K,
                           wd.stride(0), 1, 0, O.codec_id(codec), kq._DT[torch.bfloat16], None, 0, None)
    assert rc == 0
    torch.cuda.synchronize()
    want = O.gather_qmm(xb, w, codec, lhs, rhs, True, dtype)
    keep = [i for i in range(B) if i not in (3, 17)]
    assert rel_l2(dev_to_bits(out)[keep], want[keep], dtype) <= TOL
    assert bool((out[[3, 17]] == 7.0).all())


@pytest.mark.parametrize("codec", ["q8_0", "q4_k"])
def test_empty_contraction_and_empty_stack(codec):
    """K = 0: sums of nothing.  No experts: every id is outside the stack and nothing is written, in either orientation."""
    E, N, B, M = 5, 256, 40, 2
    lib, x = kq._load(), torch.ones(B * M * 256, dtype=torch.bfloat16, device="cuda")
    w = torch.zeros(1024, dtype=torch.uint8, device="cuda")
    ids = torch.arange(B, device="cuda", dtype=torch.int32) % E

    def call(out, e, k, transpose):
        rc = lib.kq_gather_qmm(x.data_ptr(), w.data_ptr(), ids.data_ptr(), ids.data_ptr(), out.data_ptr(), B, M, e, N, k, M * k, 0,
                               transpose, 0, O.codec_id(codec), kq._DT[torch.bfloat16], None, 0, None)
        torch.cuda.synchronize()
        return rc

    out = torch.full((B, M, N), 7.0, dtype=torch.bfloat16, device="cuda")
    for transpose in (0, 1):
        assert call(out, 0, 256, transpose) == 0 and bool((out == 7.0).all())
    for transpose in (0, 1):
        out.fill_(7.0)
        assert call(out, E, 0, transpose) == 0 and bool((out == 0.0).all())


@pytest.mark.parametrize("codec", ["q8_0", "q4_k", "q6_k", "iq3_s", "q5_1", "nvfp4"])
@pytest.mark.parametrize("K,M,B,dtype", [(96, 1, 40, "bfloat16"), (130, 3, 31, "float16"), (64, 8, 200, "bfloat16"),
                                         (192, 16, 30, "bfloat16"), (100, 24, 23, "bfloat16"),
                                         (64, 16, 350, "bfloat16"), (40, 24, 180, "float16")])
def test_other_orientation_merges_entries(codec, K, M, B, dtype):
    """transpose=False, entries of one expert in shared tiles: most of them on one expert (several rounds), experts without any,
    rows that cannot be read 16 bytes at a time, a last step of K that is not whole, a last column tile that is not."""
    E, N, L = 11, 768 if codec in ("q4_k", "q6_k", "iq3_s") else 320, 9
    rng = np.random.default_rng(79)
    rhs = np.where(rng.random(B) < 0.7, 4, rng.integers(0, E - 2, B))
    w = _stack(codec, E, K, N, seed=551)  # K wire rows of N weights
    lhs = rng.integers(0, L, B)
    xb = O.f32_to_bits((rng.standard_normal((L, M, K)) * 10.0 ** rng.uniform(-2, 2, (L, M, 1))).astype(np.float32), dtype)
    xt = bits_to_dev(xb, dtype)
    got = dev_to_bits(kq.gather_qmm(xt, wire_to_dev(w), None, codec, lhs_indices=_idx_dev(lhs), rhs_indices=_idx_dev(rhs),
                                    transpose=False))
    want = O.gather_qmm(xb, w, codec, lhs, rhs, False, dtype)
    assert rel_l2(got, want, dtype) <= TOL, codec
    assert _per_row(got, want, dtype) <= ROW_TOL[dtype], codec
