"""GPU parity of the batched MoE kernel for segments of up to 96 pairs where its tiling can go wrong: segments at the edges of their
blocks of 32 pairs, experts cut into several, ragged slabs, one step of K, f32 slot rows, ids outside
the stack."""
import numpy as np
import pytest
import torch

import kq
import oracle_lib as O
from gpu_util import dev_to_bits, make_x, rel_l2, wire_to_dev
from test_gpu_moe_ext import TOL, _idx_dev, _stack

pytestmark = pytest.mark.gpu
# pairs per expert: full and ragged segments of one, two and three blocks, two and three segments, none
COUNTS = [96, 97, 64, 65, 32, 33, 1, 0, 200, 95, 193, 84]


def takes(codec, idx, E, N, K, glu):
    """The call runs on this kernel."""
    lib = kq._load()
    return lib.kq_moe_segment_rows(idx.shape[0], idx.shape[1], E, N, K, glu, lib.kq_codec_id(codec.encode())) == 96


def routing(counts, R, seed):
    idx = np.random.default_rng(seed).permutation(np.repeat(np.arange(len(counts)), counts))
    return idx[:len(idx) // R * R].reshape(-1, R)


@pytest.mark.parametrize("codec", ["q4_k", "q5_k", "q6_k"])
@pytest.mark.parametrize("N,K,act,dtype", [(456, 256, "silu", "bfloat16"), (584, 512, "gelu", "float16"), (448, 1280, "silu", "float16")])
def test_fused(codec, N, K, act, dtype):
    E, idx = len(COUNTS), routing(COUNTS, 4, 1)
    assert takes(codec, idx, E, N, K, 1)
    w, w2 = _stack(codec, E, N, K, 2), _stack(codec, E, N, K, 3)
    xb, xt = make_x((idx.shape[0], K), dtype, seed=4, scale=0.05)
    got = kq.moe_glu_gather_kq(xt, wire_to_dev(w), wire_to_dev(w2), codec, _idx_dev(idx), act)
    assert rel_l2(dev_to_bits(got), O.moe_glu_gather(xb, w, w2, codec, idx, act, dtype=dtype), dtype) <= TOL


@pytest.mark.parametrize("codec", ["q4_k", "q5_k", "q6_k"])
@pytest.mark.parametrize("N,K,dtype", [(1288, 256, "bfloat16"), (1280, 768, "float16"), (1400, 1280, "bfloat16")])
def test_plain(codec, N, K, dtype):
    E, idx = len(COUNTS), routing(COUNTS, 1, 5)
    assert takes(codec, idx, E, N, K, 0)
    w = _stack(codec, E, N, K, 6)
    xb, xt = make_x((idx.shape[0], 1, K), dtype, seed=7, scale=0.05)
    got = kq.gather_qmv_kq(xt, wire_to_dev(w), codec, _idx_dev(idx))
    one = np.ones(idx.shape, np.float32)
    assert rel_l2(dev_to_bits(got)[:, 0], O.gather_qmv_mix(xb, w, None, codec, None, idx, one, dtype), dtype) <= TOL


def test_mix_and_ids_outside():
    """The down projection's f32 slot rows; a slot whose id is outside the stack adds nothing."""
    codec, E, N, K, S = "q6_k", 4, 2056, 512, 4
    idx = routing([120, 96, 33, 151], S, 8)
    assert takes(codec, idx, E, N, K, 0)
    w = _stack(codec, E, N, K, 9)
    scores = np.random.default_rng(10).uniform(0.05, 1.0, idx.shape).astype(np.float32)
    bad, zeroed = idx.copy(), scores.copy()
    bad[3, 1], zeroed[3, 1] = E, 0.0
    xb, xt = make_x((idx.shape[0], S, K), "bfloat16", seed=11, scale=0.05)
    got = kq.gather_qmv_mix_ns_kq(xt, wire_to_dev(w), codec, _idx_dev(bad), torch.from_numpy(scores).cuda())
    assert rel_l2(dev_to_bits(got), O.gather_qmv_mix(xb, w, None, codec, None, idx, zeroed, "bfloat16"), "bfloat16") <= TOL


@pytest.mark.parametrize("codec", ["q4_k", "q6_k"])
@pytest.mark.parametrize("N,offset", [(1291, 0), (1409, 0), (1288, 1)])  # rows of no whole 16-byte pieces; an output off 16 bytes
def test_results_stored_one_by_one(codec, N, offset):
    """gather_qmm takes any N and any output address: every element of every row, and nothing behind the last one."""
    E, K, idx = len(COUNTS), 256, routing(COUNTS, 1, 12)
    assert takes(codec, idx, E, N, K, 0)
    P = idx.shape[0]
    w = _stack(codec, E, N, K, 13)
    xb, xt = make_x((P, 1, K), "bfloat16", seed=14, scale=0.05)
    wd, lhs, rhs = wire_to_dev(w), torch.arange(P, dtype=torch.int32, device="cuda"), _idx_dev(idx[:, 0]).to(torch.int32)
    buf = torch.full((P * N + 64,), 7.0, dtype=torch.bfloat16, device="cuda")
    lib, c = kq._load(), kq._load().kq_codec_id(codec.encode())
    need = lib.kq_gather_qmm_workspace_size(P, 1, E, N, K, 1, c, 2)
    ws = torch.empty(need + 256, dtype=torch.uint8, device="cuda")
    wp = -ws.data_ptr() % 256 + ws.data_ptr()
    rc = lib.kq_gather_qmm(xt.data_ptr(), wd.data_ptr(), lhs.data_ptr(), rhs.data_ptr(), buf[offset:].data_ptr(), P, 1, E, N, K, K,
                           wd[0].numel(), 1, 0, c, 2, wp, need, torch.cuda.current_stream().cuda_stream)
    assert rc == 0, lib.kq_last_error()
    got = dev_to_bits(buf)
    want = O.gather_qmm(xb, w, codec, np.arange(P), idx[:, 0], True, "bfloat16")
    assert rel_l2(got[offset:offset + P * N].reshape(P, 1, N), want, "bfloat16") <= TOL
    assert (got[:offset] == 0x40e0).all() and (got[offset + P * N:] == 0x40e0).all()


@pytest.mark.parametrize("codec", ["q4_k", "q8_0", "q4_1", "iq4_xs"])  # the last three: the code-level kernel, its sums and pairs
@pytest.mark.parametrize("dtype", ["bfloat16", "float16"])
@pytest.mark.parametrize("T,R,K,glu", [
    (2048, 1, 256, 0),   # the last count of the narrow prologue
    (2049, 1, 256, 0),   # a wave per row from here: one row in the last workgroup
    (1025, 2, 2048, 1),  # the longest such rows, fewer rows than pairs
    (2063, 1, 2304, 0),  # four rows a workgroup, three in the last
    (2731, 3, 256, 0),   # 8193 pairs: the sort counts twice
])
def test_prologue_of_many_pairs(T, R, K, glu, dtype, codec):
    E, N = 5, 40
    idx = np.random.default_rng(20).integers(0, E, (T, R))
    w, w2 = _stack(codec, E, N, K, 21), _stack(codec, E, N, K, 22)
    if glu:
        xb, xt = make_x((T, K), dtype, seed=23, scale=0.05)
        got = dev_to_bits(kq.moe_glu_gather_kq(xt, wire_to_dev(w), wire_to_dev(w2), codec, _idx_dev(idx), "silu"))
        want = O.moe_glu_gather(xb, w, w2, codec, idx, "silu", dtype=dtype)
    else:
        xb, xt = make_x((T * R, 1, K), dtype, seed=23, scale=0.05)
        got = dev_to_bits(kq.gather_qmv_kq(xt, wire_to_dev(w), codec, _idx_dev(idx.reshape(-1, 1))))[:, 0]
        want = O.gather_qmv_mix(xb, w, None, codec, None, idx.reshape(-1, 1), np.ones((T * R, 1), np.float32), dtype)
    assert rel_l2(got, want, dtype) <= TOL
    # the rows at the ends one by one
    assert rel_l2(got[:1], want[:1], dtype) <= 3 * TOL and rel_l2(got[-1:], want[-1:], dtype) <= 3 * TOL
