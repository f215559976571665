"""GPU parity of the one-launch down projection with the routing mix where its tiling can go wrong: one slot of one unit, 32 units,
several rounds of workgroups, the shared slot, ids outside the stack, activations of wide range; and its sums against
those of the kernel without tiles, bit for bit."""
import numpy as np
import pytest
import torch

import kq
import oracle_lib as O
from gpu_util import dev_to_bits, make_x, rel_l2, wire_to_dev
from test_gpu_mid import row_errors
from test_gpu_moe_ext import TOL, _idx_dev, _stack

pytestmark = pytest.mark.gpu
STREAMED = ["q2_k", "q3_k", "q4_k", "q5_k", "q6_k", "iq4_xs", "iq3_s", "iq2_xxs", "q8_0", "iq4_nl", "q4_0", "mxfp4", "nvfp4"]


def case(codec, T, S, E, N, K, seed, shared=False):
    w = _stack(codec, E, N, K, seed)
    rng = np.random.default_rng(seed + 1)
    return (w, _stack(codec, 1, N, K, seed + 2)[0] if shared else None, rng.integers(0, E, (T, S - int(shared))),
            rng.uniform(0.05, 1.0, (T, S)).astype(np.float32))


def run(xt, w, sw, codec, idx, scores):
    sc = torch.from_numpy(scores).cuda()
    if sw is None:
        return kq.gather_qmv_mix_ns_kq(xt, wire_to_dev(w), codec, _idx_dev(idx), sc)
    return kq.gather_qmv_mix_kq(xt, wire_to_dev(w), wire_to_dev(sw), codec, _idx_dev(idx), sc)


@pytest.mark.parametrize("codec", STREAMED)
def test_mix_stream_edges(codec):
    # (tokens, slots, N, K): the least, of the kernel for one token and of the streamed one; 32 units on a ragged 12-row tile; two
    # rounds of 32-row tiles
    for i, (T, S, N, K) in enumerate([(1, 1, 8, 256), (2, 8, 1064, 1024), (9, 3, 1496, 1024), (2, 1, 8, 256)]):
        dtype = ("bfloat16", "float16")[i % 2]
        w, _, idx, scores = case(codec, T, S, 4, N, K, 310 + i)
        xb, xt = make_x((T, S, K), dtype, seed=320 + i, scale=0.05)
        got = dev_to_bits(run(xt, w, None, codec, idx, scores))
        assert rel_l2(got, O.gather_qmv_mix(xb, w, None, codec, None, idx, scores, dtype), dtype) <= TOL, (codec, T, S, N, K)


@pytest.mark.parametrize("codec", ["q6_k", "iq3_s", "q8_0"])
@pytest.mark.parametrize("T", [1, 3, 5])
def test_mix_stream_shared_slot_and_ids_outside(codec, T):
    """An id outside the stack adds nothing, whatever expert 0 (which its loads read) holds; the shared slot stays."""
    S, E, N, K = 5, 3, 264, 768
    w, sw, idx, scores = case(codec, T, S, E, N, K, 330, shared=True)
    xb, xt = make_x((T, S, K), "bfloat16", seed=331, scale=0.05)
    want = O.gather_qmv_mix(xb, w, sw, codec, codec, idx, scores, "bfloat16")
    assert rel_l2(dev_to_bits(run(xt, w, sw, codec, idx, scores)), want, "bfloat16") <= TOL
    bad, zero = idx.copy(), scores.copy()
    bad[:, 1], zero[:, 1] = E, 0.0
    want = O.gather_qmv_mix(xb, w, sw, codec, codec, idx, zero, "bfloat16")
    xt = xt.clone()
    xt[:, 1] = float("inf")
    assert rel_l2(dev_to_bits(run(xt, w, sw, codec, bad, scores)), want, "bfloat16") <= TOL


@pytest.mark.parametrize("codec", STREAMED)
def test_mix_stream_rows_of_wide_range(codec):
    """Large values over zero weights beside tiny ones that are the result: every token within the roundings to bf16 (2^-9 each,
    the reference's and the kernel's)."""
    T, S, E, N, K = 2, 4, 3, 200, 768
    wpb, bpb = O.geometry(codec)
    w, _, idx, scores = case(codec, T, S, E, N, K, 340)
    w.reshape(E, N, K // wpb, bpb)[:, :, 0] = 0
    x = torch.randn((T, S, K), generator=torch.Generator().manual_seed(341))
    x[0, :, 0], x[0, 1] = 1e30, x[0, 1] * 1e-9
    x[1] *= 1e-30
    xt = x.to(torch.bfloat16)
    xb = xt.view(torch.int16).numpy().view("uint16")
    got = dev_to_bits(run(xt.cuda(), w, None, codec, idx, scores))
    assert row_errors(got, O.gather_qmv_mix(xb, w, None, codec, None, idx, scores, "bfloat16")) <= 2.0**-8, codec


def test_mix_stream_tokens_are_independent_and_replay():
    """A token's result does not depend on how many share the launch (tile heights differ; one token alone has the f32 sums of a
    kernel of its own); replays follow the inputs."""
    S, E, N, K = 8, 6, 2048, 768
    w, _, idx, scores = case("q4_k", 8, S, E, N, K, 350)
    _, xt = make_x((8, S, K), "bfloat16", seed=351, scale=0.05)
    wd, sc, ix = wire_to_dev(w), torch.from_numpy(scores).cuda(), _idx_dev(idx).to(torch.int32)
    want = torch.cat([kq.gather_qmv_mix_ns_kq(xt[t:t + 2], wd, "q4_k", ix[t:t + 2], sc[t:t + 2]) for t in range(0, 8, 2)])
    assert torch.equal(kq.gather_qmv_mix_ns_kq(xt, wd, "q4_k", ix, sc), want)
    buf = xt[:1].clone()
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        out = kq.gather_qmv_mix_ns_kq(buf, wd, "q4_k", ix[:1], sc[:1])
    for t in (0, 3, 0):
        buf.copy_(xt[t:t + 1])
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, kq.gather_qmv_mix_ns_kq(buf, wd, "q4_k", ix[:1], sc[:1]))


def c_call(xt, w, sw, codec, idx, scores):
    """The C entry point without a workspace."""
    lib, (T, S, K), (E, N) = kq._load(), xt.shape, w.shape[:2]
    out = torch.full((T, N), float("nan"), dtype=xt.dtype, device="cuda")
    c = lib.kq_codec_id(codec.encode())
    rc = lib.kq_gather_qmv_mix(xt.data_ptr(), w.data_ptr(), None if sw is None else sw.data_ptr(), idx.data_ptr(), scores.data_ptr(),
                               out.data_ptr(), T, S, E, N, K, c, -1 if sw is None else c, 1 if xt.dtype == torch.float16 else 2, None, 0,
                               torch.cuda.current_stream().cuda_stream)
    assert rc == 0, lib.kq_last_error()
    return out


def unaligned(t):
    """A copy that starts at an odd multiple of two bytes: the call runs a workgroup per output element."""
    buf = torch.empty(t.numel() + 1, dtype=t.dtype, device="cuda")
    buf[1:].copy_(t.reshape(-1))
    return buf[1:].view(t.shape)


# (tokens, slots, N, K, shared slot): the least; 32 units; three long slots; the shared slot; 32 slots; a slot of 32 units
@pytest.mark.parametrize("codec", STREAMED)
@pytest.mark.parametrize("T,S,N,K,shared", [(1, 1, 8, 256, False), (1, 8, 1064, 1024, False), (1, 3, 264, 2560, False),
                                            (3, 5, 264, 768, True), (1, 32, 40, 256, False), (1, 1, 24, 8192, False)])
def test_sums_are_those_of_the_kernel_without_tiles(codec, T, S, N, K, shared):
    """f32 products of the activations as they are, in one order: activations with a mean, whose sums cancel where weights are
    multiplied with an offset."""
    w, sw, idx, scores = case(codec, T, S, 3, N, K, 360 + S, shared)
    idx[0, 0] = 2  # the stack's last matrix
    dtype = ("bfloat16", "float16")[S % 2]
    x = (torch.randn((T, S, K), generator=torch.Generator().manual_seed(361)) * 0.1 + 1.0).to(getattr(torch, dtype)).cuda()
    args = (wire_to_dev(w), None if sw is None else wire_to_dev(sw), codec, _idx_dev(idx).to(torch.int32), torch.from_numpy(scores).cuda())
    got, want = c_call(x, *args), c_call(unaligned(x), *args)
    assert torch.isfinite(want).all()
    assert torch.equal(got.view(torch.int16), want.view(torch.int16)), (codec, float((got != want).float().mean()))


@pytest.mark.parametrize("codec,S,N,K", [(c, 8, 40, 2048) for c in STREAMED] + [
    ("q4_k", 2, 16, 4096), ("q8_0", 5, 24, 3584), ("q6_k", 13, 8, 2304),  # as many slots under way as the LDS holds, and one
    ("mxfp4", 4, 48, 2880), ("q8_0", 4, 16, 2880), ("iq4_nl", 9, 24, 736), ("q4_0", 3, 8, 32), ("nvfp4", 3, 16, 1728),
    ("q4_k", 3, 16, 8192), ("q5_1", 3, 16, 736)])  # (the kernel without tiles)
def test_one_token_needs_no_workspace(codec, S, N, K):
    """Any row length, by the C entry point with a null workspace."""
    w, _, idx, scores = case(codec, 1, S, 3, N, K, 380)
    idx[0, -1] = 2
    xb, xt = make_x((1, S, K), "bfloat16", seed=381, scale=0.05)
    args = (wire_to_dev(w), None, codec, _idx_dev(idx).to(torch.int32), torch.from_numpy(scores).cuda())
    got = c_call(xt, *args)
    assert rel_l2(dev_to_bits(got), O.gather_qmv_mix(xb, w, None, codec, None, idx, scores, "bfloat16"), "bfloat16") <= TOL
    assert torch.equal(got.view(torch.int16), c_call(unaligned(xt), *args).view(torch.int16))


@pytest.mark.parametrize("codec", STREAMED)
def test_one_token_of_long_slots_and_wide_range(codec):
    """A large value over a zero weight beside tiny ones that are the result, 64 units a token: within the roundings to bf16."""
    S, E, N, K = 8, 3, 40, 2048
    wpb, bpb = O.geometry(codec)
    w, _, idx, scores = case(codec, 1, S, E, N, K, 390)
    w.reshape(E, N, K // wpb, bpb)[:, :, 0] = 0
    x = torch.randn((1, S, K), generator=torch.Generator().manual_seed(391)) * 1e-12
    x[0, :, 0] = 1e30
    xt = x.to(torch.bfloat16)
    got = dev_to_bits(run(xt.cuda(), w, None, codec, idx, scores))
    want = O.gather_qmv_mix(xt.view(torch.int16).numpy().view("uint16"), w, None, codec, None, idx, scores, "bfloat16")
    assert row_errors(got, want) <= 2.0**-8, codec


@pytest.mark.parametrize("codec", ["q4_k", "q6_k", "q8_0"])
def test_infinite_activation(codec):
    """An infinity times a weight is an infinity of the weight's sign, as in the kernel without tiles."""
    T, S, E, N, K = 1, 4, 3, 72, 512
    w, _, idx, scores = case(codec, T, S, E, N, K, 370)
    x = (torch.randn((T, S, K), generator=torch.Generator().manual_seed(371)) * 0.1).to(torch.float16).cuda()
    x[0, 1, 77] = float("inf")
    args = (wire_to_dev(w), None, codec, _idx_dev(idx).to(torch.int32), torch.from_numpy(scores).cuda())
    got, want = c_call(x, *args), c_call(unaligned(x), *args)
    assert torch.isinf(want).any()
    assert torch.equal(got.nan_to_num(7.0, 9.0, -9.0), want.nan_to_num(7.0, 9.0, -9.0))
