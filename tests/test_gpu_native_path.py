"""The native call path of the ops against the checked Python functions behind it: same bits on the calls it takes, the
function's own conversion or error on the ones it declines, and calls from several threads on streams of their own."""
import threading

import pytest
import torch

import oracle_lib as O
from gpu_util import make_x, wire_to_dev

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def kq():
    import kq as _kq
    return _kq


def wire(codec, rows, K, seed):
    return wire_to_dev(O.synth_wire(codec, rows * K // O.geometry(codec)[0], seed).reshape(rows, -1))


class Spy:
    """The native functions, keeping what each call was answered with."""

    def __init__(self, native):
        self.native, self.answers = native, []

    def __getattr__(self, name):
        f = getattr(self.native, name)

        def call(*args):
            self.answers.append((name, f(*args)))
            return self.answers[-1][1]

        return call


def test_native_ops_take_ordinary_calls_with_the_checked_functions_bits(kq, monkeypatch):
    E, N, K, T, R = 4, 64, 512, 3, 2
    x = make_x((T, K), "bfloat16", 1)[1]
    g, u, d = (wire(c, E * n, k, s).reshape(E, n, -1) for c, n, k, s in (("q4_k", N, K, 2), ("q4_k", N, K, 3), ("q6_k", K, 256, 4)))
    mg, mu = (wire("mxfp4", E * N, K, s).reshape(E, N, -1) for s in (7, 8))
    gb, ub = torch.randn(E, N, device="cuda"), torch.randn(E, N, device="cuda")
    xs, xn = make_x((T, R, 256), "bfloat16", 5)[1], make_x((T, R, K), "float16", 9)[1]
    idx = torch.tensor([[0, 3], [1, 2], [2, 0]], dtype=torch.int32, device="cuda")
    sc = torch.rand(T, R, device="cuda")
    im = torch.rand(512, device="cuda") + 0.1
    lhs, rhs = (torch.tensor(v, dtype=torch.int32, device="cuda") for v in ([2, 0, 1], [3, 1, 1]))
    calls = {
        "quantized_matmul": [(x, g[0], None, "q4_k"), (make_x((5, N), "float16", 6)[1], g[1], None, "q4_k", False)],
        "dequantize": [(g, None, "q4_k"), (d, None, "q6_k", torch.float32), (g, None, "q4_k", torch.bfloat16)],
        "gather_qmm": [(x[:, None], g, None, "q4_k", lhs, rhs), (x[:, None, :64].contiguous(), g, None, "q4_k", lhs, rhs, False)],
        "moe_glu_gather_kq": [(x, g, u, "q4_k", idx, "gelu"), (x, g, u, "q4_k", idx, "silu_limit", 7.0),
                              (x, mg, mu, "mxfp4", idx, "swiglu_clamp", 7.0, gb, ub, 1.702)],
        "gather_qmv_kq": [(xs, d, "q6_k", idx), (xn, mg, "mxfp4", idx, gb)],
        "moe_glu_gather_shexp_kq": [(x, g, u, g[1], u[2], "q4_k", idx)],
        "gather_qmv_mix_ns_kq": [(xs, d, "q6_k", idx, sc)],
        "gather_qmv_mix_kq": [(xs, d, d[1], "q6_k", idx[:, :1].contiguous(), sc)],
        "moe_router_topk": [(torch.randn(T, E + 1, device="cuda"), 2, True),
                            (torch.randn(T, E, device="cuda"), 2, True, False, sc.new_ones(E), sc.new_zeros(E), "sqrtsoftplus", 2.5)],
        "quantize": [(torch.randn(3, 512, device="cuda"), "q5_k"), (torch.randn(3, 512, device="cuda").half(), "q2_k", im)],
    }
    spy = Spy(kq._native)
    monkeypatch.setattr(kq, "_native", spy)
    for name, variants in calls.items():
        for args in variants:
            spy.answers.clear()
            got, want = getattr(kq, name)(*args), kq._checked[name](*args)
            assert len(spy.answers) == 1 and spy.answers[0][1] is not None, name
            got, want = ((v if isinstance(v, tuple) else (v,)) for v in (got, want))
            assert len(got) == len(want), name
            for a, b in zip(got, want):
                assert a.dtype == b.dtype and a.shape == b.shape and torch.equal(a, b), name


def test_declined_calls_convert_or_raise(kq):
    w = wire("q4_k", 64, 512, 7)
    x = torch.randn(2, 512, device="cuda")
    want = kq.quantized_matmul(x.bfloat16(), w, None, "q4_k")
    assert torch.equal(kq.quantized_matmul(x, w, None, "q4_k"), want)                      # f32 is cast
    assert torch.equal(kq.quantized_matmul(x.T.contiguous().T.bfloat16(), w, None, "q4_k"), want)  # strides are packed
    y = kq.quantized_matmul(x.bfloat16().requires_grad_(True), w, None, "q4_k")
    assert y.requires_grad and torch.equal(y.detach(), want)
    for bad, exc in (((x, w, None, "nope"), ValueError), ((x[:, :256], w, None, "q4_k"), ValueError),
                     ((x.cpu(), w.cpu(), None, "q4_k"), RuntimeError), ((x.long(), w, None, "q4_k"), ValueError)):
        with pytest.raises(exc):
            kq.quantized_matmul(*bad)


def test_threads_on_their_own_streams(kq):
    w = wire("q6_k", 512, 4096, 8)
    xs = [make_x((m, 4096), "bfloat16", 20 + m)[1] for m in (1, 9, 33)]
    want = [kq.quantized_matmul(x, w, None, "q6_k") for x in xs]
    torch.cuda.synchronize()
    bad = []

    def work(i):
        s = torch.cuda.Stream()
        with torch.cuda.stream(s):
            outs = [kq.quantized_matmul(xs[i], w, None, "q6_k") for _ in range(40)]
        s.synchronize()
        if not all(torch.equal(o, want[i]) for o in outs):
            bad.append(i)

    ts = [threading.Thread(target=work, args=(i,)) for i in range(3)]
    [t.start() for t in ts]
    [t.join() for t in ts]
    assert not bad
