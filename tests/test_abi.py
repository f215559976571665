"""CPU-side checks of the C ABI: libkq.so loads, exports every symbol include/kq.h declares, and
the registry / host-only entry points behave (no GPU compute is called)."""
import ctypes as C
import os
import re
import subprocess
import sys
import warnings

import pytest
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LIB = os.path.join(ROOT, "mlx-kquant_amd", "lib", "libkq.so")


@pytest.fixture(scope="module")
def lib():
    if not os.path.exists(LIB):
        subprocess.check_call([sys.executable, os.path.join(ROOT, "mlx-kquant_amd", "build.py")])
    return C.CDLL(LIB)


def _declared_symbols():
    text = open(os.path.join(ROOT, "include", "kq.h")).read()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    return sorted(set(re.findall(r"\b(kq_[a-z0-9_]+)\s*\(", text)))


def test_header_symbols_exported(lib):
    names = _declared_symbols()
    assert len(names) >= 14
    for n in names:
        assert hasattr(lib, n), n


def test_registry_matches_python_geometry(lib):
    sys.path.insert(0, os.path.join(ROOT, "mlx-kquant_amd"))
    import kq

    assert kq.codecs() == list(kq.CODEC_GEOMETRY) or sorted(kq.codecs()) == sorted(kq.CODEC_GEOMETRY)
    import oracle_lib as O

    assert kq.codecs() == O.ALL_CODECS
    for name in kq.codecs():
        _, _, bpb, wpb = kq.codec_geometry.geometry(name)
        assert (wpb, bpb) == O.geometry(name)
        assert kq.codec_has_matmul(name) and kq.codec_has_moe_glu(name)
    assert not kq.codec_has_matmul("nope") and not kq.codec_has_moe_glu("nope")
    assert kq.bytes_per_row("q4_k", 4096) == 2304 and kq.bytes_per_row("q6_k", 14336) == 11760
    assert kq.weights_per_row("mxfp4", 1530) == 2880
    with pytest.raises(ValueError):
        kq.bytes_per_row("q4_k", 100)


def test_error_codes_without_gpu(lib):
    lib.kq_last_error.restype = C.c_char_p
    lib.kq_dequantize.argtypes = [C.c_void_p, C.c_void_p, C.c_uint64, C.c_int, C.c_int, C.c_void_p]
    assert lib.kq_dequantize(None, None, 256, 99, 0, None) == -1
    assert b"codec" in lib.kq_last_error()
    assert lib.kq_dequantize(None, None, 100, 2, 0, None) == -1  # not a whole number of blocks
    assert lib.kq_dequantize(None, None, 0, 2, 0, None) == 0  # empty tensor is a no-op
    assert lib.kq_codec_id(b"q4_k") == 2 and lib.kq_codec_id(b"zzz") == -1


def test_python_front_end_refuses_cpu_tensors():
    sys.path.insert(0, os.path.join(ROOT, "mlx-kquant_amd"))
    import torch

    import kq

    w = torch.zeros((4, 144), dtype=torch.uint8)
    with pytest.raises(RuntimeError):
        kq.dequantize(w, None, "q4_k")
    with pytest.raises(RuntimeError):
        kq.quantized_matmul(torch.zeros((1, 256), dtype=torch.float16), w, None, "q4_k")
    with pytest.raises(ValueError):
        kq.quantized_matmul(torch.zeros((1, 128), dtype=torch.float16), w, None, "q4_k")


@pytest.mark.parametrize("content", [None, b"not a shared library"])
def test_ops_do_without_the_native_call_path(monkeypatch, tmp_path, content):
    """_kqhost.so missing or unloadable: one warning, every native function declines, and an op's own checks answer."""
    import kq

    path = tmp_path / "_kqhost.so"
    if content is not None:
        path.write_bytes(content)
    monkeypatch.setattr(kq, "_HOST_PATH", str(path))
    monkeypatch.setattr(kq, "_native", kq._Native())
    with pytest.warns(RuntimeWarning, match="native call path"):
        with pytest.raises(ValueError, match="uint8"):
            kq.quantized_matmul(torch.zeros(1, 256), torch.zeros(8, 144), None, "q4_k")
    with warnings.catch_warnings():
        warnings.simplefilter("error")
        assert all(getattr(kq._native, k)() is None for k in kq._NATIVE_OPS)


def _workspace(lib, codec, M, N, K):
    lib.kq_qmm_workspace_size.restype = C.c_size_t
    return lib.kq_qmm_workspace_size(M, N, K, 1, lib.kq_codec_id(codec.encode()), 2)


def _streamed(lib, codec, M, N, K):
    """Whether a dense call is given the streamed kernel's workspace: 18 KiB per 32 rows and 256 weights of K."""
    return _workspace(lib, codec, M, N, K) >= -(-M // 32) * -(-K // 256) * 18 * 1024


@pytest.mark.parametrize("codec,M,N,K", [("iq4_xs", 140, 33024, 4096), ("q2_k", 255, 128256, 4096), ("q3_k", 129, 32768, 4096),
                                         ("q8_0", 333, 28672, 4128), ("q4_1", 512, 28672, 4128), ("iq4_nl", 160, 28672, 4128)])
def test_streamed_kernel_takes_what_the_tall_tiles_cannot(lib, codec, M, N, K):
    """Calls wide enough for tall tiles, with fewer rows or another K than the codec's tall-tile GEMM accepts."""
    assert _streamed(lib, codec, M, N, K)


@pytest.mark.parametrize("codec,M,N", [("q8_0", 1024, 2048), ("q4_0", 1024, 2048), ("iq3_s", 1024, 2048), ("iq2_xxs", 768, 2880),
                                       ("q4_1", 1024, 4096), ("q5_1", 640, 4096)])
def test_any_codec_kernel_keeps_calls_of_few_tall_tiles(lib, codec, M, N):
    """Beyond the streamed kernel's rows, K long enough for the f16 activations of the tall tiles to be the larger workspace:
    the any-codec kernel's is a multiple of the output (partial sums)."""
    assert _workspace(lib, codec, M, N, 65536) % (4 * M * N) == 0
    assert _workspace(lib, codec, M, 3 * N, 65536) > 2 * M * 65536


@pytest.mark.parametrize("codec,M,N,streamed", [("iq2_xs", 256, 4096, False),
                                                ("iq2_xs", 160, 8192, True), ("iq2_xs", 256, 1024, True),
                                                ("iq1_m", 512, 4096, False), ("iq1_s", 512, 2880, True), ("iq2_s", 512, 4096, True)])
def test_any_codec_kernel_keeps_full_tiles_of_short_decode(lib, codec, M, N, streamed):
    if streamed:
        assert _streamed(lib, codec, M, N, 65536)
    else:
        assert _workspace(lib, codec, M, N, 65536) % (4 * M * N) == 0


@pytest.mark.parametrize("codec,M,N,K,ranges", [
    ("q8_0", 600, 4096, 4096, 4),      # three row tiles of 256: 192 workgroups in two ranges, against 640 of 128 rows in four
    ("q6_k", 640, 4096, 14336, 4),
    ("q8_0", 1024, 4096, 4096, 2),     # (either kernel)
    ("q4_k", 512, 768, 16384, 21),     # 256-row tiles: 12 in 21 ranges
    ("q8_0", 1800, 1024, 1536, 5),     # 128-row tiles: 120 in five, against 64 of 256 rows in four
    ("iq2_xs", 512, 768, 16384, 22),   # 128-row tiles for the codebook codecs: 24 in 22
])
def test_transposed_product_takes_256_row_tiles_where_they_fill(lib, codec, M, N, K, ranges):
    """The route of y = x W as its workspace shows it: f32 partial sums of so many K ranges."""
    lib.kq_qmm_workspace_size.restype = C.c_size_t
    assert lib.kq_qmm_workspace_size(M, N, K, 0, lib.kq_codec_id(codec.encode()), 2) == ranges * M * N * 4


def moe_segments(lib, codec, ppe, glu, E=128, N=768, K=2048, R=8):
    return lib.kq_moe_segment_rows(ppe * E // R, R, E, N, K, glu, lib.kq_codec_id(codec.encode()))


@pytest.mark.parametrize("codec", ["q4_k", "q5_k", "q6_k"])
def test_moe_segments_by_pairs_per_expert(lib, codec):
    """In which segments the launcher runs a call: 32 pairs or up to 96, on both sides of its lines."""
    assert [moe_segments(lib, codec, p, 1) for p in (4, 21, 22, 62, 250)] == [32, 32, 96, 96, 96]
    assert [moe_segments(lib, codec, p, 0, N=2048, K=768) for p in (4, 27, 28, 62, 250)] == [32, 32, 96, 96, 96]
    # nothing to save where the 32-pair segments are a workgroup per CU: 8 experts of 2048 -> 512, 1536 and back
    assert [moe_segments(lib, codec, p, 1, E=8, N=512, R=2) for p in (32, 64, 96, 140)] == [32, 32, 32, 96]
    assert [moe_segments(lib, codec, p, 1, E=8, N=1536, R=2) for p in (32, 64)] == [96, 96]
    assert [moe_segments(lib, codec, p, 0, E=8, N=1024, K=512, R=2) for p in (32, 64, 96)] == [32, 32, 32]
    assert [moe_segments(lib, codec, p, 0, E=8, N=2048, K=1536, R=2) for p in (40, 64, 96, 128)] == [32, 32 if codec == "q4_k" else 96, 96, 96]
    assert [moe_segments(lib, codec, p, 0, E=16, N=2048, K=1536, R=2) for p in (32, 64)] == [96, 96]
    assert moe_segments(lib, "q8_0", 62, 1) == 0  # not theirs
    assert moe_segments(lib, codec, 1, 1, E=16) == 0  # too few pairs for the grouped kernels


@pytest.mark.parametrize("codec,S,N,K", [("q6_k", 8, 2048, 768), ("q4_k", 8, 2048, 1536), ("q4_k", 2, 4096, 14336), ("mxfp4", 4, 2880, 2880),
                                         ("q8_0", 32, 2048, 2048), ("iq1_s", 8, 2048, 2048)])
def test_mix_of_one_token_needs_no_workspace(lib, codec, S, N, K):
    """One token without a shared expert, up to 32 slots of any length; up to three with one; more of either need it."""
    f = lib.kq_gather_qmv_mix_workspace_size
    f.restype = C.c_size_t
    c = lib.kq_codec_id(codec.encode())
    assert f(1, S, 64, N, K, c, -1, 2) == 0
    assert f(3, S, 64, N, K, c, c, 2) == 0
    assert f(2, S, 64, N, K, c, -1, 2) > 0
    assert f(4, S, 64, N, K, c, c, 2) > 0
    assert f(1, 33, 64, N, K, c, -1, 2) > 0


@pytest.mark.parametrize("codec,K", [("q8_0", 512), ("q4_k", 256), ("nvfp4", 512)])
def test_gather_of_short_rows_uses_no_workspace(lib, codec, K):
    """128 heads, four tokens each, run in one launch; not from activations or weights that its loads cannot take, nor longer rows."""
    size, used = lib.kq_gather_qmm_workspace_size, lib.kq_gather_qmm_workspace_used
    size.restype = used.restype = C.c_size_t
    c = lib.kq_codec_id(codec.encode())

    def call(x=4096, w=8192, B=512, K=K, transpose=1):
        return used(C.c_void_p(x), C.c_void_p(w), B, 1, 128, 128, K, C.c_int64(K), C.c_int64(1 << 16), transpose, c, 2)

    assert size(512, 1, 128, 128, K, 1, c, 2) > 0 and call() == 0
    assert call(w=8193) == call(x=4098) == size(512, 1, 128, 128, K, 1, c, 2)
    assert call(K=2048) == size(512, 1, 128, 128, 2048, 1, c, 2) > 0
    assert call(B=16) == call(transpose=0) == 0
    assert call(B=24) == 0  # entry by entry, or the one launch
