"""The C-ABI shared library: it loads, exports every symbol include/axn.h
declares, and rejects bad arguments with the documented codes before touching
the GPU (so all of this runs on a host without one)."""

import ctypes
import os
import re
import subprocess
import sysconfig
import zlib

import pytest

from axonn_amd import _native as nv

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def declared_symbols():
    text = open(os.path.join(ROOT, "include", "axn.h")).read()
    return sorted(set(re.findall(r"AXN_API\s+[\w\s\*]+?\b(axn_[a-z0-9_]+)\s*\(", text)))


def test_header_declares_the_expected_entry_points():
    names = declared_symbols()
    assert len(names) >= 14
    assert set(names) == set(nv.SYMBOLS), "binding table and header disagree"


def test_library_loads_and_exports_every_declared_symbol():
    lib = ctypes.CDLL(nv.lib_path())
    for name in declared_symbols():
        assert hasattr(lib, name), "libaxn_gfx950.so does not export %s" % name
    assert nv.load().axn_abi_version() == nv.ABI_VERSION


def test_the_version_goes_with_the_entry_points():
    """A change of the entry points takes a version of its own: raise it together with what is written here."""
    assert (nv.ABI_VERSION, len(nv.SYMBOLS)) == (16, 43)


def test_the_version_goes_with_the_flags_and_arguments():
    """So does a new constant or argument: a library that does not know it would fail in the middle of a step."""
    text = open(os.path.join(ROOT, "include", "axn.h")).read()
    text = re.sub(r"#define AXN_ABI_VERSION[^\n]*", "", re.sub(r"/\*.*?\*/", " ", text, flags=re.S))
    assert "AXN_ANY_SIZES" in text and "axn_mt_adam" in text
    assert (nv.ABI_VERSION, "%08x" % zlib.crc32(" ".join(text.split()).encode())) == (16, "eec76e83")


def test_a_library_of_another_version_is_refused_by_its_version(tmp_path, monkeypatch):
    """Also one that lacks entry points: the message names the versions, not the first missing symbol."""
    source = tmp_path / "old.c"
    source.write_text("int axn_abi_version(void) { return 14; }\n")
    old = tmp_path / "libold.so"
    subprocess.run(["gcc", "-shared", "-fPIC", "-o", str(old), str(source)], check=True)
    monkeypatch.setattr(nv, "_LIB_PATH", str(old))
    monkeypatch.setattr(nv, "_lib", None)
    with pytest.raises(ImportError, match="ABI version 14"):
        nv.load()
    assert nv._lib is None


def test_library_is_a_gfx950_code_object():
    blob = open(nv.lib_path(), "rb").read()
    assert b"gfx950" in blob


def test_workspace_queries():
    lib = nv.load()
    assert lib.axn_mt_scan_workspace_bytes(64, 1_300_000_000) >= (1_300_000_000 // 65536 + 64) * 16
    assert lib.axn_mt_scan_workspace_bytes(-1, 5) == 0
    assert lib.axn_dgelu_dbias_workspace_bytes(8192, 5120) == 64 * 5120 * 4
    assert lib.axn_dgelu_dbias_workspace_bytes(0, 8) == 0
    # split contraction: fp32 partial products, only for problems with few 128 x 128 tiles
    assert lib.axn_gemm_workspace_bytes(1, 512, 8192, 3584) == 4 * 512 * 3584 * 4   # dgrad, 112 tiles
    assert lib.axn_gemm_workspace_bytes(0, 512, 8192, 3584) == 2 * 512 * 8192 * 4   # fwd, 128 tiles of 256 x 128, 2 parts
    assert lib.axn_gemm_workspace_bytes(2, 512, 8192, 3584) == 0                    # wgrad, 448 large tiles
    assert lib.axn_gemm_workspace_bytes(0, 4096, 6144, 4096) == 0                   # 384 large tiles: no split
    assert lib.axn_gemm_workspace_bytes(0, 4096, 4096, 4096) == 0                   # one whole round
    assert lib.axn_gemm_workspace_bytes(0, 100, 128, 1024) == 0                     # ragged: no split
    assert lib.axn_gemm_workspace_bytes(0, 128, 128, 512) == 0                      # contraction too short
    assert lib.axn_gemm_workspace_bytes(0, 128, 128, 4096) == 8 * 128 * 128 * 4
    assert lib.axn_gemm_workspace_bytes(3, 128, 128, 4096) == 0 and lib.axn_gemm_workspace_bytes(0, 0, 8, 8) == 0
    # the parts are chosen by estimated time: a short contraction over an output that already has a
    # workgroup for every CU is not split, few tiles take as many parts as still pay for their sums
    assert lib.axn_gemm_workspace_bytes(0, 1024, 4096, 2560) == 0                   # 256 small tiles, 40 stages
    assert lib.axn_gemm_workspace_bytes(0, 256, 2560, 2560) == 4 * 256 * 2560 * 4   # 40 small tiles: 4 parts
    assert lib.axn_gemm_workspace_bytes(0, 512, 4096, 2560) == 2 * 512 * 4096 * 4   # 128 small tiles: 2, not 4
    assert lib.axn_gemm_workspace_bytes(0, 256, 4096, 14336) == 8 * 256 * 4096 * 4  # long contraction: 8
    # few tokens: a stream over the weights, unless a few workgroups would walk a long contraction
    for m, n, k, parts in ((16, 4096, 14336, 0), (32, 4096, 65536, 0), (64, 14336, 14336, 0), (64, 4096, 8192, 0),
                           (64, 512, 2048, 0), (8, 512, 14336, 0), (64, 512, 5120, 1), (32, 512, 28672, 1),
                           (16, 64, 14336, 1), (64, 4096, 14336, 1), (15, 3904, 16256, 0), (8, 1024, 57344, 0),
                           (14, 3072, 14336, 0), (24, 3584, 14336, 0), (40, 3584, 14336, 1)):
        assert (lib.axn_gemm_workspace_bytes(0, m, n, k) > 0) == bool(parts), (m, n, k)
    # embedding: four int32 arrays over the tokens, one over the rows, and the sort's digit
    # counts (17 key bits = two passes of 9 and 8 bits, one count per digit and 512 tokens)
    T, V = 16384, 128256
    need = lib.axn_embedding_workspace_bytes(T, V)
    counts = (512 + 256) * (T // 512) * 4
    assert 4 * T * 4 + V * 4 + counts <= need <= 4 * T * 4 + V * 4 + counts + 4096
    assert lib.axn_embedding_workspace_bytes(0, V) >= V * 4
    assert lib.axn_embedding_workspace_bytes(T, 0) == 0 and lib.axn_embedding_workspace_bytes(-1, V) == 0


def test_fp32_workspace_queries():
    """Parts for problems of 2^32 multiply-adds and more, except thin ones, which the native kernel does faster."""
    q = nv.load().axn_gemm_f32_workspace_bytes
    assert q(0, 64, 1024, 4096) == 0                                                  # below the line
    assert q(0, 2048, 4096, 1024) == 0 and q(0, 512, 4096, 2048) > 0                   # one part, several
    assert q(0, 300, 2048, 8192) > 0 and q(1, 300, 8192, 2048) > 0 and q(2, 8192, 300, 2048) > 0
    assert q(0, 8, 8192, 65536) == 0 and q(0, 8192, 8, 65536) == 0 and q(0, 16, 16384, 16384) == 0


def _err():
    return nv.load().axn_last_error().decode()


A = ctypes.c_void_p(0x1000)  # never dereferenced: validation fails first


def test_gemm_argument_errors():
    lib = nv.load()
    f = lib.axn_gemm_fwd
    assert f(None, A, None, A, None, 8, 8, 8, 8, 8, 8, 0, None) == nv.AXN_EINVAL
    assert "null" in _err()
    assert f(A, A, None, A, None, 0, 8, 8, 8, 8, 8, 0, None) == nv.AXN_EINVAL
    assert f(A, A, None, A, None, 8, 12, 8, 8, 8, 16, 0, None) == nv.AXN_ESHAPE
    assert "multiples of 8" in _err()
    assert f(A, A, None, A, None, 8, 8, 8, 4, 8, 8, 0, None) == nv.AXN_EINVAL  # ld < row
    assert f(A, A, None, A, None, 8, 8, 8, 12, 8, 8, 0, None) == nv.AXN_EALIGN  # ld % 8
    assert f(ctypes.c_void_p(0x1004), A, None, A, None, 8, 8, 8, 8, 8, 8, 0, None) == nv.AXN_EALIGN
    assert f(A, A, None, A, None, 8, 8, 8, 8, 8, 8, 7, None) == nv.AXN_EINVAL  # epilogue
    assert f(A, A, None, A, None, 8, 8, 8, 8, 8, 8, nv.EPI_BIAS, None) == nv.AXN_EINVAL
    assert "bias" in _err()
    assert f(A, A, None, A, None, 2 ** 31, 8, 8, 8, 8, 8, 0, None) == nv.AXN_ELIMIT
    assert lib.axn_gemm_dgrad(A, A, None, 8, 8, 8, 8, 8, 8, None) == nv.AXN_EINVAL
    assert lib.axn_gemm_wgrad(A, A, A, 8, 8, 8, 8, 8, 8, 2, nv.BF16, None) == nv.AXN_EINVAL
    assert lib.axn_gemm_wgrad(A, A, A, 8, 8, 8, 8, 8, 8, 0, nv.F16, None) == nv.AXN_EINVAL
    # both gradients in one call: the checks of the two calls
    fb = lib.axn_gemm_bwd
    assert fb(A, A, A, A, A, nv.F32, 8, 8, 8, 8, 8, 8, 8, 8, 0, nv.F32, None) == nv.AXN_EINVAL
    assert fb(A, A, A, A, A, nv.BF16, 8, 8, 8, 8, 8, 8, 8, 8, 2, nv.BF16, None) == nv.AXN_EINVAL
    assert fb(A, A, A, A, A, nv.BF16, 8, 8, 8, 8, 8, 8, 8, 8, 0, nv.F16, None) == nv.AXN_EINVAL
    assert fb(A, A, None, A, A, nv.BF16, 8, 8, 8, 8, 8, 8, 8, 8, 0, nv.BF16, None) == nv.AXN_EINVAL
    assert fb(A, A, A, A, A, nv.BF16, 8, 12, 8, 16, 8, 8, 8, 8, 0, nv.BF16, None) == nv.AXN_ESHAPE
    assert "axn_gemm_bwd" in _err()
    # the same with the input gradient in parts: only sizes that have a workspace, with that workspace
    need = lib.axn_gemm_bwd_workspace_bytes(777, 6144, 4096, 0)
    assert need > 0 and need % (777 * 4096 * 4) == 0
    assert lib.axn_gemm_bwd_workspace_bytes(777, 6144, 4092, 0) == lib.axn_gemm_bwd_workspace_bytes(0, 8, 8, 1) == 0
    fp = lib.axn_gemm_bwd_ws
    sizes = (777, 6144, 4096, 6144, 4096, 4096, 4096, 4096)
    assert fp(A, A, A, A, A, nv.BF16, *sizes, 0, nv.BF16, A, need - 1, None) == nv.AXN_EINVAL
    assert fp(A, A, A, A, A, nv.BF16, *sizes, 0, nv.BF16, None, need, None) == nv.AXN_EINVAL
    assert fp(A, A, A, A, A, nv.BF16, 8, 8, 8, 8, 8, 8, 8, 8, 0, nv.BF16, A, need, None) == nv.AXN_EINVAL
    assert fp(A, A, A, A, A, nv.F32, *sizes, 0, nv.F32, A, need, None) == nv.AXN_EINVAL
    assert fp(A, A, A, A, A, nv.BF16, 777, 6144, 4096, 1 << 22, 4096, 4096, 4096, 4096, 0, nv.BF16, A, need,
              None) == nv.AXN_ESHAPE
    # fp32 result: the promotion of an fp32 bias, so only with a bias epilogue
    fo = lib.axn_gemm_fwd_f32out
    assert fo(A, A, A, A, None, nv.BF16, 8, 8, 8, 8, 8, 8, nv.EPI_NONE, None) == nv.AXN_EINVAL
    assert "BIAS" in _err()
    assert fo(A, A, A, A, None, nv.F32, 8, 8, 8, 8, 8, 8, nv.EPI_BIAS, None) == nv.AXN_EINVAL
    assert fo(A, A, None, A, None, nv.F16, 8, 8, 8, 8, 8, 8, nv.EPI_BIAS, None) == nv.AXN_EINVAL
    assert fo(A, A, A, A, None, nv.BF16, 8, 12, 8, 8, 8, 16, nv.EPI_BIAS, None) == nv.AXN_ESHAPE
    # the fp16 entry points share the checks; dW there is fp16 or fp32, never bf16
    assert lib.axn_gemm_fwd_f16(A, A, None, A, None, 8, 12, 8, 8, 8, 16, 0, None) == nv.AXN_ESHAPE
    assert "axn_gemm_fwd_f16" in _err()
    assert lib.axn_gemm_dgrad_f16(A, None, A, 8, 8, 8, 8, 8, 8, None) == nv.AXN_EINVAL
    assert lib.axn_gemm_wgrad_f16(A, A, A, 8, 8, 8, 8, 8, 8, 0, nv.BF16, None) == nv.AXN_EINVAL
    assert "fp16 or fp32" in _err()
    # any number of output features: the pre-activation is stored in 16-byte vectors, as Y's first row
    fn = lib.axn_gemm_any_n
    half_aligned = ctypes.c_void_p(0x1008)
    for n, ld in ((16, 16), (17, 17)):
        assert fn(0, A, A, A, A, half_aligned, nv.BF16, 8, n, 8, 8, 8, ld, nv.EPI_BIAS_GELU, 0, nv.BF16, None, 0,
                  None) == nv.AXN_EALIGN
        assert "Zsave" in _err()
    # split-contraction variants
    ws = lib.axn_gemm_dgrad_ws
    assert ws(A, A, A, nv.F32, 512, 8192, 3584, 8192, 3584, 3584, A, 1 << 30, None) == nv.AXN_EINVAL
    assert ws(A, A, A, nv.BF16, 512, 8192, 3584, 8192, 3584, 3584, A, 1024, None) == nv.AXN_EINVAL
    assert "workspace too small" in _err()
    assert ws(A, A, A, nv.BF16, 512, 8192, 3584, 8192, 3584, 3584, ctypes.c_void_p(0x1008), 1 << 30,
              None) == nv.AXN_EALIGN
    assert ws(A, None, A, nv.BF16, 512, 8192, 3584, 8192, 3584, 3584, A, 1 << 30, None) == nv.AXN_EINVAL
    assert lib.axn_gemm_wgrad_ws(A, A, A, nv.BF16, 8, 8, 8, 8, 8, 8, 0, nv.F16, A, 64, None) == nv.AXN_EINVAL
    assert lib.axn_gemm_fwd_ws(A, A, None, A, None, nv.F16, 8, 12, 8, 8, 8, 16, 0, None, 0, None) == nv.AXN_ESHAPE
    assert lib.axn_gemm_fwd_ws(A, A, None, A, None, nv.F16, 8, 16, 8, 8, 8, 16, 1, None, 0, None) == nv.AXN_EINVAL  # bias missing
    assert lib.axn_gemm_fwd_f32(A, None, None, A, None, 4, 4, 4, 0, None) == nv.AXN_EINVAL
    assert lib.axn_gemm_wgrad_f32(A, A, A, 4, 4, 4, 3, None) == nv.AXN_EINVAL
    assert lib.axn_gemm_dgrad_f32(ctypes.c_void_p(0x1002), A, A, 4, 4, 4, None) == nv.AXN_EALIGN


def test_swiglu_argument_errors():
    lib = nv.load()
    f, b = lib.axn_swiglu_fwd, lib.axn_swiglu_bwd
    assert f(None, A, A, nv.BF16, 8, 8, 8, None) == nv.AXN_EINVAL
    assert f(A, A, A, 7, 8, 8, 8, None) == nv.AXN_EINVAL
    assert f(A, A, A, nv.BF16, 8, 12, 16, None) == nv.AXN_ESHAPE
    assert f(A, A, A, nv.BF16, 8, 8, 4, None) == nv.AXN_EALIGN          # ld < N
    assert f(ctypes.c_void_p(0x1008), A, A, nv.BF16, 8, 8, 8, None) == nv.AXN_EALIGN
    assert b(A, A, A, A, None, nv.BF16, 8, 8, 8, None) == nv.AXN_EINVAL
    assert b(A, A, A, A, A, nv.F32, 0, 8, 8, None) == nv.AXN_EINVAL
    assert "axn_swiglu_bwd" in _err()


def test_gate_up_forward_argument_errors():
    f = nv.load().axn_gemm_swiglu_fwd
    ok = (nv.BF16, 256, 128, 64, 64, 64, 128, None)
    assert f(A, A, None, A, A, A, *ok) == nv.AXN_EINVAL                  # no up weights
    assert f(None, A, A, A, A, A, *ok) == nv.AXN_EINVAL
    assert f(A, A, A, A, A, A, nv.F32, *ok[1:]) == nv.AXN_EINVAL         # 16-bit types only
    assert "bf16 or fp16" in _err()
    assert f(A, A, A, A, ctypes.c_void_p(0x1008), A, *ok) == nv.AXN_EALIGN
    assert f(A, A, A, A, None, None, nv.BF16, 256, 132, 64, 64, 64, 136, None) == nv.AXN_ESHAPE  # N % 8
    # a valid GEMM shape that is not made of whole tiles is refused before any launch
    assert f(A, A, A, A, None, None, nv.BF16, 128, 128, 64, 64, 64, 128, None) == nv.AXN_ESHAPE
    assert "M % 256 == 0" in _err()


@pytest.mark.parametrize("M,N,K,beta,joint", [
    # where one launch of both gradients was measured slower than two, and neighbours where it is faster
    (1536, 3072, 1024, 0, False), (1280, 2560, 1280, 0, False), (1536, 6144, 1024, 0, True),
    (256, 11136, 1664, 0, False), (256, 9728, 1792, 1, False), (768, 4864, 1792, 1, True),
    (512, 11008, 8192, 0, False), (1024, 32000, 3584, 0, False), (1280, 15360, 2304, 0, True),
    (256, 18560, 5632, 1, False), (512, 13312, 3712, 1, False), (249, 25472, 4864, 1, False), (237, 13312, 5376, 1, False),
    (256, 14336, 4096, 0, True), (1376, 9088, 2112, 0, True), (649, 4032, 2176, 1, True), (1024, 6144, 4096, 0, True),
    (2100, 7424, 1536, 1, False), (3136, 11392, 1152, 0, False), (2688, 11203, 768, 0, False), (2944, 13824, 2048, 0, False),
    (2624, 12189, 512, 0, True), (3584, 8707, 1024, 1, True),
])
def test_sizes_whose_gradients_take_one_launch(M, N, K, beta, joint):
    parts = nv.load().axn_gemm_bwd_workspace_bytes(M, N, K, beta) // (M * K * 4)
    assert (parts > 1) == joint
    if joint:   # the input gradient's own parts
        assert parts * M * K * 4 == nv.load().axn_gemm_workspace_bytes(1, M, N, K)


def test_gate_up_forward_of_few_rows_argument_errors():
    f = nv.load().axn_gemm_swiglu_fwd_few
    ok = (nv.BF16, 16, 128, 64, 64, 64, 128, None)
    assert f(A, A, None, A, A, A, *ok) == nv.AXN_EINVAL                  # no up weights
    assert f(A, A, A, A, A, A, nv.F32, *ok[1:]) == nv.AXN_EINVAL         # 16-bit types only
    assert f(A, A, A, A, ctypes.c_void_p(0x1008), A, *ok) == nv.AXN_EALIGN
    assert f(A, A, A, A, None, None, nv.BF16, 16, 132, 64, 64, 64, 136, None) == nv.AXN_ESHAPE  # N % 8
    assert f(A, A, A, A, None, None, nv.BF16, 65, 128, 64, 64, 64, 128, None) == nv.AXN_ESHAPE  # a row too many
    assert f(A, A, A, A, None, None, nv.BF16, 16, 128, 64, 64, 1 << 24, 128, None) == nv.AXN_ESHAPE
    assert "axn_gemm_swiglu_fwd_few" in _err()


def test_dgrad_pair_argument_errors():
    f = nv.load().axn_gemm_dgrad_pair
    tail = (128, 128, 128, 128, 128, 128, None)      # N2, K, lddy, ldw, lddx, stream
    assert f(A, A, None, A, A, nv.BF16, 128, 128, *tail[:-1], None) == nv.AXN_EINVAL   # dY2 missing
    assert f(A, A, A, A, A, nv.F32, 128, 128, *tail) == nv.AXN_EINVAL
    assert f(A, A, A, A, A, nv.BF16, 128, 128, 0, 128, 128, 128, 128, None) == nv.AXN_EINVAL  # N2 = 0
    assert f(A, A, A, A, A, nv.BF16, 128, 128, 12, 128, 128, 128, 128, None) == nv.AXN_ESHAPE  # N2 % 8
    assert f(A, A, A, A, A, nv.BF16, 128, 256, 128, 128, 128, 128, 128, None) == nv.AXN_EINVAL  # lddy < N1
    assert f(A, A, ctypes.c_void_p(0x1008), A, A, nv.BF16, 128, 128, *tail) == nv.AXN_EALIGN
    # valid operands, but the first contraction is shorter than two stages
    assert f(A, A, A, A, A, nv.BF16, 128, 64, 64, 128, 64, 128, 128, None) == nv.AXN_ESHAPE
    assert "gemm_pair" in _err()


def test_embedding_argument_errors():
    lib = nv.load()
    f, b, r = lib.axn_embedding_fwd, lib.axn_embedding_bwd, lib.axn_embedding_renorm
    big = 1 << 30
    assert f(A, None, A, nv.F32, 4, 16, 8, 8, 8, None, None) == nv.AXN_EINVAL
    assert f(None, A, A, nv.F32, 4, 16, 8, 8, 8, None, None) == nv.AXN_EINVAL  # ids missing
    assert f(A, A, A, 7, 4, 16, 8, 8, 8, None, None) == nv.AXN_EINVAL
    assert f(A, A, A, nv.F32, -1, 16, 8, 8, 8, None, None) == nv.AXN_EINVAL
    assert f(A, A, A, nv.F32, 4, 16, 6, 8, 8, None, None) == nv.AXN_ESHAPE      # fp32 rows of 24 bytes
    assert f(A, A, A, nv.BF16, 4, 16, 12, 16, 16, None, None) == nv.AXN_ESHAPE  # bf16 rows of 24 bytes
    assert f(A, A, A, nv.F32, 4, 16, 8, 4, 8, None, None) == nv.AXN_EALIGN      # ldw < H
    assert f(A, A, A, nv.F32, 4, 16, 8, 8, 10, None, None) == nv.AXN_EALIGN
    assert f(A, ctypes.c_void_p(0x1004), A, nv.F32, 4, 16, 8, 8, 8, None, None) == nv.AXN_EALIGN
    assert f(A, A, A, nv.F32, 1 << 31, 16, 8, 8, 8, None, None) == nv.AXN_ELIMIT
    assert "axn_embedding_fwd" in _err()
    assert b(A, A, None, nv.F32, nv.F32, 4, 16, 8, 8, 8, -1, 0, 0, A, big, None) == nv.AXN_EINVAL
    assert b(A, A, A, nv.F16, nv.F32, 4, 16, 8, 8, 8, -1, 0, 0, A, big, None) == nv.AXN_EINVAL
    assert b(A, A, A, nv.BF16, nv.F32, 4, 16, 12, 16, 12, -1, 0, 0, A, big, None) == nv.AXN_ESHAPE
    assert b(A, A, A, nv.F32, nv.F32, 4, 16, 8, 8, 8, 16, 0, 0, A, big, None) == nv.AXN_EINVAL  # padding row
    assert b(A, A, A, nv.F32, nv.F32, 4, 16, 8, 8, 8, -2, 0, 0, A, big, None) == nv.AXN_EINVAL
    assert b(A, A, A, nv.F32, nv.F32, 4, 16, 8, 8, 8, -1, 0, 2, A, big, None) == nv.AXN_EINVAL  # beta
    assert b(A, A, A, nv.F32, nv.F32, 4, 16, 8, 8, 8, -1, 0, 0, A, 64, None) == nv.AXN_EINVAL
    assert "workspace" in _err()
    assert b(A, A, A, nv.F32, nv.F32, 4, 16, 8, 8, 8, -1, 0, 0, None, big, None) == nv.AXN_EINVAL
    assert r(A, None, nv.F32, 4, 16, 8, 8, 1.0, 2.0, A, big, None) == nv.AXN_EINVAL
    assert r(A, A, 7, 4, 16, 8, 8, 1.0, 2.0, A, big, None) == nv.AXN_EINVAL            # unknown dtype
    assert r(A, A, nv.F32, 4, 16, 8, 8, 0.0, 2.0, A, big, None) == nv.AXN_EINVAL
    assert r(A, A, nv.F32, 4, 16, 8, 8, 1.0, -1.0, A, big, None) == nv.AXN_EINVAL
    assert r(A, A, nv.F32, 4, 16, 8, 8, 1.0, 2.0, A, 16, None) == nv.AXN_EINVAL


def test_elementwise_argument_errors():
    lib = nv.load()
    f = lib.axn_dgelu_dbias
    assert f(None, None, None, nv.BF16, A, 8, 8, 8, 0, A, 1024, None) == nv.AXN_EINVAL
    assert f(A, A, None, nv.BF16, A, 8, 8, 8, 0, A, 1024, None) == nv.AXN_EINVAL  # Z without dZ
    assert f(A, None, None, nv.BF16, None, 8, 8, 8, 0, A, 1024, None) == nv.AXN_EINVAL  # nothing to do
    assert f(A, None, None, 7, A, 8, 8, 8, 0, A, 1024, None) == nv.AXN_EINVAL
    assert f(A, None, None, nv.BF16, A, 8, 12, 16, 0, A, 1024, None) == nv.AXN_ESHAPE
    assert f(A, None, None, nv.BF16, A, 8, 8, 8, 0, A, 4, None) == nv.AXN_EINVAL  # workspace too small
    assert "workspace" in _err()


def test_an_fp32_gradient_is_not_rounded_in_place():
    """dZ's elements are half as wide as dY's: its rows would overwrite others of dY that are still to be read.  (The
    workspace is too small throughout: what gets past the check is refused for that.)"""
    f = nv.load().axn_dgelu_dbias
    M, N, ld, Y = 5, 16, 24, 0x100000
    used = (M - 1) * ld + N
    for dtype in (nv.BF16 | nv.DY_F32, nv.F16 | nv.DY_F32 | nv.DBIAS_16BIT):
        for z, apart in [(Y, False), (Y + 16, False), (Y + 4 * used - 16, False), (Y + 4 * used, True),
                         (Y - 2 * used + 16, False), (Y - 2 * used, True)]:
            for Z in (None, 2 * Y):
                assert f(Y, Z, z, dtype, Y, M, N, ld, 0, Y, 4, None) == nv.AXN_EINVAL
                assert ("overlap" in _err()) != apart and ("workspace" in _err()) == apart, (z - Y, _err())
    # of one type, in place: accepted as it was
    assert f(Y, Y, Y, nv.BF16, Y, M, N, ld, 0, Y, 4, None) == nv.AXN_EINVAL and "workspace" in _err()


def test_multi_tensor_argument_errors():
    lib = nv.load()
    ptrs = (ctypes.c_void_p * 2)(0x1000, 0x2001)
    sizes = (ctypes.c_int64 * 2)(4, 4)
    res = ctypes.c_void_p(0x3000)
    assert lib.axn_mt_scan(ptrs, sizes, 2, nv.BF16, 1.0, 0.0, 0, res, A, 4096, None) == nv.AXN_EALIGN
    assert "g[1]" in _err()
    sizes[1] = -1
    assert lib.axn_mt_scan(ptrs, sizes, 2, nv.BF16, 1.0, 0.0, 0, res, A, 4096, None) == nv.AXN_EINVAL
    sizes[1] = 0  # empty tensors may carry any pointer
    assert lib.axn_mt_scan(ptrs, sizes, 2, 9, 1.0, 0.0, 0, res, A, 4096, None) == nv.AXN_EINVAL
    assert lib.axn_mt_scan(ptrs, sizes, 2, nv.BF16, 1.0, 0.0, 0, None, A, 4096, None) == nv.AXN_EINVAL
    assert lib.axn_mt_scan(ptrs, sizes, 2, nv.BF16, 1.0, 0.0, 5, res, A, 4096, None) == nv.AXN_EINVAL
    assert lib.axn_mt_scan(ptrs, sizes, 2, nv.BF16, 1.0, 0.0, 0, res, A, 0, None) == nv.AXN_EINVAL
    assert "workspace" in _err()
    hp = nv.AdamHParams()
    assert lib.axn_mt_adam(ptrs, ptrs, ptrs, ptrs, None, sizes, 2, nv.BF16, nv.BF16, 1.0, None,
                           None, None) == nv.AXN_EINVAL
    assert lib.axn_mt_adam(ptrs, None, ptrs, ptrs, None, sizes, 2, nv.BF16, nv.BF16, 1.0, None,
                           hp, None) == nv.AXN_EINVAL
    assert lib.axn_mt_adam(ptrs, ptrs, ptrs, ptrs, ptrs, sizes, 2, nv.BF16, nv.F32, 1.0, None,
                           hp, None) == nv.AXN_EINVAL
    assert lib.axn_mt_scale(ptrs, sizes, 2, nv.BF16, 1.0, None, 1, None) == nv.AXN_EINVAL
    assert "scan" in _err()
    assert lib.axn_mt_scale(ptrs, sizes, -1, nv.BF16, 1.0, None, 0, None) == nv.AXN_EINVAL


def test_scan_variants_argument_errors():
    """The norm's order may be anything but NaN; the entry point without a workspace rejects
    what its built-in array cannot hold before it touches the device."""
    lib = nv.load()
    ptrs = (ctypes.c_void_p * 2)(0x1000, 0x2000)
    sizes = (ctypes.c_int64 * 2)(4, 4)
    res = ctypes.c_void_p(0x3000)
    assert lib.axn_mt_scan_norm(ptrs, sizes, 2, nv.BF16, 1.0, 0.0, float("nan"), 0, res, A, 4096,
                                None) == nv.AXN_EINVAL
    assert "NaN" in _err()
    assert lib.axn_mt_scan_norm(ptrs, sizes, 2, nv.BF16, 1.0, 0.0, 3.0, 0, res, A, 0,
                                None) == nv.AXN_EINVAL          # workspace too small
    assert lib.axn_mt_scan_noalloc(ptrs, sizes, 2, 9, 1.0, 0.0, 0, res, None) == nv.AXN_EINVAL
    assert lib.axn_mt_scan_noalloc(ptrs, sizes, 2, nv.BF16, 1.0, 0.0, 0, None, None) == nv.AXN_EINVAL
    # 65536 chunks of 65536 elements fit the 1 MiB array; three tensors of 2^31 elements do not
    limit = 1048576
    assert lib.axn_mt_scan_workspace_bytes(3, 3 * 2 ** 31) > limit
    ptrs3 = (ctypes.c_void_p * 3)(0x1000, 0x2000, 0x4000)
    sizes3 = (ctypes.c_int64 * 3)(2 ** 31, 2 ** 31, 2 ** 31)
    assert lib.axn_mt_scan_noalloc(ptrs3, sizes3, 3, nv.BF16, 1.0, 0.0, 0, res, None) == nv.AXN_ELIMIT
    assert "scratch" in _err() and "axn_mt_scan" in _err()


def test_probe_library_loads_and_checks_its_arguments():
    """The benchmark-only library (include/axn_probe.h) is built beside the product
    library, exports what its header declares and rejects bad arguments before any launch."""
    text = open(os.path.join(ROOT, "include", "axn_probe.h")).read()
    assert re.findall(r"AXN_PROBE_API\s+int\s+(axn_\w+)\s*\(", text) == ["axn_probe_stream"]
    assert "axn_probe" not in open(os.path.join(ROOT, "include", "axn.h")).read()
    lib = nv.load_probe()
    assert lib.axn_probe_stream(7, A, A, 1024, None) == -1
    assert lib.axn_probe_stream(2, None, A, 1024, None) == -1
    assert lib.axn_probe_stream(1, None, None, 1024, None) == -1
    assert lib.axn_probe_stream(2, ctypes.c_void_p(0x1008), A, 1024, None) == -2
    assert lib.axn_probe_stream(1, None, A, 0, None) == 0     # nothing to do, nothing launched


def test_adam_hparams_struct_layout():
    assert ctypes.sizeof(nv.AdamHParams) == 32
    assert nv.SCAN_RESULT_BYTES == 32


def test_missing_library_fails_loudly(monkeypatch):
    monkeypatch.setattr(nv, "_lib", None)
    monkeypatch.setattr(nv, "_LIB_PATH", "/nonexistent/libaxn_gfx950.so")
    with pytest.raises(ImportError, match="not built"):
        nv.load()


FOREIGN = {
    "a symbol that this PyTorch lacks": "extern int of_another_pytorch(void); void* PyInit_axn_fast(void) { of_another_pytorch(); return 0; }",
    "no module": "int nothing;",
    "another version": """
        #include <Python.h>
        static struct PyModuleDef def = {PyModuleDef_HEAD_INIT, "axn_fast", 0, -1, 0};
        PyMODINIT_FUNC PyInit_axn_fast(void) {
          PyObject* m = PyModule_Create(&def);
          PyModule_AddIntConstant(m, "ABI_VERSION", %d);
          PyModule_AddStringConstant(m, "BUILT_FOR", "cpython-310, PyTorch 1.0");
          return m;
        }""" % nv.ABI_VERSION,
}


@pytest.mark.parametrize("what", sorted(FOREIGN))
def test_a_host_side_that_does_not_fit_is_left_alone(tmp_path, monkeypatch, what):
    """axn_fast.so is tied to one PyTorch and one Python, the library is not: it is used without the other."""
    source = tmp_path / "fast.c"
    source.write_text(FOREIGN[what])
    subprocess.run(["gcc", "-shared", "-fPIC", "-I" + sysconfig.get_paths()["include"], "-o", str(tmp_path / "axn_fast.so"), str(source)],
                   check=True)
    os.symlink(nv.lib_path(), tmp_path / "libaxn_gfx950.so")
    monkeypatch.setattr(nv, "_LIB_PATH", str(tmp_path / "libaxn_gfx950.so"))
    monkeypatch.setattr(nv, "_lib", None)
    monkeypatch.setattr(nv, "fast", None)
    with pytest.warns(UserWarning, match="axn_fast.so is not used"):
        lib = nv.load()
    assert lib.axn_abi_version() == nv.ABI_VERSION and nv.fast is None


def test_the_library_is_built_without_a_compiler_for_the_host_side(tmp_path, monkeypatch, capsys):
    from axonn_amd.csrc import build

    stale = tmp_path / "axn_fast.so"
    stale.write_bytes(b"of an earlier build")
    monkeypatch.setattr(build, "FAST_PATH", str(stale))
    monkeypatch.setenv("CXX", str(tmp_path / "no_compiler"))
    build.build_fast_if_possible()
    assert not stale.exists() and "axn_fast.so is not built" in capsys.readouterr().err
