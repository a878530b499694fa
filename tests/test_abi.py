"""The C ABI: every symbol declared in include/*.h is exported, and the
argument checks that run before any HIP call return the documented status codes.
CPU only: no call here reaches a kernel launch."""
import ctypes
import re
from pathlib import Path

import pytest

from intent_amd import _native
from intent_amd import errors

HEADERS = sorted((Path(__file__).resolve().parent.parent / "include").glob("*.h"))


def declared_symbols():
    text = "\n".join(h.read_text() for h in HEADERS)
    return sorted(set(re.findall(r"^\s*(?:int|size_t|const char\*)\s+(intent_\w+)\s*\(", text, re.M)))


def test_header_declares_expected_entries():
    names = declared_symbols()
    assert len(names) >= 16
    assert set(names) == set(_native.SIGNATURES), "ctypes signature table and header disagree"


def test_library_exports_every_declared_symbol():
    lib = _native.library()
    for name in declared_symbols():
        assert hasattr(lib, name), name
    assert lib.intent_amd_abi_version() == _native.ABI_VERSION


def status(entry, *args):
    return getattr(_native.library(), entry)(*args)


P = ctypes.c_void_p
FAKE = 0x1000  # a 16-byte aligned non-null address; never dereferenced by the checks


def test_w4a16_argument_checks():
    # Shapes outside the tiled kernels (K not a multiple of 128, groups of other sizes, unaligned
    # rows) run the generic kernel (GPU tests); here only calls that are invalid, which fail before
    # any launch. K odd:
    assert status("intent_w4a16_matmul", FAKE, 1, 101, 101, FAKE, 8, 51, FAKE, FAKE, 1, 101, FAKE, 8, None) == \
        errors.INTENT_ERR_INVALID_ARGUMENT
    assert "even" in _native.last_error()
    # K not a multiple of the group size
    assert status("intent_w4a16_gemv", FAKE, 1, 96, 96, FAKE, 8, 48, FAKE, FAKE, 2, 64, FAKE, 8, None) == \
        errors.INTENT_ERR_INVALID_ARGUMENT
    # group size 0
    assert status("intent_w4a16_gemm", FAKE, 4, 256, 256, FAKE, 8, 128, FAKE, FAKE, 2, 0, FAKE, 8, None) == \
        errors.INTENT_ERR_INVALID_ARGUMENT
    # null pointer
    assert status("intent_w4a16_gemm", None, 4, 256, 256, FAKE, 8, 128, FAKE, FAKE, 2, 128, FAKE, 8, None) == \
        errors.INTENT_ERR_INVALID_ARGUMENT
    # row stride smaller than the row
    assert status("intent_w4a16_gemm", FAKE, 4, 256, 128, FAKE, 8, 128, FAKE, FAKE, 2, 128, FAKE, 8, None) == \
        errors.INTENT_ERR_INVALID_ARGUMENT
    # GEMV covers M <= 16 only
    assert status("intent_w4a16_gemv", FAKE, 17, 256, 256, FAKE, 8, 128, FAKE, FAKE, 2, 128, FAKE, 8, None) == \
        errors.INTENT_ERR_UNSUPPORTED
    # empty problems are a no-op success
    assert status("intent_w4a16_matmul", FAKE, 0, 256, 256, FAKE, 8, 128, FAKE, FAKE, 2, 128, FAKE, 8, None) == 0


def test_int8_and_w8a16_checks():
    # any K and any alignment run (the generic kernel off the tiled shapes); invalid calls fail first
    assert status("intent_w8a8_gemm", FAKE, 4, 128, 128, None, FAKE, 4, 128, FAKE, FAKE, 4, None) == \
        errors.INTENT_ERR_INVALID_ARGUMENT
    assert status("intent_w8a8_gemm", FAKE, 4, 100, 90, FAKE, FAKE, 4, 100, FAKE, FAKE, 4, None) == \
        errors.INTENT_ERR_INVALID_ARGUMENT  # a_ld < K
    assert status("intent_i8_gemm_i32", FAKE, 4, 128, 136, FAKE, 4, 100, None, FAKE, 4, None) == \
        errors.INTENT_ERR_INVALID_ARGUMENT  # w_ld < K
    assert status("intent_w8a16_matmul", FAKE, 4, 96, 96, None, 4, 96, FAKE, FAKE, 4, None) == \
        errors.INTENT_ERR_INVALID_ARGUMENT
    assert status("intent_w8a16_matmul", FAKE, 4, 96, 96, FAKE, 4, 96, FAKE, FAKE, 3, None) == \
        errors.INTENT_ERR_INVALID_ARGUMENT  # y_ld < N
    assert status("intent_i8_gemm_i32", FAKE, 0, 128, 128, FAKE, 4, 128, None, FAKE, 4, None) == 0


def test_moe_checks():
    assert status("intent_moe_route", FAKE, 8, 8, 9, 1, FAKE, FAKE, None) == errors.INTENT_ERR_UNSUPPORTED
    assert status("intent_moe_route", FAKE, 8, 0, 1, 1, FAKE, FAKE, None) == errors.INTENT_ERR_INVALID_ARGUMENT
    assert status("intent_moe_route", FAKE, 0, 8, 2, 1, FAKE, FAKE, None) == 0
    # capacity below R + E*(B-1)
    assert status("intent_moe_align", FAKE, 16, 2, 4, 128, FAKE, 100, FAKE, 10, FAKE, FAKE, None) == \
        errors.INTENT_ERR_INVALID_ARGUMENT
    assert "needs" in _native.last_error()
    assert status("intent_moe_align", FAKE, 16, 2, 3000, 128, FAKE, 10 ** 6, FAKE, 10 ** 4, FAKE, FAKE, None) == \
        errors.INTENT_ERR_UNSUPPORTED  # more than 2048 experts
    # other block sizes and dimensions off the tiles run the generic kernels (GPU tests); invalid calls:
    assert status("intent_moe_gate_up_w4", FAKE, 4, 256, 256, FAKE, FAKE, 2, 0, 2, FAKE, FAKE, FAKE, 2, 128, 128,
                  FAKE, 128, None) == errors.INTENT_ERR_INVALID_ARGUMENT  # block size 0
    assert status("intent_moe_gate_up_w4", FAKE, 4, 250, 256, FAKE, FAKE, 2, 32, 2, FAKE, FAKE, FAKE, 2, 128, 128,
                  FAKE, 128, None) == errors.INTENT_ERR_INVALID_ARGUMENT  # group 128 does not divide H = 250
    assert status("intent_moe_down_w4", FAKE, 95, FAKE, FAKE, 2, 128, 8, FAKE, FAKE, FAKE, 2, 256, 95, 32,
                  FAKE, 256, None) == errors.INTENT_ERR_INVALID_ARGUMENT  # F odd
    assert _native.library().intent_moe_workspace_size(512, 2, 8, 4096, 14336, 128) >= \
        16 * 128 * 14336 * 2 + 1024 * 4096 * 4  # block 128: padded activations + route outputs
    need = _native.library().intent_moe_workspace_size(512, 2, 8, 4096, 14336, 0)  # composite plan
    # 128 routes per expert: the composite may take 128- or 160-row blocks and sizes for either
    assert need == max(_native.library().intent_moe_workspace_size(512, 2, 8, 4096, 14336, b) for b in (128, 160))
    # 8 routes per expert: 128-row blocks only
    assert _native.library().intent_moe_workspace_size(32, 2, 8, 4096, 14336, 0) == \
        _native.library().intent_moe_workspace_size(32, 2, 8, 4096, 14336, 128)
    assert status("intent_moe_expert_ffn_w4", FAKE, FAKE, 512, 4096, 8, 2, 1, FAKE, FAKE, FAKE, FAKE, FAKE, FAKE,
                  14336, 128, FAKE, FAKE, need - 1, None, None, None) == errors.INTENT_ERR_WORKSPACE
    assert _native.library().intent_moe_workspace_size(-1, 2, 8, 64, 64, 128) == 0


def test_moe_expert_ffn_workspace_holds_what_the_plan_uses():
    lib = _native.library()
    every, exact = lib.intent_moe_expert_ffn_workspace_size, lib.intent_moe_expert_ffn_workspace_size_for
    D, F, round256 = 4096, 14336, lambda v: (v + 255) // 256 * 256
    for T, R, E in ((2048, 4096, 8), (512, 1024, 8), (4096, 8192, 8), (5000, 5000, 64)):  # many routes, or more than 4096
        base = sum(round256(b) for b in (2 * R * F, 4 * R * D, 4 * T, 4 * (T + 1), 4 * R))
        assert exact(T, R, D, F, E) == base, (T, R, E)  # no room for K runs that the plan does not take
    for T, R, E in ((16, 32, 8), (200, 400, 8)):  # few routes per expert: up to three results beside the first
        extra = exact(T, R, D, F, E) - sum(round256(b) for b in (2 * R * F, 4 * R * D, 4 * T, 4 * (T + 1), 4 * R))
        assert extra in (4 * R * D, 12 * R * D), (T, R, E)
    for T, R, E in ((1, 2, 8), (16, 32, 8), (512, 1024, 8), (2048, 4096, 8), (300, 4096, 64), (4096, 8192, 8)):
        assert exact(T, R, D, F, E) <= every(T, R, D, F), (T, R, E)
    assert exact(4, 8, 64, 64, 0) == 0 and exact(-1, 8, 64, 64, 2) == 0


def test_w4a16_streaming_kernel_against_the_gemv():
    # Up to 7 rows and parameter rows off whole quads of groups the GEMV is the faster for K just above 8192.
    size = _native.library().intent_w4a16_matmul_workspace_size
    for M in (3, 4, 6):
        for K, N in ((8320, 2304), (8320, 4096), (9344, 2304), (9344, 4096)):
            assert size(M, K, N, 128) == 0, (M, K, N)
    assert size(7, 8320, 2304, 128) == 0
    for M, K, N in ((7, 9344, 3072), (8, 8320, 2304), (12, 8320, 2304), (6, 8320, 2048), (6, 10240, 2304), (6, 10368, 4096),
                    (6, 14208, 2304), (3, 8192, 8200)):
        assert size(M, K, N, 128) > 0, (M, K, N)


def test_w4a16_streaming_kernel_at_short_k():
    # Below K = 1024 its partial sums weigh as much as the weights: wide outputs go to the tiles without runs.
    size = _native.library().intent_w4a16_matmul_workspace_size
    for M, K, N, group in ((100, 768, 2048, 128), (128, 896, 1024, 64), (26, 256, 106112, 128), (17, 640, 38400, 64), (17, 768, 22848, 128), (64, 896, 106112, 64)):
        assert size(M, K, N, group) == 0, (M, K, N)
    for M, K, N, group in ((17, 512, 8192, 128), (40, 768, 12288, 64), (17, 1024, 22848, 128)):
        assert size(M, K, N, group) > 0, (M, K, N)


def test_w4a16_wide_outputs_scratch():
    # Very wide outputs (a vocabulary head): the streaming kernel is weighed against the tiles there too, and
    # whatever takes the call keeps its partial sums within 64 MB.
    size = _native.library().intent_w4a16_matmul_workspace_size
    for N in (50304, 98304, 128256, 131072, 200000, 1 << 20):
        for K in (1024, 4096, 8192, 16384):
            for M in (2, 6, 16, 17, 33, 60, 77, 100, 128, 129, 300):
                assert size(M, K, N, 128) <= 64 << 20, (M, K, N)
    for M in (60, 77, 100, 128):  # 128-row tiles without K runs are the faster there
        assert size(M, 4096, 128256, 128) == 0, M
    for M in (6, 12, 16, 17, 33):  # the streaming kernel is
        assert size(M, 8192, 128256, 128) > 0, M


def test_kquant_checks():
    # Q8_K: x must be 16-byte aligned; rows of at least 256 values / 292 bytes
    assert status("intent_q8k_quantize", FAKE + 4, 3, 256, FAKE, 292, None) == errors.INTENT_ERR_ALIGNMENT
    assert status("intent_q8k_quantize", FAKE, 3, 128, FAKE, 292, None) == errors.INTENT_ERR_INVALID_ARGUMENT
    assert status("intent_q8k_quantize", FAKE, 3, 256, FAKE, 291, None) == errors.INTENT_ERR_INVALID_ARGUMENT
    assert status("intent_q8k_quantize", None, 0, 256, None, 292, None) == 0  # G = 0: nothing to do
    # Q4_K rows: stride below G records, misaligned rows, null inputs
    assert status("intent_q4k_q8k_gemv", FAKE, 4, 3, 400, FAKE, FAKE, None) == errors.INTENT_ERR_INVALID_ARGUMENT
    assert status("intent_q4k_q8k_gemv", FAKE, 4, 3, 440, FAKE, FAKE, None) == errors.INTENT_ERR_ALIGNMENT
    assert status("intent_q4k_q8k_gemv", FAKE, 4, 3, 432, FAKE + 2, FAKE, None) == errors.INTENT_ERR_ALIGNMENT
    assert status("intent_q4k_q8k_gemv", None, 4, 3, 432, FAKE, FAKE, None) == errors.INTENT_ERR_INVALID_ARGUMENT
    assert status("intent_q4k_q8k_gemv", FAKE, 0, 3, 432, FAKE, FAKE, None) == 0  # N = 0
    assert status("intent_q4k_projection", FAKE, 4, 3, 432, FAKE + 8, 256, FAKE, FAKE, None) == \
        errors.INTENT_ERR_ALIGNMENT


def test_probe_checks():
    e = errors
    rp = "intent_hbm_read_probe"
    assert status(rp, P(FAKE), 4095, 1, 0, P(FAKE), 256, None) == e.INTENT_ERR_INVALID_ARGUMENT  # bytes % 16
    assert status(rp, P(FAKE), 4096, 3, 0, P(FAKE), 256, None) == e.INTENT_ERR_UNSUPPORTED  # unroll
    assert status(rp, P(FAKE), 4096, 1, 4, P(FAKE), 256, None) == e.INTENT_ERR_INVALID_ARGUMENT  # store mode 0..3
    assert status(rp, P(FAKE), 4096, 1, 0, P(FAKE), 255, None) == e.INTENT_ERR_INVALID_ARGUMENT  # sink < 256
    # store mode: one workgroup of four waves per 4096 bytes at unroll 1, two words per wave
    assert status(rp, P(FAKE), 65536, 1, 1, P(FAKE), 127, None) == e.INTENT_ERR_INVALID_ARGUMENT
    assert status(rp, P(FAKE + 8), 4096, 1, 0, P(FAKE), 256, None) == e.INTENT_ERR_ALIGNMENT
    assert status("intent_mfma_peak_probe", 0, 0, 1, P(FAKE), None) == e.INTENT_ERR_INVALID_ARGUMENT


def test_status_mapping():
    assert isinstance(errors.status_error(-1, "e", "m"), ValueError)
    assert isinstance(errors.status_error(-2, "e", "m"), ValueError)
    assert isinstance(errors.status_error(-3, "e", "m"), NotImplementedError)
    assert isinstance(errors.status_error(-4, "e", "m"), RuntimeError)
    assert isinstance(errors.status_error(-5, "e", "m"), ValueError)
    with pytest.raises(NotImplementedError, match="M <= 16"):
        _native.call("intent_w4a16_gemv", FAKE, 17, 256, 256, FAKE, 8, 128, FAKE, FAKE, 2, 128, FAKE, 8, None)
    with pytest.raises(ValueError, match="multiple of group_size"):
        _native.call("intent_w4a16_matmul", FAKE, 1, 100, 100, FAKE, 8, 50, FAKE, FAKE, 4, 32, FAKE, 8, None)
