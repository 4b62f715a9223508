"""The C-ABI library loads, exports every symbol the public header declares,
and rejects bad arguments before touching the GPU (host logic only)."""
import ctypes
import os
import re

import pytest

from nanovllm_amd import _native

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
INCLUDE = os.path.join(ROOT, "include")


def _declared():
    text = "".join(open(os.path.join(INCLUDE, f)).read() for f in sorted(os.listdir(INCLUDE)) if f.endswith(".h"))
    return sorted(set(re.findall(r"\b(nvamd_[a-z0-9_]+)\s*\(", text)))


def test_header_declares_the_entry_points():
    assert _declared() == sorted(_native.SIGNATURES)


def test_library_exports_every_declared_symbol():
    lib = _native.load()
    for name in _declared():
        assert hasattr(lib, name), name
    assert lib.nvamd_abi_version() == _native.ABI_VERSION


def test_rejects_unsupported_head_dim_without_gpu():
    lib = _native.load()
    st = lib.nvamd_fp8_decode_attention(None, None, None, None, None, None, 4, 8, 2, 64, 16, 256, 4,
                                        0.1, 0, None, 0, 0, None)
    assert st == 2
    assert b"head_dim" in lib.nvamd_last_error()


def test_rejects_bad_gqa_and_block_size_without_gpu():
    lib = _native.load()
    assert lib.nvamd_fp8_decode_attention(None, None, None, None, None, None, 4, 6, 4, 128, 16, 256, 4,
                                          0.1, 0, None, 0, 0, None) == 1
    # block sizes must be multiples of 16 (nanovllm/config.py:30): 40 is rejected as unsupported;
    # 48 passes that check and fails later on the null pointers
    assert lib.nvamd_fp8_decode_attention(None, None, None, None, None, None, 4, 8, 2, 128, 16, 40, 4,
                                          0.1, 0, None, 0, 0, None) == 2
    assert b"multiple of 16" in lib.nvamd_last_error()
    assert lib.nvamd_fp8_decode_attention(None, None, None, None, None, None, 4, 8, 2, 128, 16, 48, 4,
                                          0.1, 0, None, 0, 0, None) == 1
    assert b"null pointer" in lib.nvamd_last_error()
    assert lib.nvamd_fp8_prefill_attention(None, None, None, None, None, None, None, 4, 1, 8, 2, 128, 100,
                                           256, 2, 4, 4, 0.1, 100, None, 0, 0, None) == 1  # part_tokens % 256
    assert b"part_tokens" in lib.nvamd_last_error()
    assert lib.nvamd_store_kvcache(None, 0, None, 0, None, None, None, -1, 8, 128, 10, 0, None) == 1


def test_rejects_partition_wider_than_the_block_table_window():
    """A paged split-KV partition may span at most 63 KV blocks."""
    lib = _native.load()
    st = lib.nvamd_fp8_decode_attention(None, None, None, None, None, None, 4, 8, 2, 128, 16, 256, 4,
                                        0.1, 64 * 256, None, 0, 0, None)
    assert st == 1 and b"63 blocks" in lib.nvamd_last_error()
    fake_table = 0x1000  # validation fails before any pointer is used
    st = lib.nvamd_fp8_prefill_attention(None, None, None, None, fake_table, None, None, 4, 1, 8, 2, 128,
                                         1024, 64, 2, 4, 4, 0.1, 64 * 64, None, 0, 0, None)
    assert st == 1 and b"63 blocks" in lib.nvamd_last_error()
    # the automatic choice never exceeds the window
    nb = lib.nvamd_decode_workspace_bytes(1, 8, 2, 4096, 256, 0)
    assert nb > 0  # 1M-token capacity must be split


def test_qk_norm_rope_store_rejects_more_than_128_head_rows_without_gpu():
    """One workgroup per token takes at most 128 head rows (q + k + v)."""
    lib = _native.load()
    args = lambda hq, hkv: (None, (hq + 2 * hkv) * 128, None, None, None, 1e-6, None, 4096, None, None, None, None,
                            None, 1, hq, hkv, 128, 16, None)
    assert lib.nvamd_qk_norm_rope_store(*args(112, 16)) == 2
    assert b"128 head rows" in lib.nvamd_last_error()
    assert lib.nvamd_qk_norm_rope_store(*args(96, 16)) == 1   # 128 rows pass the shape checks (then: null pointers)
    assert b"null pointer" in lib.nvamd_last_error()


def test_fp8_linear_rejects_bad_shapes_without_gpu():
    """K and N must be multiples of the 128 block (fp8_linear.py:114)."""
    lib = _native.load()
    assert lib.nvamd_fp8_act_quant(None, 100, 0, None, None, 4, 100, None) == 1
    assert b"K % 128" in lib.nvamd_last_error()
    assert lib.nvamd_fp8_act_quant(None, 128, 2, None, None, 4, 128, None) == 2
    assert lib.nvamd_fp8_act_quant(None, 128, 0, None, None, 4, 128, None) == 1
    assert b"null pointer" in lib.nvamd_last_error()
    assert lib.nvamd_fp8_block_gemm(None, None, None, 256, None, None, 200, 0, 4, 200, 256, None, 0, None) == 1
    assert lib.nvamd_fp8_block_gemm(None, None, None, 256, None, None, 256, 3, 4, 256, 256, None, 0, None) == 2
    assert lib.nvamd_fp8_block_gemm(None, None, None, 256, None, None, 256, 0, 0, 256, 256, None, 0, None) == 0
    assert lib.nvamd_fp8_block_gemm(None, None, None, 256, None, None, 256, 0, 4, 256, 256, None, 64, None) == 1
    assert b"null workspace" in lib.nvamd_last_error()
    assert lib.nvamd_fp8_block_gemm_workspace_bytes(0, 256, 256) == 0
    assert lib.nvamd_fp8_block_gemm_workspace_bytes(4, 200, 256) == 0


@pytest.mark.parametrize("quantised", [0, 1])
def test_fp8_linear_plans_fit_the_lds_without_gpu(quantised):
    """Every size has a kernel, and its workgroups ask for no more LDS than a
    gfx950 workgroup can have: few tokens over all K (four tokens of K 7,296 to
    8,192 with eight waves that quantise would ask for 165,376 bytes), each
    kernel at its largest sizes."""
    lib = _native.load()
    lds = ctypes.c_int64()
    for M in [*range(1, 34), 64, 129, 192, 193, 256, 257, 1888, 8192]:
        for N in (128, 1280, 4096, 4224, 24576, 51200):
            for K in range(128, 32768 + 128, 128 if M <= 5 else 1920):
                kernel = lib.nvamd_fp8_linear_kernel(M, N, K, quantised, ctypes.byref(lds))
                assert 0 <= kernel <= 8, (M, N, K)
                assert 0 < lds.value <= 160 * 1024, (M, N, K, kernel, lds.value)
                if quantised == 0:
                    assert (lib.nvamd_fp8_block_linear_workspace_bytes(M, N, K) == 0) == (kernel == 8), (M, N, K)


def test_fp8_block_linear_checks_without_gpu():
    """The checks of the whole layer are those of its two steps: an empty batch
    (any row stride, null pointers) is accepted, a row stride that is shorter
    than a row or, with rows, not a multiple of 8 elements is not."""
    lib = _native.load()

    def call(M, x_stride, x=None):
        return lib.nvamd_fp8_block_linear(x, x_stride, 0, x, 128, x, x, 256, M, 256, 128, None, 0, None)

    for stride in (128, 130, 132):
        assert call(0, stride) == 0
        assert lib.nvamd_fp8_act_quant(None, stride, 0, None, None, 0, 128, None) == 0
    assert call(0, 100) == 1 and call(4, 100) == 1
    assert call(4, 128) == 1 and b"null pointer" in lib.nvamd_last_error()
    assert call(4, 132, x=0x1000) == 2 and b"row stride" in lib.nvamd_last_error()
