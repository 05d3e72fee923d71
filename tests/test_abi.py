"""CPU: libsglk.so loads and exports every entry point that include/sglk.h declares; the ctypes table of the
host layer covers the same set; host-only calls (no GPU needed) behave."""
import ctypes
import os
import re

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HEADER = os.path.join(ROOT, "include", "sglk.h")


def declared_symbols():
    text = open(HEADER).read()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    return sorted(set(re.findall(r"SGLK_API\s+[\w\s\*]+?\b(sglk_\w+)\s*\(", text)))


def test_header_declares_entry_points():
    syms = declared_symbols()
    assert len(syms) > 50
    for must in ("sglk_decode_attention", "sglk_awq_gemm", "sglk_radix_match_prefix", "sglk_extend_attention",
                 "sglk_fp8_scaled_mm", "sglk_ar_all_reduce"):
        assert must in syms


def test_library_exports_every_declared_symbol():
    from sglang_security_amd import _lib

    assert os.path.exists(_lib.LIB_PATH), "libsglk.so has not been built (python -m sglang_security_amd.build)"
    L = ctypes.CDLL(_lib.LIB_PATH)
    missing = [s for s in declared_symbols() if not hasattr(L, s)]
    assert not missing, f"declared in sglk.h but not exported: {missing}"


def test_ctypes_table_matches_header():
    from sglang_security_amd import _lib

    assert set(_lib._SIGS) == set(declared_symbols())
    assert not _lib._PENDING


def test_host_only_calls():
    from sglang_security_amd import _lib

    L = _lib.lib()
    assert L.sglk_version() > 0
    assert L.sglk_ar_meta_size() > 0 and L.sglk_ipc_handle_bytes() == 64
    assert L.sglk_awq_gemm_workspace_bytes(64, 4096, 4096) > 0
    # counters + error word + tail tickets (rounded to 256), partials + log-sum-exps of 8 prefix splits and 2 x 4
    # remainder splits, one split count per request (rounded to 256)
    assert L.sglk_decode_shared_workspace_bytes(64, 32, 128, 8) == ((2 * 64 * 32 + 2) * 4 + 255) // 256 * 256 + \
        64 * 32 * (8 + 8) * 129 * 4 + 256
    # block sums are read from 17 rows on, and where the kernel of few rows does not take the shape
    assert [L.sglk_awq_gemm_reads_xsum(m, 4096, 4096, 128) for m in (1, 16, 17, 64)] == [0, 0, 1, 1]
    assert L.sglk_awq_gemm_reads_xsum(16, 4096 + 64, 4096, 128) == 1 and L.sglk_awq_gemm_reads_xsum(16, 4096, 4096, 256) == 1
    # argument validation happens before any GPU call
    rc = L.sglk_rmsnorm(None, None, None, 1, 128, 128, 128, 1e-6, 0, 2, None)
    assert rc == -1 and b"null" in L.sglk_last_error().lower()
    with pytest.raises(_lib.SglkError):
        _lib.check(rc, "rmsnorm")


def test_missing_library_fails_loudly(monkeypatch):
    from sglang_security_amd import _lib

    monkeypatch.setattr(_lib, "_lib", None)
    monkeypatch.setattr(_lib, "LIB_PATH", "/nonexistent/libsglk.so")
    with pytest.raises(ImportError, match="no CPU fallback"):
        _lib.lib()


def test_modules_import_where_torch_knows_no_gpu():
    """A torch without GPU support has no stream look-up; nothing below needs one before its first launch."""
    import subprocess
    import sys

    code = ("import torch\n"
            "if hasattr(torch._C, '_cuda_getCurrentRawStream'): del torch._C._cuda_getCurrentRawStream\n"
            "import sglang_security_amd.ops, sglang_security_amd.mem_cache.memory_pool, sglang_security_amd.attention.backend\n"
            "import sglang_security_amd.quantization.awq, sglang_security_amd.quantization.w8a8_fp8\n")
    subprocess.run([sys.executable, "-c", code], cwd=ROOT, check=True, timeout=300)


@pytest.mark.parametrize("columns", [512, 1280, 3072, 4080, 4096, 5120, 6144, 7168, 10240])
def test_fp8_splits_fill_the_units(columns):
    """64 rows of a long inner dimension, where what a unit has to walk is all that counts: at most a third more than with the
    best number of splits (blocks of two strips, one after the other on 256 units)."""
    from sglang_security_amd import ops

    def walk(splits):
        return -(-columns // 32 * splits // 256) / splits

    got = ops.fp8_mm_packed_partial_splits(64, columns, 18432)
    assert 1 <= got <= 8 and walk(got) <= 1.34 * min(walk(n) for n in range(1, 9))
