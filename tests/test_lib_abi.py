"""The C ABI (CPU): libmiq.so loads, exports every function include/miq.h declares, the
Python binding covers them, and argument validation fails cleanly without touching a GPU."""
import ctypes
import os
import re

import pytest

from webpytorch_amd import _lib

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def declared_functions():
    src = open(os.path.join(ROOT, "include", "miq.h")).read()
    src = re.sub(r"/\*.*?\*/", "", src, flags=re.S)
    return sorted(set(re.findall(r"\b(miq_[a-z0-9_]+)\s*\(", src)))


def test_header_declares_entry_points():
    names = declared_functions()
    assert "miq_gptq_gemv" in names and "miq_q4k_gemv" in names and len(names) >= 8


def test_library_exports_every_declared_symbol():
    L = _lib.lib()
    missing = [n for n in declared_functions() if not hasattr(L, n)]
    assert not missing, missing
    assert L.miq_version() == 1


def test_binding_covers_every_compute_entry_point():
    skip = {"miq_last_error", "miq_version", "miq_decode_state_words", "miq_gptq_gemv_noalloc_max_bytes"}
    assert set(declared_functions()) - skip == set(_lib.SIGNATURES)


def test_validation_errors_raise_without_gpu():
    # rejected before any HIP call: unsupported bit width, bad divisibility, bad Q4_K K
    with pytest.raises(NotImplementedError, match="bits=3"):
        _lib.call("miq_gptq_gemv", None, 1, None, None, None, None, 1, None, None, 1, 1, 64, 64, 32, 3, 0.0,
                  None, 0, None)
    with pytest.raises(ValueError, match="divide"):
        _lib.call("miq_gptq_gemv", None, 1, None, None, None, None, 1, None, None, 1, 1, 100, 64, 32, 4, 0.0,
                  None, 0, None)
    with pytest.raises(ValueError, match="multiple of 256"):
        _lib.call("miq_q4k_gemv", None, 1, None, None, None, 0, 1, 300, 8, None)
    with pytest.raises(ValueError, match="divide"):
        _lib.call("miq_gptq_quantize", None, 0, 0, 100, 8, 32, 4, None, None, None, None)
    msg = _lib.lib().miq_last_error().decode()
    assert "gptq_quantize" in msg


def test_missing_library_fails_loudly(monkeypatch, tmp_path):
    monkeypatch.setattr(_lib, "LIB_PATH", str(tmp_path / "libmiq.so"))
    monkeypatch.setattr(_lib, "_lib", None)
    with pytest.raises(_lib.MiqError, match="not built"):
        _lib.lib()


def test_gemv_workspace_query_is_host_only():
    """The split-K plan is computed on the host: a K range longer than one workgroup's batches
    gets a workspace (counters + partials), a short one none."""
    from webpytorch_amd import core
    small = core.gemv_workspace_bytes(1, 896, 4864, 128, 4, _lib.MIQ_F16)
    assert small > 0 and small % 4 == 0
    assert small >= 4864 * 4 * 2  # at least two K slices of fp32 partials
    assert core.gemv_workspace_bytes(1, 128, 151936, 128, 4, _lib.MIQ_F16) == 0
    assert core.gemv_workspace_bytes(0, 896, 4864, 128, 4, _lib.MIQ_F16) == 0
    with pytest.raises(NotImplementedError, match="group size"):
        core.gemv_workspace_bytes(1, 896, 4864, 16, 4, _lib.MIQ_F16)


@pytest.mark.parametrize("dt,rows", [(_lib.MIQ_F16, 1), (_lib.MIQ_F32, 2)])
def test_ggml_gemm_workspace_holds_sums_for_types_with_mins_only(dt, rows):
    """The 8-byte sums of 32 staged values, which only Q4_K and Q5_K multiply (by their mins)."""
    from webpytorch_amd import core
    M, K, N = 1024, 4096, 14336  # a grid that does not split K
    need = {t: core.ggml_gemm_workspace_bytes(M, K, N, dt, t)
            for t in ("Q4_K", "Q5_K", "Q6_K", "Q8_0", "Q4_0", "Q5_0", "IQ4_NL")}
    staged = rows * M * K * 2 + 4 * M + (4 << 20)
    for t, n in need.items():
        assert n == staged + (rows * M * K // 32 * 8 if t in ("Q4_K", "Q5_K") else 0), t


def test_few_rows_workspace_says_what_the_kernel_covers():
    """0 where K is not split, counters and fp32 slice sums where it is, None where another kernel
    runs (more rows, other groups or code widths, more than 32 slices or 256 column tiles)."""
    from webpytorch_amd import core
    need = core.few_rows_workspace_bytes
    assert need(6, 4096, 11008, 128, 4) == 0
    assert need(6, 4096, 4096, 128, 4) == (4 << 20) + 8 * 64 * 4096  # slices x tiles x 16 x 64 floats
    for M, K, N, gs, bits in ((17, 4096, 4096, 128, 4), (6, 4096, 4096, 64, 4), (6, 4096, 4096, 128, 8),
                              (6, 16512, 512, 128, 4), (6, 8192, 16448, 128, 4)):
        assert need(M, K, N, gs, bits) is None
