"""The C-ABI library loads and exports every symbol include/*.h declares.
Runs without a GPU: only symbol lookup and argument validation that happens
before any HIP call."""
import ctypes as C
import re
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parents[1]


def declared_symbols():
    names = set()
    for h in (ROOT / "include").glob("*.h"):
        text = h.read_text()
        text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
        for m in re.finditer(r"\b(pgd_[a-z0-9_]+)\s*\(", text):
            names.add(m.group(1))
    return sorted(names)


def test_header_declares_entry_points():
    names = declared_symbols()
    assert "pgd_device_open" in names and "pgd_matrix_gemv" in names
    assert len(names) >= 15


def test_library_exports_every_declared_symbol():
    from pagoda_amd import _lib

    l = _lib.lib()
    missing = [n for n in declared_symbols() if not hasattr(l, n)]
    assert not missing, missing
    # the Python binding covers the whole header too
    assert not [n for n in declared_symbols() if n not in _lib.SIGNATURES]


def test_unknown_device_spec_is_an_error():
    """device_from_env: an unknown value must not silently fall back to CPU
    (pagoda-hf/src/lib.rs:424)."""
    from pagoda_amd import _lib

    h = C.c_void_p()
    rc = _lib.lib().pgd_device_open(b"cpu", C.byref(h))
    assert rc == -1
    assert "unknown device spec" in _lib.last_error()
    rc = _lib.lib().pgd_device_open(b"hip:x", C.byref(h))
    assert rc == -1


def test_device_from_env_rejects_non_hip(monkeypatch):
    from pagoda_amd import device_from_env

    monkeypatch.setenv("PAGODA_DEVICE", "metal")
    with pytest.raises(ValueError):
        device_from_env()


def test_product_package_does_not_import_oracle():
    for p in (ROOT / "pagoda_amd").rglob("*"):
        if p.suffix in (".py", ".hip", ".cpp", ".h"):
            t = p.read_text()
            assert "oracle" not in t.replace("pagoda_amd", ""), p


@pytest.mark.parametrize("tiles16,n_in,rows,nm,fused", [
    (72, 896, 4, 1, True),      # 4 waves, small LDS
    (304, 896, 4, 2, True),     # two workgroups of 8 waves per CU
    (304, 896, 5, 2, False),    # more rows than the few-row kernel's
    (288, 3584, 1, 1, False),   # 14 waves: one per CU, 32 tiles left for a second round
    (256, 3584, 1, 2, True),    # one round
    (512, 2048, 1, 2, False),   # 16 waves
    (300, 2048, 4, 1, True),    # 71 KB of LDS: two per CU
    (300, 2048, 5, 1, False),   # 89 KB: one
    (513, 256, 1, 1, False),
    (64, 8448, 1, 1, False),    # wider than the ordered-sum norm
])
def test_norm_goes_into_launches_of_one_round(tiles16, n_in, rows, nm, fused):
    """The RMSNorm runs inside a quantized-activation launch only where all its
    workgroups are resident at once (each repeats the norm's ordered sum): the
    library's own rule, at the limits of waves, LDS, rows and width."""
    from pagoda_amd import _lib

    rule = _lib.lib()["_ZN3pgd4gemv16q8act_norm_fusedEiiiiii"]  # pgd::gemv::q8act_norm_fused
    rule.restype = C.c_bool
    for fmt in (1, 2):
        assert rule(fmt, tiles16, (n_in + 255) // 256, n_in, rows, nm) is fused, fmt


@pytest.mark.parametrize("fmt,n_out,n_in,few", [
    (1, 5120, 5120, 3),     # two workgroups per CU; the rows of 4 fill the LDS
    (2, 5120, 5120, 3),
    (1, 3840, 5120, 6),     # one workgroup per CU
    (1, 18944, 3584, 1),    # five workgroups of 14 waves per CU
    (1, 2048, 11008, 3),    # 4 rows do not fit the LDS: one launch each
    (2, 2048, 11008, 4),
    (1, 3584, 18944, 4),
    (1, 4864, 896, 4),
    (1, 152064, 896, 1),
])
def test_few_row_kernel_takes_the_rows_it_is_faster_for(fmt, n_out, n_in, few):
    """The most rows of a Q4_K / Q6_K launch that run in the few-row kernel
    instead of on the matrix cores (same bits): the library's own rule, where
    the measured times of both cross."""
    from pagoda_amd import _lib

    rule = _lib.lib()["_ZN3pgd4gemv14q8act_few_rowsEiiiiid"]  # pgd::gemv::q8act_few_rows
    rule.restype, rule.argtypes = C.c_bool, [C.c_int] * 5 + [C.c_double]
    got = [rule(fmt, (n_out + 15) // 16, (n_in + 255) // 256, r, 1, 0.0) for r in range(1, 9)]
    assert got == [r <= few for r in range(1, 9)], got
