"""The C-ABI library loads without a GPU and exports every function the header declares."""
import ctypes
import os
import subprocess

from nmtgminor_amd import _lib


def test_library_is_built():
    assert os.path.exists(_lib.LIB_PATH), "run `make -C nmtgminor_amd/csrc` first"


def test_every_declared_symbol_is_exported():
    lib = ctypes.CDLL(_lib.LIB_PATH)
    names = _lib.header_functions()
    assert "nmtg_ln_fwd" in names and "nmtg_last_error" in names
    missing = [n for n in names if not hasattr(lib, n)]
    assert not missing, f"declared in include/nmtg_hip.h but not exported: {missing}"


def test_no_undeclared_exports():
    out = subprocess.run(["nm", "-D", "--defined-only", _lib.LIB_PATH], capture_output=True, text=True).stdout
    exported = {line.split()[-1] for line in out.splitlines() if " T nmtg_" in line}
    assert exported == set(_lib.header_functions())


def test_version_and_error_text():
    lib = _lib.load()
    assert lib.nmtg_version() >= 100
    # argument validation happens before any device work, so this is safe without a GPU
    rc = lib.nmtg_ln_fwd(None, None, None, None, None, None, _lib.i64(4), _lib.i64(8), _lib.f32(1e-5),
                         _lib.i32(0), _lib.i32(0), None)
    assert rc == -1
    assert b"null pointer" in lib.nmtg_last_error()


def test_header_compiles_as_plain_c(tmp_path):
    src = tmp_path / "t.c"
    src.write_text('#include "nmtg_hip.h"\nint main(void){return NMTG_OK;}\n')
    inc = os.path.join(os.path.dirname(os.path.dirname(_lib.LIB_PATH)), "include")
    subprocess.run(["gcc", "-std=c99", "-Wall", "-Werror", "-I", inc, "-c", str(src), "-o", str(tmp_path / "t.o")],
                   check=True)


def test_attention_of_an_empty_batch_needs_no_address():
    """Sizes are looked at before pointers: torch gives a tensor without elements the null address."""
    lib = _lib.load()
    n, s = None, [_lib.i64(64)] * 12
    for fn, extra in ((lib.nmtg_flash_attn_batched_fwd, ()), (lib.nmtg_flash_attn_batched_fwd_probs, (n, _lib.i32(1)))):
        for batch, len_q in ((0, 6), (2, 0), (0, 0), (2, 6)):
            rc = fn(n, n, n, n, n, n, n, n, n, _lib.i64(batch), _lib.i64(2), _lib.i64(64), _lib.i64(len_q), _lib.i64(6), *s, _lib.f32(0.125),
                    _lib.i32(0), _lib.i32(0), _lib.f32(0.0), n, n, n, ctypes.c_uint64(0), ctypes.c_uint64(0), _lib.i32(_lib.BF16), n, *extra)
            assert rc == (-1 if batch and len_q else 0)
            assert rc == 0 or b"null pointer" in lib.nmtg_last_error()


def test_which_inference_calls_need_a_score_buffer(monkeypatch):
    lib = _lib.load()
    need = lambda tk, d, dtype=_lib.F16: lib.nmtg_attn_scores_needed(_lib.i64(tk), _lib.i64(d), _lib.i32(dtype))
    monkeypatch.delenv("NMTG_ATTN_PROBS", raising=False)
    assert [need(4, 64), need(1500, 128, _lib.BF16)] == [0, 0]
    assert [need(61, 64), need(0, 64), need(64, 32), need(64, 64, _lib.F32)] == [1, 1, 1, 1]
    monkeypatch.setenv("NMTG_ATTN_PROBS", "0")
    assert need(4, 64) == 1


def test_build_needs_nothing_under_tests(monkeypatch):
    """build() compiles and checks the two libraries. The CPU build of the kernels under tests/ may lack an instruction of theirs, or
    not be there at all."""
    import sys
    import types
    import __graft_entry__ as entry

    def broken():
        raise RuntimeError("hostsim: compilation failed")
    ran = []
    monkeypatch.setattr(entry.subprocess, "run", lambda cmd, **kw: ran.append(cmd))      # the libraries themselves are built
    monkeypatch.setitem(sys.modules, "hostsim_build", types.SimpleNamespace(available=lambda: True, build=broken, ensure=broken))
    monkeypatch.setattr(sys, "path", list(sys.path))
    entry.build()
    assert len(ran) == 1 and ran[0][0] == "make"
