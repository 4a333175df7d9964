"""CPU-side checks: the C-ABI library loads and exports every declared symbol."""
import os
import re

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _declared(header, folder="include"):
    text = open(os.path.join(ROOT, folder, header)).read()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    return sorted(set(re.findall(r"\b((?:dq8|tao_ral|disc_ral)_[a-z0-9_]+)\s*\(", text)))


def test_exports_every_declared_symbol():
    from bladedisc_amd import _lib
    L = _lib.lib()
    headers = [h for h in os.listdir(os.path.join(ROOT, "include")) if h.endswith(".h")]
    assert headers
    total = 0
    for h in headers:
        for name in _declared(h):
            assert hasattr(L, name), "%s declared in %s but not exported" % (name, h)
            total += 1
    assert total >= 10


def test_the_product_library_exports_its_headers_and_nothing_else():
    """The variant-forcing entry points and the MFMA layout probe are declared in a tests-only
    header and live in libdisc_q8_testhooks.so; libdisc_q8_ral.so exports the C ABI of
    include/*.h and no other symbol."""
    import subprocess
    from bladedisc_amd import _lib
    L, H = _lib.lib(), _lib.hooks()
    hooks = _declared("dq8_test_hooks.h", "tests")
    assert "dq8_qgemm_variant" in hooks and "dq8_mfma_probe" in hooks
    public = set()
    for h in os.listdir(os.path.join(ROOT, "include")):
        public |= set(_declared(h))
    assert not public & set(hooks)
    for name in hooks:
        assert hasattr(H, name), name
        assert not hasattr(L, name), name + " is exported by the product library"
    for name in public:
        assert hasattr(H, name), name
    out = subprocess.run(["nm", "-D", "--defined-only", _lib.LIB_PATH], capture_output=True,
                         text=True, check=True).stdout
    exported = {line.split()[-1] for line in out.splitlines() if line.strip()}
    extra = {e for e in exported if e not in public and e != "kMlirLoweredEntry"}
    assert not extra, sorted(extra)[:20]


def test_variant_table_and_version():
    from bladedisc_amd import kernels
    names = kernels.variant_names()
    assert names[0] == "generic" and len(names) >= 4


def test_missing_library_fails_loudly(monkeypatch, tmp_path):
    """No CPU fallback: without the built library every operator raises."""
    import pytest
    from bladedisc_amd import _lib
    monkeypatch.setattr(_lib, "_lib", None)
    monkeypatch.setattr(_lib, "LIB_PATH", str(tmp_path / "libdisc_q8_ral.so"))
    with pytest.raises(RuntimeError, match="no CPU fallback"):
        _lib.lib()
    monkeypatch.setattr(_lib, "_hooks", None)
    monkeypatch.setattr(_lib, "HOOKS_LIB_PATH", str(tmp_path / "libdisc_q8_testhooks.so"))
    from bladedisc_amd import kernels
    with pytest.raises(RuntimeError, match="no CPU fallback"):
        kernels.variant_names()
    with pytest.raises(RuntimeError, match="no CPU fallback"):
        kernels.qlinear_f32_fused_max_rows(768, 768)


def test_the_libraries_build_without_python_headers(monkeypatch, tmp_path, capsys):
    """A machine without Python's headers still gets the C ABI and RAL libraries; the native
    callers are left out, by name, and nothing of an earlier build of them is touched."""
    import sysconfig

    import pytest
    from bladedisc_amd import build as b
    paths = dict(sysconfig.get_paths(), include=str(tmp_path))
    monkeypatch.setattr(sysconfig, "get_paths", lambda *a, **k: paths)
    with pytest.raises(RuntimeError, match="Python.h"):
        b.build_torch_calls()
    # (nothing to compile: the objects and libraries that are there pass for new ones)
    monkeypatch.setattr(b, "_compile", lambda *a, **k: (b.EXPORTS, ""))
    monkeypatch.setattr(b, "sources", lambda: [b.EXPORTS])
    for name in ("LIB", "HOOKS_LIB"):
        lib = tmp_path / name
        lib.write_bytes(b"")
        monkeypatch.setattr(b, name, str(lib))
    monkeypatch.setattr(b, "OBJ", str(tmp_path / "build"))
    assert b.build() == b.LIB
    assert "Python.h" in capsys.readouterr().err


def test_native_callers_of_another_torch_are_not_loaded(monkeypatch):
    """The module is on torch's C++ ABI: one that was built for another torch (or interpreter) is
    not found, instead of being loaded and going wrong somewhere."""
    import pytest
    import torch
    from bladedisc_amd import _lib
    assert torch.__version__ in os.path.basename(_lib.torch_calls_path())
    assert _lib.torch_calls().qgemm
    monkeypatch.setattr(torch, "__version__", "9.9.9")
    with pytest.raises(RuntimeError, match="9.9.9.*build it for this torch"):
        _lib.torch_calls()
