"""The extension with the native checks loads under the Python and torch it was built for; without it Python does every call."""

import subprocess
import sys

import pytest


def test_without_the_extension_the_library_loads(monkeypatch):
    import nunchaku_rocm_amd
    from nunchaku_rocm_amd import _lib

    monkeypatch.setattr(_lib, "_host", None)
    monkeypatch.setattr(_lib, "_lib", None)
    monkeypatch.delattr(nunchaku_rocm_amd, "_host", raising=False)
    monkeypatch.setitem(sys.modules, "nunchaku_rocm_amd._host", None)  # as if there were no such file
    with pytest.warns(RuntimeWarning, match="_host.so is missing"):
        assert _lib.load().svdq_abi_version() == _lib.ABI_VERSION
    host = _lib.host()
    assert host.same_source((), None) is None
    assert not any(getattr(host, name)(1, 2) for name in ("quantize_buffers", "quantize", "gemm", "gemv", "attention"))


@pytest.mark.parametrize("version", [None, "2.9.1+rocm7.0", "2.10.0"])
def test_another_torch_is_refused(version):
    import torch

    assert version != torch.__version__
    code = "import warnings, torch\n" + (f"torch.__version__ = {version!r}\n" if version else "") + (
        "from nunchaku_rocm_amd import _lib\n"
        "with warnings.catch_warnings(record=True) as w:\n"
        "    warnings.simplefilter('always')\n"
        "    host = _lib.host()\n"
        "print(host is _lib._NoHost, [str(x.message) for x in w if 'built for torch' in str(x.message)] != [])\n"
    )  # fmt: skip
    out = subprocess.run([sys.executable, "-c", code], capture_output=True, text=True, check=True, timeout=300)
    assert out.stdout.split() == ([str(version is not None)] * 2), out
