"""When the operators' native host path (host/torch_ops.cpp) is used and when it is left alone.  No GPU."""
import sys
import sysconfig
import types

import pytest

torch = pytest.importorskip("torch")

import luminal_amd  # noqa: E402
from luminal_amd import build, capi, quantized  # noqa: E402


def operator_with(monkeypatch, module):
    """quantized's choice with `module` in the extension's place (None: its import fails)."""
    monkeypatch.setitem(sys.modules, "luminal_amd._torch_ops", module)
    if module is None:
        monkeypatch.delattr(luminal_amd, "_torch_ops", raising=False)
    else:
        monkeypatch.setattr(luminal_amd, "_torch_ops", module, raising=False)
    return quantized._native_operator()


def extension(**differs):
    built_for = {"torch_version": str(torch.__version__), "c_header": capi.header_digest(), **differs}
    return types.SimpleNamespace(quantized_matmul=lambda *_: "native", **{k: v for k, v in built_for.items() if v})


def test_an_extension_built_for_what_runs_is_used(monkeypatch):
    assert operator_with(monkeypatch, extension())() == "native"
    monkeypatch.setattr(capi, "HEADER", "/nonexistent")  # installed without the header: nothing to compare it with
    assert operator_with(monkeypatch, extension(c_header="0"))() == "native"


@pytest.mark.parametrize("module", [None, extension(torch_version="1.0"), extension(c_header="0"),
                                    extension(torch_version=None), extension(c_header=None)],
                         ids=["not built", "other torch", "other header", "no torch version", "no header"])
def test_any_other_leaves_the_calls_to_ctypes(monkeypatch, module):
    assert operator_with(monkeypatch, module)(torch.zeros(1), torch.zeros(1), 1, 1, False, 0, 0) is None


def test_the_extension_is_named_for_the_python_it_is_built_for():
    assert build.TORCH_OPS.endswith("_torch_ops" + sysconfig.get_config_var("EXT_SUFFIX"))
    assert sys.implementation.cache_tag.split("-")[1] in sysconfig.get_config_var("EXT_SUFFIX")


def test_the_built_extension_names_what_it_was_built_for():
    ops = pytest.importorskip("luminal_amd._torch_ops")
    assert (ops.torch_version, ops.c_header) == (str(torch.__version__), capi.header_digest())


@pytest.mark.parametrize("missing", ["torch", "Python's headers", "torch's headers"])
def test_the_build_goes_on_without_it_where_headers_are_missing(monkeypatch, tmp_path, missing):
    from torch.utils import cpp_extension

    stale = tmp_path / "_torch_ops.so"
    stale.write_bytes(b"an earlier build's")
    monkeypatch.setattr(build, "TORCH_OPS", str(stale))
    monkeypatch.setattr(build, "_run", lambda cmd: pytest.fail("compiled"))
    if missing == "torch":
        monkeypatch.setitem(sys.modules, "torch.utils", None)
    elif missing == "Python's headers":
        monkeypatch.setattr(build.sysconfig, "get_paths", lambda: {"include": str(tmp_path)})
    else:
        monkeypatch.setattr(cpp_extension, "include_paths", lambda: [str(tmp_path)])
    assert build.build_torch_ops(verbose=False) is None
    assert not stale.exists()  # (it would go with another library)
