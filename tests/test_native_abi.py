"""The native module and the library it is bound to (on the CPU)."""
import os
import re
import subprocess

import pytest

from bitsparse_amd import _lib
from bitsparse_amd.build import INCLUDE


def _header_version():
    with open(os.path.join(INCLUDE, "bitsparse_hip.h")) as f:
        return int(re.search(r"#define BS_ABI_VERSION (\d+)", f.read()).group(1))


def test_one_version():
    assert _header_version() == _lib.ABI_VERSION == _lib.load().bs_abi_version()
    assert _lib.native().EPOCH_LIMIT == _lib._EPOCH_LIMIT


def test_library_of_another_version_is_refused(tmp_path):
    """_native is compiled against the header, the library may be another
    build: with other signatures its calls would get shifted arguments."""
    src, so = tmp_path / "other.cpp", tmp_path / "other.so"
    names = sorted(set(re.findall(r"\b(bs_[a-z0-9_]+)\(", open(os.path.join(INCLUDE, "bitsparse_hip.h")).read())))
    src.write_text("".join(f'extern "C" int {n}() {{ return {_lib.ABI_VERSION + 1}; }}\n' for n in names))
    subprocess.run(["g++", "-shared", "-fPIC", str(src), "-o", str(so)], check=True)
    native = _lib.native()
    try:
        with pytest.raises(ImportError, match="ABI"):
            native.init(str(so))
        assert native.abi_version() == _lib.ABI_VERSION          # still bound to the library it had
    finally:
        native.init(_lib.LIB_PATH)


@pytest.mark.parametrize("status,error", [(_lib.BS_OK, None), (_lib.BS_ERR_INVALID, ValueError),
                                          (2, _lib.BitsparseHipError)])
def test_errors_of_native_calls(status, error):
    """The native calls raise what the Python ones raise for the same status."""
    native = _lib.native()
    for check in (_lib.check, native.check):
        if error is None:
            check(status, "bs_compress")
            continue
        with pytest.raises(Exception) as e:
            check(status, "bs_compress")
        assert type(e.value) is error and str(e.value).startswith("bs_compress")
