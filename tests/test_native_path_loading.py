"""Loading the native call path (CPU): a missing, broken or foreign extension leaves the library and its Python calls usable."""

import os
import shutil
import subprocess
import sys

import pytest

from moespresso_amd import _lib

pytestmark = pytest.mark.skipif(not (os.path.exists(_lib.LIB_PATH) and os.path.exists(_lib.DISPATCH_PATH)),
                                reason="the library is not built")

CHECK = """
import warnings
import torch
if {version!r}:
    torch.__version__ = {version!r}
with warnings.catch_warnings(record=True) as seen:
    warnings.simplefilter("always")
    from moespresso_amd import _lib
assert _lib.library_available()
assert _lib.lib().mspr_abi_version() > 0
native = not isinstance(_lib.dispatch, _lib._NoNativePath)
assert native or _lib.dispatch.topk_select(None, 1) is None
from moespresso_amd.runtime.qwen import kquant
print(native, [str(w.message) for w in seen if "native call path" in str(w.message)])
"""


def _load(tmp_path, extension, version=None):
    root = os.path.dirname(_lib.LIB_PATH)
    shutil.copytree(root, tmp_path / "moespresso_amd", ignore=shutil.ignore_patterns("_obj", "__pycache__", "csrc", "_dispatch.so"))
    target = tmp_path / "moespresso_amd" / "_dispatch.so"
    if extension == "built":
        shutil.copy(_lib.DISPATCH_PATH, target)
    elif extension == "broken":
        target.write_bytes(b"not a shared object")
    run = subprocess.run([sys.executable, "-c", CHECK.format(version=version)], cwd=tmp_path, capture_output=True, text=True,
                         env={**os.environ, "PYTHONPATH": str(tmp_path)})
    assert run.returncode == 0, run.stderr
    return run.stdout


def test_the_extension_of_this_torch_is_taken(tmp_path):
    assert _load(tmp_path, "built").startswith("True []")


@pytest.mark.parametrize("extension,version,says", [("missing", None, "is missing"), ("broken", None, "cannot be loaded"),
                                                    ("built", "1.2.3", "it was built for torch")])
def test_without_it_the_library_is_called_from_python(tmp_path, extension, version, says):
    out = _load(tmp_path, extension, version)
    assert out.startswith("False ") and says in out
