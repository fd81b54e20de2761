"""Loading of the native functions behind the package (mops_amd/lib/_array_ops.so): where the file cannot be
loaded, `import mops_amd` says so and goes through ctypes. In processes of their own; no GPU needed."""
import os
import shutil
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROBE = """
import sys, warnings
with warnings.catch_warnings(record=True) as caught:
    warnings.simplefilter("always")
    import mops_amd
    from mops_amd import _c_lib, ops
native = not isinstance(ops._native, _c_lib._NoFunctions)
said = [str(w.message) for w in caught if "_array_ops.so" in str(w.message)]
print("native" if native else "ctypes", len(said), *said)
"""


def package(tmp_path, array_functions):
    """A copy of the package's Python files, with `array_functions` as its _array_ops.so."""
    target = tmp_path / "mops_amd"
    shutil.copytree(os.path.join(ROOT, "mops_amd"), target, ignore=shutil.ignore_patterns("csrc", "lib", "__pycache__"))
    (target / "lib").mkdir()
    library = os.path.join(ROOT, "mops_amd", "lib", "libmops.so")
    if os.path.exists(library):
        os.symlink(library, target / "lib" / "libmops.so")
    if array_functions is not None:
        (target / "lib" / "_array_ops.so").write_bytes(array_functions)


def imported(tmp_path, probe=PROBE, **environment):
    done = subprocess.run(
        [sys.executable, "-c", probe], cwd=str(tmp_path), env=dict(os.environ, **environment), capture_output=True, text=True
    )
    assert done.returncode == 0, done.stdout + done.stderr
    return done.stdout


def foreign_extension(tmp_path):
    """A shared object that asks for a symbol nobody has, as one built for another PyTorch does."""
    source = tmp_path / "foreign.c"
    source.write_text("extern void symbol_of_another_pytorch(void);\nvoid* PyInit__array_ops(void) { symbol_of_another_pytorch(); return 0; }\n")
    target = tmp_path / "foreign.so"
    subprocess.run(["gcc", "-shared", "-fPIC", "-Wl,-z,now", "-o", str(target), str(source)], check=True)
    return target.read_bytes()


@pytest.mark.parametrize("content", ["not a library", "foreign"])
def test_a_file_that_does_not_load_is_reported_and_left_out(tmp_path, content):
    package(tmp_path, b"not a shared object" if content == "not a library" else foreign_extension(tmp_path))
    assert imported(tmp_path).startswith("ctypes 1 ")


def test_without_pytorch_the_package_is_importable(tmp_path):
    """(as before there were native functions: only a call needs PyTorch)"""
    package(tmp_path, b"never looked at")
    without = "import sys\nsys.modules['torch'] = None\n"
    assert imported(tmp_path, without + PROBE).startswith("ctypes 0")


def test_nothing_is_said_where_there_is_no_file_or_ctypes_is_asked_for(tmp_path):
    package(tmp_path, None)
    assert imported(tmp_path).startswith("ctypes 0")
    (tmp_path / "mops_amd" / "lib" / "_array_ops.so").write_bytes(b"not a shared object")
    assert imported(tmp_path, MOPS_AMD_ARRAY_PYTHON="1").startswith("ctypes 0")
