"""The native launch path (csrc/launch.cpp) does what the Python functions of _lib.py do, and hands them what it does not take.  No GPU: device and stream are stood in for, the entry
points are asked for what they refuse on the host."""
import importlib.machinery
import os
import shutil
import subprocess
import sys
import sysconfig
import threading

import pytest
import torch

from llm_quest_amd import _lib

launch = _lib._launch
if launch is None and not (shutil.which("g++") and os.path.exists(os.path.join(sysconfig.get_paths()["include"], "Python.h"))):
    pytest.skip("no compiler or headers to build the extension with", allow_module_level=True)  # (with them a missing or broken extension fails below)
BAD_FORM = (7, 1, 1, 8, None, 8, None, 8, None, 8, 0, None, None, 0, 0, None, 0, 0)


class Fake:
    """A tensor as far as the launch path looks."""

    def __init__(self, index, address=4096):
        self.index, self.address, self.is_cuda, self.device = index, address, index >= 0, torch.device("cuda", index) if index >= 0 else torch.device("cpu")

    def get_device(self):
        return self.index

    def data_ptr(self):
        return self.address


@pytest.fixture
def slow():
    """Calls that reach the Python forms are recorded; device 0 is current, its stream is the null stream."""
    got = []
    _lib.load()
    launch.setup(lambda: 0, lambda i: 0, lambda *a: got.append(a), lambda *t: got.append(t), _lib._fail)
    yield got
    launch.setup(torch._C._cuda_getDevice, torch._C._cuda_getCurrentRawStream, _lib._python_call, _lib._python_require_gpu, _lib._fail)
    launch.set_device(-1)


def test_every_entry_point_of_the_binding_is_known():
    assert sorted(launch.names()) == sorted(_lib.SIGNATURES)


def test_a_call_reaches_the_library_and_its_error_comes_back(slow):
    launch.require_gpu(Fake(0))
    with pytest.raises(RuntimeError, match=r"mi355_gemm_bf16 failed \(rc=1\).*bad form"):
        launch.call("mi355_gemm_bf16", *BAD_FORM)
    # pointers as integers, floats from integers and floats, 64-bit integers whole
    with pytest.raises(RuntimeError, match=r"head_dim must|head_dim"):
        launch.call("mi355_attn_fwd", 1, 4, 2, 1, 96, 4096, 0, None, 0, None, 0, None, 0, None, None, True, 1)
    with pytest.raises(RuntimeError, match=r"rc="):
        launch.call("mi355_zc_weight", -(1 << 40), 4096, 4096)
    assert not slow


@pytest.mark.parametrize("args", [BAD_FORM[:-1], BAD_FORM + (0,), (7.0,) + BAD_FORM[1:], BAD_FORM[:4] + ("x",) + BAD_FORM[5:]])
def test_what_does_not_convert_goes_to_python(slow, args):
    launch.require_gpu(Fake(0))
    launch.call("mi355_gemm_bf16", *args)
    assert slow == [("mi355_gemm_bf16",) + args]


def test_other_devices_and_unknown_names_go_to_python(slow):
    launch.require_gpu(Fake(1), None)
    assert launch.device() == 1
    launch.call("mi355_gemm_bf16", *BAD_FORM)  # device 1 is not the current one
    launch.require_gpu(None)
    assert launch.device() == -1
    launch.call("mi355_gemm_bf16", *BAD_FORM)  # no operand said where
    launch.require_gpu(Fake(0))
    launch.call("mi355_no_such_entry", 1)
    assert [a[0] for a in slow] == ["mi355_gemm_bf16"] * 2 + ["mi355_no_such_entry"]


def test_operands_off_the_gpu_or_on_two_go_to_python(slow):
    a, b, c = Fake(0), Fake(1), Fake(-1)
    launch.require_gpu(a, b)
    launch.require_gpu(None, c)
    assert slow == [(a, b), (None, c)]
    with pytest.raises(RuntimeError, match="no CPU fallback"):
        _lib._python_require_gpu(torch.zeros(2))
    with pytest.raises(RuntimeError, match="different devices"):
        _lib._python_require_gpu(a, b)
    assert launch.ptr(None) is None and launch.ptr(Fake(0, 77)) == 77


def test_the_device_belongs_to_the_thread(slow):
    launch.require_gpu(Fake(0))
    seen = []
    t = threading.Thread(target=lambda: (seen.append(launch.device()), launch.set_device(3)))
    t.start()
    t.join()
    assert seen == [-1] and launch.device() == 0


def _sources(tmp_path):
    """The extension's part of the source tree, built nowhere yet."""
    root = os.path.dirname(os.path.dirname(os.path.abspath(_lib.__file__)))
    for f in ("llm_quest_amd/csrc/launch.cpp", "llm_quest_amd/csrc/Makefile", "llm_quest_amd/_lib.py", "include/mi355_vlm.h"):
        (tmp_path / f).parent.mkdir(parents=True, exist_ok=True)
        shutil.copy(os.path.join(root, f), tmp_path / f)
    (tmp_path / "llm_quest_amd" / "__init__.py").touch()
    return tmp_path / "llm_quest_amd"


@pytest.mark.parametrize("target", ["all", "serve"])
@pytest.mark.parametrize("compiler", ["g++", "false"])
def test_the_library_builds_without_the_extension(tmp_path, target, compiler):
    """A host compiler that fails costs the extension, not the build; one that works leaves a file that no other interpreter takes, and none that any would take."""
    package = _sources(tmp_path)
    (package / "_launch.so").touch()
    have = ["-o", "../libmi355vlm.so", "-o", "../libmi355serve.so"]  # the libraries count as built
    for lib in have[1::2]:
        (package / "csrc" / lib).touch()
    done = subprocess.run(["make", "-C", str(package / "csrc"), "PYTHON=" + sys.executable, "CXX=" + compiler, *have, target], capture_output=True, text=True)
    assert done.returncode == 0, done.stderr
    built = sorted(p.name for p in package.glob("_launch*"))
    assert built == (["_launch" + importlib.machinery.EXTENSION_SUFFIXES[0]] if compiler == "g++" else [])


def test_an_extension_that_does_not_load_is_said(tmp_path):
    package = _sources(tmp_path)
    (package / ("_launch" + importlib.machinery.EXTENSION_SUFFIXES[0])).write_bytes(b"not a library")
    done = subprocess.run([sys.executable, "-c", "from llm_quest_amd import _lib; assert _lib._launch is None and _lib.call is _lib._python_call"], cwd=tmp_path, capture_output=True, text=True)
    assert done.returncode == 0 and "does not load" in done.stderr, done.stderr
