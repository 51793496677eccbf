"""CPU checks through native test programs (tests/native/): the oracle and the C-ABI op layer
(argument validation, kernel planning over a sweep of shapes) built with AddressSanitizer and
UndefinedBehaviorSanitizer. No GPU work: every call either fails validation before any HIP
call or only plans."""
import os
import shutil
import subprocess

import pytest

from helpers import ROOT

NATIVE = os.path.join(ROOT, "tests", "native")


def _build(target):
    r = subprocess.run(["make", "-C", NATIVE, target], capture_output=True, text=True, timeout=600)
    assert r.returncode == 0, r.stdout[-2000:] + r.stderr[-2000:]
    return os.path.join(NATIVE, target)


def _run_sanitized(path):
    env = dict(os.environ, ASAN_OPTIONS="detect_leaks=0:abort_on_error=0",
               UBSAN_OPTIONS="print_stacktrace=1")
    r = subprocess.run([path], capture_output=True, text=True, timeout=600, env=env)
    report = r.stdout + r.stderr
    assert "ERROR: AddressSanitizer" not in report, report[-4000:]
    assert "runtime error" not in report, report[-4000:]
    assert r.returncode == 0, report[-4000:]
    return r.stdout


def test_oracle_under_sanitizers():
    out = _run_sanitized(_build("_build/orc_selftest"))
    assert "all checks passed" in out


def test_c_abi_validation_under_sanitizers():
    if not os.path.exists(os.path.join(ROOT, "triton-rs_amd", "_build", "kernels_gemv.o")):
        pytest.fail("kernel objects missing: run __graft_entry__.build() first")
    out = _run_sanitized(_build("_build/abi_selftest"))
    assert "all checks passed" in out


def test_native_programs_link_every_kernel_object(tmp_path):
    """A kernel source added to the library needs no edit under tests/: the makefile takes whatever
    objects there are, and the build names its own, so that a makefile with an older list links."""
    for d in ("tests/native", "triton-rs_amd/_build", "triton-rs_amd/csrc", "include"):
        (tmp_path / d).mkdir(parents=True)
    for f in ("_build/api.o", "_build/hiprt.o", "_build/kernels_gemv.o", "_build/added_later.o",
              "csrc/api.cpp", "csrc/hiprt.cpp", "csrc/launch.h"):
        (tmp_path / "triton-rs_amd" / f).touch()
    (tmp_path / "include" / "w4a16.h").touch()
    for f in ("Makefile", "abi_selftest.cpp"):
        shutil.copy(os.path.join(NATIVE, f), tmp_path / "tests" / "native" / f)
    r = subprocess.run(["make", "-n", "-C", str(tmp_path / "tests" / "native"), "_build/abi_selftest"],
                       capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    link = [l for l in r.stdout.replace("\\\n", " ").splitlines() if " abi_selftest.cpp " in l][-1].split()
    objs = [os.path.basename(w) for w in link if w.endswith(".o") and "triton-rs_amd/_build" in w]
    assert sorted(objs) == ["added_later.o", "kernels_gemv.o"]

    import __graft_entry__ as entry
    module = entry._load_build_module()
    given = [a for a in entry.native_make_command(module) if a.startswith("KOBJ=")]
    names = {os.path.basename(o) for o in given[0][5:].split()}
    assert names == {os.path.splitext(s)[0] + ".o" for s in module.SOURCES} - {"api.o", "hiprt.o"}
