"""Sources compiled at run time (sbz_compile, the route of sbz_model_create without a cached code
object): the code of a source does not depend on what the process compiled before it, the flags are
those of the ahead-of-time build, and a source that does not compile is an error with the log."""
import os
import re
import subprocess
import sys
from pathlib import Path

import pytest

from symboltz import _lib, build, models
from symboltz.solver import _declare, model_source

ROOT = Path(__file__).resolve().parent.parent

SCRIPT = """
import sys
sys.path.insert(0, sys.argv[1])
from symboltz import _lib, models
from symboltz.solver import _declare, model_source
L = _lib.lib()
_declare(L)
plain = b'extern "C" __global__ void k(double* p) { p[threadIdx.x] += 1.0; }'
if sys.argv[3] == "second":
    assert L.sbz_compile(plain, sys.argv[2].encode() + b".plain") == 0
assert L.sbz_compile(model_source(models.LCDM(lmax=5)).full_src.encode(), sys.argv[2].encode()) == 0
"""


def test_code_does_not_depend_on_what_the_process_compiled_before(tmp_path):
    """A source without kernels of one hierarchy per lane, compiled first, must not take the scalar
    register allocator's option from the model compiled after it."""
    model_source(models.LCDM(lmax=5))
    procs = [subprocess.Popen([sys.executable, "-c", SCRIPT, str(ROOT / "symboltz.jl_amd"), str(tmp_path / w), w],
                              env=dict(os.environ, AMD_COMGR_CACHE="0")) for w in ("first", "second")]
    assert [p.wait(timeout=600) for p in procs] == [0, 0]
    same = (tmp_path / "first").read_bytes() == (tmp_path / "second").read_bytes()
    assert same


def test_flags_are_those_of_the_ahead_of_time_build():
    src = (build.CSRC / "sbz_rtc.cpp").read_text()
    opts = re.findall(r'"([^"]*)"', re.search(r"opts\[\] = \{(.*?)\};", src, re.S).group(1))
    assert opts == build.KERNEL_FLAGS and opts[:-4] == build.HIP_FLAGS
    one = model_source(models.LCDM(lmax=5)).full_src
    assert build.kernel_flags(one) == build.KERNEL_FLAGS
    # another set of flags is another code object
    assert build.code_hash(one) == model_source(models.LCDM(lmax=5)).full_hash
    assert build.code_hash(one) != build.code_hash(one.replace("\n#define SBZ_GROUP_OK 1\n", "\n#define SBZ_GROUP_OK 0\n"))


def test_what_a_preloaded_library_prints_is_not_in_the_code(tmp_path, monkeypatch):
    (tmp_path / "p.c").write_text("""#include <unistd.h>
__attribute__((constructor)) static void hello(void) { if (write(1, "hello\\n", 6) < 0) _exit(9); }
""")
    subprocess.run(["gcc", "-shared", "-fPIC", str(tmp_path / "p.c"), "-o", str(tmp_path / "p.so")], check=True)
    L = _lib.lib()
    _declare(L)
    src = b'extern "C" __global__ void k(double* p) { p[threadIdx.x] += 1.0; }'
    assert L.sbz_compile(src, str(tmp_path / "a").encode()) == 0
    monkeypatch.setenv("LD_PRELOAD", f"{os.environ.get('LD_PRELOAD', '')} {tmp_path / 'p.so'}".strip())
    assert L.sbz_compile(src, str(tmp_path / "b").encode()) == 0
    assert (tmp_path / "a").read_bytes() == (tmp_path / "b").read_bytes()


def test_a_source_that_does_not_compile_is_an_error(tmp_path):
    L = _lib.lib()
    _declare(L)
    with pytest.raises(_lib.SbzError, match="no_such_type"):
        _lib.check(L.sbz_compile(b"no_such_type x;", str(tmp_path / "x").encode()), "sbz_compile")
    assert not (tmp_path / "x").exists()
