"""Error and bookkeeping paths of the library's host code, run without a GPU: its
HIP sources are compiled for the host alone and linked against a stand-in runtime
that can refuse a chosen call (tests/native/host_paths.hip)."""
import glob
import os
import subprocess

import pytest

from conftest import ROOT

HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")


@pytest.fixture(scope="module")
def host_paths(tmp_path_factory):
    if not os.path.exists(HIPCC):
        pytest.skip("hipcc is not available")
    d = tmp_path_factory.mktemp("host_paths")
    csrc = os.path.join(ROOT, "cvc_amd", "csrc")
    part = ("dslash.hip", "solver.hip")   # included by the program
    srcs = [s for s in glob.glob(os.path.join(csrc, "*.hip")) if os.path.basename(s) not in part]
    srcs.append(os.path.join(ROOT, "tests", "native", "host_paths.hip"))
    objs = [str(d / (os.path.basename(s) + ".o")) for s in srcs]
    flags = ["--cuda-host-only", "-O1", "-g", "-std=c++17", "-fPIC", f"-I{ROOT}/include"]
    procs = [subprocess.Popen([HIPCC, *flags, "-c", s, "-o", o], stdout=subprocess.PIPE, stderr=subprocess.STDOUT)
             for s, o in zip(srcs, objs)]
    for p in procs:
        out = p.communicate(timeout=300)[0].decode(errors="replace")
        assert p.returncode == 0, out[-3000:]
    # the device code that the objects name is not there
    nm = subprocess.run(["nm", "-u", *objs], check=True, capture_output=True, text=True).stdout.split()
    stub = d / "device_code.c"
    stub.write_text("".join(f"char {n}[16];\n" for n in sorted({w for w in nm if w.startswith("__hip_fatbin")})))
    exe = d / "host_paths"
    r = subprocess.run(["gcc", "-c", str(stub), "-o", str(d / "device_code.o")], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    r = subprocess.run(["g++", *objs, str(d / "device_code.o"), "-o", str(exe), "-lpthread"], capture_output=True,
                       text=True)
    assert r.returncode == 0, r.stderr[-3000:]
    return exe


@pytest.mark.parametrize("scenario", ["scratch", "solver_buffers", "refused_calls", "refused_host_memory",
                                      "streamed_conn", "one_by_one", "unconverged_source", "counted_applications",
                                      "column_extents", "block_lanes", "march_rule"])
def test_host_path(host_paths, scenario):
    r = subprocess.run([str(host_paths), scenario], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0 and r.stdout.endswith("ok\n"), (r.returncode, r.stdout[-2000:], r.stderr[-2000:])
