"""Host code under a full device memory, on the CPU: the library's host sources
are compiled with AddressSanitizer and linked with a device-less HIP runtime
(tests/native), and each scenario (the request server's admission, a crossover
plan's segments) runs in a process of its own."""
import os
import subprocess
from concurrent.futures import ThreadPoolExecutor

import pytest

from tests.conftest import ROOT

NATIVE = os.path.join(ROOT, "tests", "native")
CSRC = os.path.join(ROOT, "vectorta_amd", "csrc")
ROCM = os.environ.get("ROCM", "/opt/rocm")
PROGRAMS = ("server_admission", "cross_memory")
SOURCES = ["runtime", "alma", "rec", "rolling", "cross", "fir", "server", "dlpack", "graph", "tune"]


@pytest.fixture(scope="session")
def programs(tmp_path_factory):
    """{program: its path}"""
    out = tmp_path_factory.mktemp("native")
    flags = ["-O1", "-g", "-std=c++17", "-pthread", "-fsanitize=address", "-D__HIP_PLATFORM_AMD__",
             f"-I{ROCM}/include", f"-I{ROOT}/include", f"-I{CSRC}", f"-I{NATIVE}"]

    def compile_one(src):
        obj = str(out / (os.path.basename(src) + ".o"))
        subprocess.run(["g++", *flags, "-c", src, "-o", obj], check=True)
        return obj

    srcs = [os.path.join(CSRC, s + ".cpp") for s in SOURCES]
    srcs += [os.path.join(NATIVE, s) for s in ("fake_hip.cpp", *(p + ".cpp" for p in PROGRAMS))]
    with ThreadPoolExecutor(4) as pool:
        objs = list(pool.map(compile_one, srcs))
    common, mains = objs[:-len(PROGRAMS)], objs[-len(PROGRAMS):]
    for obj, name in zip(mains, PROGRAMS):
        subprocess.run(["g++", "-fsanitize=address", "-pthread", *common, obj, "-o",
                        str(out / name), "-ldl"], check=True)
    return {name: str(out / name) for name in PROGRAMS}


def _run(*command):
    # (another preloaded library may come before the sanitizer's)
    env = dict(os.environ, ASAN_OPTIONS="verify_asan_link_order=0:detect_leaks=0")
    r = subprocess.run(command, env=env, capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout + r.stderr


@pytest.mark.parametrize("scenario", ["hit_evicts_another", "hit_never_fits", "hit_served_as_miss",
                                      "hit_waits_for_release", "pack_of_hits",
                                      "fragmented_arena"])
def test_admission(programs, scenario):
    _run(programs["server_admission"], scenario)


def test_crossover_plan_takes_the_segments_that_fit(programs):
    _run(programs["cross_memory"])
