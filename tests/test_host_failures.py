"""The library's host code on a HIP runtime without a device
(tests/host_checks): what a prompt leaves behind when one of its allocations,
launches or copies fails."""
import os
import subprocess
from concurrent.futures import ThreadPoolExecutor

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
RUNTIME = os.path.join(ROOT, "ai-research_amd", "csrc", "runtime")


@pytest.fixture(scope="session")
def checks(tmp_path_factory):
    """The check program and the folder its stand-in code object lies in."""
    out = tmp_path_factory.mktemp("host_checks")
    here = os.path.join(ROOT, "tests", "host_checks")
    sources = [os.path.join(RUNTIME, s + ".cpp") for s in ("runtime", "engine", "model", "ring")]
    sources += [os.path.join(here, s) for s in ("fake_hip.cpp", "checks.cpp")]
    rocm = os.environ.get("ROCM_PATH", "/opt/rocm")

    def compile_one(src):
        obj = str(out / (os.path.basename(src) + ".o"))
        subprocess.run(["g++", "-O1", "-g", "-std=c++17", "-pthread", "-D__HIP_PLATFORM_AMD__", "-w",
                        "-I", os.path.join(rocm, "include"), "-I", os.path.join(ROOT, "include"),
                        "-I", os.path.dirname(RUNTIME), "-c", src, "-o", obj], check=True)
        return obj

    with ThreadPoolExecutor(4) as ex:
        objs = list(ex.map(compile_one, sources))
    exe = str(out / "checks")
    subprocess.run(["g++", "-pthread", *objs, "-ldl", "-o", exe], check=True)
    (out / "gh_gemv.hsaco").write_bytes(b"")
    return exe, str(out)


# (tokens, clock of the first, head dim, lists given by the caller, buffers of an
# earlier prompt there): a new ring, whose batch writes its slots directly; a
# wrapped one, whose batch is staged, in one part and in several (24 staging
# rows); the per-token, 4-token and matrix-core attention's lists
CASES = [(12, 0, 64, 0, 1), (12, 0, 64, 0, 0), (12, 30, 64, 0, 1), (40, 30, 64, 0, 1), (20, 0, 64, 1, 1),
         (12, 30, 64, 1, 1), (20, 0, 256, 0, 1), (80, 30, 256, 0, 1)]


@pytest.mark.parametrize("kind", ["new", "launch", "copy"])
@pytest.mark.parametrize("case", CASES, ids=lambda c: "-".join(map(str, c)))
def test_failed_prompts(checks, kind, case):
    exe, folder = checks
    r = subprocess.run([exe, folder, "failures", kind, *map(str, case)], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stdout[-3000:] + r.stderr[-1000:]
    assert int(r.stdout.split()[0]) > 5, r.stdout  # so many calls were there to fail
