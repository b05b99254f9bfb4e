"""Device allocations and staged host copies (hostio.hpp) on the CPU, against a
fake HIP runtime: tests/native/hostio_check.cpp, built host-only."""
import glob
import os
import re
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "welvet.metal_amd", "csrc")
OUT = os.path.join(ROOT, "welvet.metal_amd", "_build", "hostio")
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")


def _run(cmd, **kw):
    r = subprocess.run(cmd, capture_output=True, text=True, **kw)
    assert r.returncode == 0, f"{' '.join(cmd)}\n{r.stdout[-4000:]}\n{r.stderr[-4000:]}"
    return r


def test_pool_gives_way_and_copies_are_whole():
    src = os.path.join(ROOT, "tests", "native", "hostio_check.cpp")
    exe = os.path.join(OUT, "hostio_check")
    deps = [src] + glob.glob(os.path.join(CSRC, "*.hpp"))
    if not (os.path.exists(exe) and os.path.getmtime(exe) > max(os.path.getmtime(d) for d in deps)):
        os.makedirs(OUT, exist_ok=True)
        obj = exe + ".o"
        _run([HIPCC, "-x", "hip", "--offload-host-only", "-fgpu-rdc", "-std=c++17", "-O2", "-ffp-contract=off",
              "-I", CSRC, "-c", src, "-o", obj])
        _run([HIPCC, "-fgpu-rdc", "--offload-arch=gfx950", obj, "-o", exe, "-lpthread"])
    r = _run([exe], timeout=120)
    assert "hostio_check: ok" in r.stdout, r.stdout[-2000:]


def test_every_device_allocation_can_have_the_pool():
    """hipMalloc is called in one place: the function that gives the pool's
    idle blocks back when memory runs out."""
    calls = []
    for f in glob.glob(os.path.join(CSRC, "*")):
        with open(f) as s:
            calls += [os.path.basename(f) for line in s
                      if re.search(r"\bhipMalloc\(", line.split("//")[0])]
    assert set(calls) == {"hostio.hpp"} and len(calls) == 2, calls
