"""The split-x GEMM's plans and the kernels that serve them, on the CPU:
tests/native/plans_check.cpp, built host-only."""
import glob
import os
import re
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "welvet.metal_amd", "csrc")
OUT = os.path.join(ROOT, "welvet.metal_amd", "_build", "plans")
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")


def _run(cmd, **kw):
    r = subprocess.run(cmd, capture_output=True, text=True, **kw)
    assert r.returncode == 0, f"{' '.join(cmd)}\n{r.stdout[-4000:]}\n{r.stderr[-4000:]}"
    return r


def _built():
    """The check and its object."""
    src = os.path.join(ROOT, "tests", "native", "plans_check.cpp")
    exe = os.path.join(OUT, "plans_check")
    obj = exe + ".o"
    deps = [src, os.path.join(CSRC, "dense.hip")] + glob.glob(os.path.join(CSRC, "*.hpp"))
    if not (os.path.exists(exe) and os.path.getmtime(exe) > max(os.path.getmtime(d) for d in deps)):
        os.makedirs(OUT, exist_ok=True)
        _run([HIPCC, "-x", "hip", "--offload-host-only", "-fgpu-rdc", "-std=c++17", "-O1", "-ffp-contract=off",
              "-I", CSRC, "-c", src, "-o", obj])
        _run([HIPCC, "-fgpu-rdc", "--offload-arch=gfx950", obj, "-o", exe])
    return exe, obj


def test_every_plan_has_its_kernel_and_every_kernel_a_plan():
    exe, obj = _built()
    symbols = _run(["nm", obj]).stdout
    kernels = set(re.findall(r"__device_stub__gemm_bf3[sk]?_kernel\w*", symbols))
    r = subprocess.run([exe, str(len(kernels))], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0 and "plans_check: ok" in r.stdout, r.stdout[-2000:]


def test_plans_of_the_edge_shapes():
    """The shapes whose results test_gpu_split_tiles.py checks run the kernels
    that the table says."""
    import split_shapes as S
    exe = _built()[0]
    wrong = []
    for out, inn, batch, single, pair in S.SHAPES:
        for p, plans in ((0, single), (1, pair)):
            for kind, want in plans.items():
                got = _run([exe, "plan", str(kind), str(batch), str(out), str(inn), str(p)]).stdout.strip()
                if got != want:
                    wrong.append((out, inn, batch, p, kind, got, want))
    assert not wrong, wrong
