"""Which kernels the host code launches for a call, without a GPU: runs a few
lines against libhelio_hip.so in a child process where tests/hip_stub.c stands
in for the HIP runtime."""
import json
import subprocess
import sys
import tempfile
from pathlib import Path

ROOT = Path(__file__).resolve().parent.parent

PRELUDE = r"""
import ctypes as C, json, re, sys
stub = C.CDLL(sys.argv[1], mode=C.RTLD_GLOBAL)
stub.stub_log.restype = C.c_char_p
stub.stub_reset.argtypes = [C.c_size_t]
stub.stub_largest.restype = C.c_size_t
sys.path.insert(0, sys.argv[2])
import numpy as np
from helio_amd import abi, synth
from helio_amd.batch import BatchPlan, BatchView
from helio_amd.device import Context, DeferredLightPass, LightCullPass, upload_scene

ctx = Context(0)
NO_LIMIT = 2**64 - 1
result = []

def calls(f, limit=NO_LIMIT):
    '''[(kernel, template values, blocks)] that f launches, allocations of more than limit bytes failing.'''
    stub.stub_reset(limit)
    f()
    out = []
    for line in stub.stub_log().decode().splitlines():
        what, name, blocks = line.split()
        if what == "launch":
            m = re.match(r"_ZN2hl\d+(k_\w+?)(?:I((?:L[a-z]\d+E)+)E)?(?:Ev|E)", name)
            vals = [int(v) for v in re.findall(r"L[a-z](\d+)E", m.group(2))] if m.group(2) else []
            out.append((m.group(1), vals, int(blocks)))
    stub.stub_reset(NO_LIMIT)
    return out

def scene(n, w, h):
    return synth.make_scene("c2_1080p_1k", width=w, height=h, num_lights=n)

def cull_pass(sc, grid=None, pool_cap=1 << 16):
    ds = upload_scene(ctx, sc)
    clusters = synth.cluster_params(ctx.lib, sc, grid=grid) if grid else None
    cull = LightCullPass(ctx, sc.width, sc.height, clusters=clusters, pool_cap=pool_cap)
    cull.prepare(ds)
    return ds, cull
"""


def routes(script: str):
    """What the script's `result` holds at its end."""
    with tempfile.TemporaryDirectory() as d:
        so = Path(d) / "libhip_stub.so"
        subprocess.run(["gcc", "-O1", "-shared", "-fPIC", "-Wall", "-Wextra", "-Werror",
                        str(ROOT / "tests" / "hip_stub.c"), "-o", str(so)], check=True)
        prog = Path(d) / "prog.py"
        prog.write_text(PRELUDE + script + "\nprint('RESULT ' + json.dumps(result), flush=True)\n")
        r = subprocess.run([sys.executable, str(prog), str(so), str(ROOT)], capture_output=True, text=True,
                           timeout=600)
    assert r.returncode == 0, r.stdout[-2000:] + r.stderr[-4000:]
    return json.loads(r.stdout.split("RESULT ", 1)[1])
