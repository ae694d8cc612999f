"""Host-side GEMM plans for the tests: builds tests/gemm_plan.cpp against the library and asks it."""
import collections
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PKG = os.path.join(ROOT, "thinksound-native_amd")
STORE, RESID, QKV, SWIGLU, SNAKE, RSNAKE = range(6)

Plan = collections.namedtuple("Plan", "kernel height sk splits tiles")


def build(out_dir):
    exe = os.path.join(str(out_dir), "gemm_plan")
    subprocess.run(["/opt/rocm/bin/hipcc", "--offload-arch=gfx950", "-std=c++17", "-O1", "-Xclang", "-target-feature",
                    "-Xclang", "-packed-fp32-ops", "-x", "hip", os.path.join(ROOT, "tests", "gemm_plan.cpp"),
                    "-I" + os.path.join(PKG, "csrc"), "-I" + os.path.join(ROOT, "include"), "-o", exe,
                    "-L" + os.path.join(PKG, "lib"), "-ltsn", "-Wl,-rpath," + os.path.join(PKG, "lib")],
                   check=True, capture_output=True, text=True)
    return exe


def ask(exe, epi, probs, ws=40 << 20, pair=0, half=1, split_waves=0, counters=1 << 16):
    """Plan of a batch of (M, N, K, taps[, half, pair]) problems; height: rows of a tile of the one-round hi|lo kernel, or 0."""
    line = "%d %d %d %d %d" % (epi, ws, split_waves, counters, len(probs))
    for p in probs:
        line += " %d %d %d %d %d %d" % (tuple(p) + (half, pair)[len(p) - 4:])
    r = subprocess.run([exe], input=line + "\n", capture_output=True, text=True, check=True)
    rc, name, hl2, sk, splits, tiles = r.stdout.split("\n")[0].rsplit(" ", 5)
    assert rc == "0", r.stdout
    return Plan(name, 16 * int(hl2), int(sk), int(splits), int(tiles))
