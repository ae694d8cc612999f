"""Host-side GEMM plans for the tests: builds tests/gemm_plan.cpp against the library and asks it."""
import collections
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PKG = os.path.join(ROOT, "thinksound-native_amd")
STORE, RESID, QKV, SWIGLU, SNAKE, RSNAKE = range(6)

# Sizes at which the GPU tests run the one-round hi|lo kernel, with the tile rows and K splits that the plans have
# there (asserted in test_gemm_plan.py). Launcher GEMMs: rows around the edges of every tile height, one K step to
# 17, and K splits.
STORE_ROWS = [(1, 32), (31, 32), (33, 32), (256, 32), (257, 64), (320, 64), (321, 64), (512, 64), (513, 96), (575, 96),
              (577, 96), (768, 96), (769, 128), (895, 128), (897, 128), (1024, 128)]   # rows, height at 4096 columns
STORE_KS = [64, 128, 192, 1088]
STORE_OTHER = [(1, 8, 64, 32, 1), (33, 8, 64, 32, 1), (31, 136, 1088, 32, 4), (129, 136, 1088, 32, 4),   # M, N, K,
               (31, 1024, 4096, 32, 16), (65, 1024, 4096, 64, 16), (97, 1024, 4096, 32, 8), (129, 1024, 4096, 32, 6),
               (300, 1024, 4096, 64, 6)]                                                 # height, splits
# The reference graph's fused block (H = 1024, F = 2816): latent rows -> tile rows of QKV, SwiGLU, output projection and
# second FFN layer; 0: the kernels of grids past one round
REF_ROWS = {150: (32, 32, 32, 96), 314: (32, 64, 32, 64), 470: (64, 96, 32, 96), 622: (64, 128, 32, 128),
            902: (96, 0, 32, 128), 1202: (128, 0, 64, 128), 1302: (0, 0, 64, 96)}

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
