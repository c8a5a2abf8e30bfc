"""What the split GEMM's planner decides (tests/cpp/plan_query.cpp, built by
__graft_entry__.build(); no GPU)."""
import os
import subprocess

BIN = os.path.join(os.path.dirname(os.path.abspath(__file__)), "cpp", "plan_query")
LAYOUTS = ("NN", "NT", "TN")
CUS = 256  # compute units of an MI355X


def ask(*queries):
    """One answer a query, as text."""
    out = subprocess.run([BIN], input="".join(" ".join(map(str, q)) + "\n" for q in queries),
                         capture_output=True, text=True, timeout=60, check=True)
    return out.stdout.splitlines()


def built():
    return os.path.exists(BIN)


# Products that reach each tile of the split GEMM in every layout, ragged in
# rows, columns and depth and whole; test_gemm_plan.py holds them to it.
TILES = [  # rows, cols, inner, tile
    ((3559, 2933, 37), "256x256x16"), ((4096, 4096, 48), "256x256x16"),
    ((1466, 2125, 133), "128x128x32"), ((2048, 1920, 160), "128x128x32"),
    ((2191, 1377, 37), "64x128x32"), ((2048, 2048, 64), "64x128x32"),
    ((700, 650, 177), "64x64x64"), ((1024, 1024, 192), "64x64x64"),
    ((1000, 1333, 65), "64x64x32"), ((1024, 1536, 64), "64x64x32"),
]

# Layers whose forward and stride-1 input gradient reach the wide tiles of the
# split convolutions, with channels that are and are not whole k steps.
CONV_TILES = [  # n, c_in, c_out, h, w, kh, kw, stride, pad; forward and input gradient
    ((29, 68, 96, 23, 37, 3, 3, 1, 1), "128x128x32", "128x128x32"),
    ((50, 32, 65, 19, 26, 3, 3, 1, 1), "128x128x32", "-"),
    ((31, 68, 132, 34, 24, 1, 1, 1, 0), "64x128x32", "128x128x32"),
    ((13, 68, 96, 26, 25, 1, 1, 1, 0), "64x128x32", "64x128x32"),
    ((18, 64, 65, 24, 19, 1, 1, 1, 0), "64x128x32", "-"),
    ((20, 68, 40, 27, 17, 1, 1, 1, 0), "64x64x32", "64x128x32"),
    ((50, 36, 68, 21, 30, 1, 1, 2, 0), "64x128x32", "-"),
    ((1, 64, 40, 19, 25, 3, 3, 1, 1), "64x64x64", "-"),
    ((1, 36, 96, 23, 18, 3, 3, 1, 1), "-", "64x64x64"),
]
