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
