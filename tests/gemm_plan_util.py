"""The tile planner of the prompt GEMMs (cccc-lite_amd/csrc/gemm_plan.h, host arithmetic) behind a C window, compiled on first use."""
import ctypes
import subprocess
import tempfile
from pathlib import Path

LINEAR, PAIR, SEGMENTS = 0, 1, 2

SOURCE = r"""
#include "gemm_plan.h"
using namespace ccq;
extern "C" void plan(int kind, int fp4, int row_major, int scaled, int tokens, int n_out, int K, int n_segments, const int* segments, int scratch, int cus, int* out)
{
    LinearArgs a{};
    a.tokens = tokens;
    a.n_out = n_out;
    a.K = K;
    a.n_segments = n_segments;
    for (int s = 0; s < n_segments; s++) { a.seg_n_out[s] = segments[s]; }
    const GemmPlan p = plan_gemm(a, (GemmKind)kind, GemmWeights{ fp4 != 0, row_major != 0, scaled != 0 }, cus, scratch != 0);
    out[0] = p.mb;
    out[1] = p.nb;
    out[2] = p.splits;
    out[3] = p.small;
    out[4] = p.ranges;
}
"""

_lib = None


def plan(kind, tokens, n_out, K, fp4=False, row_major=False, scaled=False, scratch=True, cus=256):
    """(tokens / 16, features / 64, k ranges, small tile?, k ranges of the scratch held); n_out: a list for segments."""
    global _lib
    if _lib is None:
        csrc = Path(__file__).resolve().parent.parent / "cccc-lite_amd" / "csrc"
        with tempfile.TemporaryDirectory() as d:
            (Path(d) / "plan.cpp").write_text(SOURCE)
            subprocess.run(["g++", "-O1", "-std=c++17", "-Wall", "-Werror", "-shared", "-fPIC", "-I", str(csrc), "plan.cpp", "-o", "plan.so"], cwd=d, check=True)
            _lib = ctypes.CDLL(str(Path(d) / "plan.so"))
    segments = list(n_out) if kind == SEGMENTS else []
    out = (ctypes.c_int * 5)()
    _lib.plan(kind, fp4, row_major, scaled, tokens, 0 if segments else n_out, K, len(segments), (ctypes.c_int * 3)(*segments), scratch, cus, out)
    return tuple(out)
