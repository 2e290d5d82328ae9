"""Host rules of the GEMM launches and of the prepared operators, compiled with g++
from the library's own headers: nothing here touches a GPU."""
import shutil
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parents[1]
ROCM = Path("/opt/rocm/include")
HEAD = r"""
#include <cstdio>
#include "gemm.h"
#include "ops.h"
using namespace mk;
// device buffers stay empty here
void mk::DevBuf::release() {}
#define CHECK(c) do { if (!(c)) { std::printf("line %d: %s\n", __LINE__, #c); return 1; } } while (0)
int main() {
"""


def run(tmp_path, body):
    """Compile `body`, statements of main, and run it: 0 if its checks hold."""
    gxx = shutil.which("g++")
    if gxx is None or not ROCM.is_dir():
        pytest.skip("needs g++ and the HIP headers")
    src, exe = tmp_path / "h.cpp", tmp_path / "h"
    src.write_text(HEAD + body + "\nreturn 0;\n}\n")
    subprocess.run([gxx, "-O1", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-I", str(ROCM), "-I",
                    str(ROOT / "mpskit.jl_amd" / "csrc"), str(src), "-o", str(exe)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout


def test_a_full_segment_list_refuses_the_next(tmp_path):
    """One product more than a problem holds changes nothing beside the list and marks the problem."""
    run(tmp_path, r"""
    double a, b, y;
    ProbSpec p;
    p.C = &y; p.ldc = 11; p.alpha = 0.5; p.beta = -2.0; p.phys.b = 3;
    for (int s = 0; s < MAX_SEG; ++s) p.add(&a, 1, &b, 1, s + 1);
    CHECK(p.nseg == MAX_SEG && !p.full);
    p.add(&a, 77, &b, 78, 79);
    CHECK(p.full && p.nseg == MAX_SEG);
    CHECK(p.seg[MAX_SEG - 1].K == MAX_SEG && p.seg[MAX_SEG - 1].lda == 1);
    CHECK(p.C == &y && p.ldc == 11 && p.alpha == 0.5 && p.beta == -2.0 && p.phys.b == 3);
    """)


def test_the_channel_form_joins_only_lists_with_room(tmp_path):
    """A d = 2 two-site operator whose blocks are all full has 4 right and 4 left segments per output block."""
    run(tmp_path, r"""
    double g;
    for (int right = 0; right <= 4; ++right)
      for (int left = 0; left <= 4; ++left) {
        Op op;
        op.xrl.L.view('A', &g, 1, 1);
        for (int e = 0; e < 2; ++e)
          for (int b = 0; b < 2; ++b) {
            Op::JProb jp{b, e, {}};
            for (int q = 0; q < right; ++q) jp.seg.push_back({'R', q & 1, q >> 1, q});
            if (b == 1 && e == 1)   // the last block's list is the longest
              for (int q = 0; q < left; ++q) jp.seg.push_back({'L', q & 1, q >> 1, q});
            op.jprobs.push_back(jp);
          }
        CHECK(op.xrl_joins() == (right + left + 1 <= MAX_SEG));
      }
    Op none;
    none.jprobs.push_back({0, 0, {}});
    CHECK(!none.xrl_joins());
    """)
