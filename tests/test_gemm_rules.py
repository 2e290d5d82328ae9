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
#include "gemm_plan.h"
#include "ops.h"
#include "ws_table.h"
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


def test_f64_offsets_of_the_last_k_step_stay_below_2_gib(tmp_path):
    """gemm_f64_dma_kernel adds an unmasked scalar offset to every load, the rows past K of the last
    step among them: none of a problem that f64_fit takes reaches 2^31 - 1 (num_records)."""
    run(tmp_path, r"""
    // largest scalar offset of an operand with R rows (or columns) a tile, as the kernel forms them
    auto largest = [](bool along_k, int64_t R, int64_t ld, int64_t K) {
      int64_t m = 0;
      const int64_t k0 = (K - 1) / 16 * 16;
      for (int64_t wave = 0; wave < 4; ++wave)
        for (int64_t c = 0; c < R * 16 * 8 / 1024 / 4; ++c)
          m = std::max(m, along_k ? 8 * wave * ld * 8 + c * 32 * ld * 8 + k0 * 8
                                  : 128 / R * wave * ld * 8 + c * 4 * (128 / R) * ld * 8 + k0 * ld * 8);
      return m;
    };
    int taken = 0, left = 0;
    for (int64_t ld : {64ll, 4097ll, 1ll << 17, 1000003ll, 2000000ll, 8000000ll, 9000000ll, 16000000ll, 16700000ll, 100000000ll})
      for (int64_t K : {1, 2, 3, 8, 15, 16, 17, 18, 19, 29, 31, 32, 33, 100, 1031})
        for (int bits = 0; bits < 4; ++bits)
          for (int t : {64, 128}) {
            const GemmShape sh{(bits & 1) != 0, (bits & 2) != 0};
            ProbSpec p;
            p.M = p.N = 4096;
            p.add(reinterpret_cast<const void*>(1 << 20), ld, reinterpret_cast<const void*>(1 << 20), ld, K);
            const bool fits = f64_fit(p, sh, t, t) != BUF_NO;
            if (fits) CHECK(largest(sh.ta, t, ld, K) + 16 < (1ll << 31) && largest(!sh.tb, t, ld, K) + 16 < (1ll << 31));
            (fits ? taken : left) += 1;
          }
    CHECK(taken > 200 && left > 200);
    // the product of a Krylov basis with the coefficients of its Ritz vectors, at D = 1500 and 2048
    auto ritz = [](int64_t n, int64_t K) {
      ProbSpec p;
      p.M = n; p.N = 5;
      p.add(reinterpret_cast<const void*>(1 << 20), n, reinterpret_cast<const void*>(1 << 20), K, K);
      return f64_fit(p, GemmShape{}, 64, 64);
    };
    CHECK(ritz(4 * 1500 * 1500, 16) == BUF_EVEN && ritz(4 * 1500 * 1500, 17) == BUF_NO);
    CHECK(ritz(16000000, 17) == BUF_NO && ritz(4 * 2048 * 2048, 16) == BUF_EVEN);
    CHECK(ritz(4 * 1024 * 1024, 30) == BUF_EVEN && ritz(4 * 1024 * 1024, 29) == BUF_ODD);
    CHECK(ritz(20000000, 8) == BUF_NO);
    """)


def test_workspace_table_hands_idle_slots_on(tmp_path):
    """Streams past the slots get a workspace once one of the others has been idle, after a wait for the
    device; a rotation over too many streams swaps none; a refused allocation is tried again later."""
    run(tmp_path, r"""
    static char mem[64];
    static int allocs = 0, waits = 0;
    static bool refuse = false;
    auto alloc = [] { return refuse ? (void*)nullptr : (void*)&mem[allocs++]; };
    auto wait = [] { ++waits; return true; };
    auto st = [](int i) { return reinterpret_cast<const void*>((uintptr_t)(1000 + i)); };
    WsTable t;
    void* own[WsTable::SLOTS];
    for (int i = 0; i < WsTable::SLOTS; ++i) own[i] = t.get(st(i), alloc, wait);
    for (int i = 0; i < WsTable::SLOTS; ++i) {
      CHECK(own[i] && t.get(st(i), alloc, wait) == own[i]);
      for (int j = 0; j < i; ++j) CHECK(own[i] != own[j]);
    }
    CHECK(allocs == WsTable::SLOTS);
    // all in use: the streams past the slots go without, in any number of rounds
    for (int r = 0; r < 1000; ++r)
      for (int i = 0; i < WsTable::SLOTS + 2; ++i)
        CHECK(t.get(st(i), alloc, wait) == (i < WsTable::SLOTS ? own[i] : nullptr));
    CHECK(waits == 0);
    // stream 3 is heard of no more: its slot goes to the next one past them, once
    int got = -1;
    for (uint64_t r = 0; r < 2 * WsTable::IDLE && got < 0; ++r)
      for (int i = 0; i < WsTable::SLOTS + 1; ++i) {
        if (i == 3) continue;
        void* p = t.get(st(i), alloc, wait);
        if (i == WsTable::SLOTS && p) { CHECK(p == own[3]); got = (int)r; }
      }
    CHECK(got > 0 && waits == 1 && allocs == WsTable::SLOTS);
    CHECK(t.get(st(3), alloc, wait) == nullptr);
    // a wait that fails hands nothing on
    WsTable u;
    for (int i = 0; i < WsTable::SLOTS; ++i) u.get(st(i), alloc, wait);
    for (uint64_t r = 0; r < 3 * WsTable::IDLE; ++r) u.get(st(0), alloc, wait);
    CHECK(u.get(st(99), alloc, [] { return false; }) == nullptr && u.slot[1].stream == st(1));
    // refused allocations
    WsTable v;
    refuse = true;
    for (uint64_t r = 0; r + 1 < WsTable::IDLE; ++r) CHECK(v.get(st(0), alloc, wait) == nullptr);
    refuse = false;
    CHECK(v.get(st(0), alloc, wait) == nullptr);
    for (uint64_t r = 0; r < 3; ++r) v.get(st(0), alloc, wait);
    CHECK(v.get(st(0), alloc, wait) != nullptr);
    int freed = 0;
    t.clear([&](void*) { ++freed; });
    CHECK(freed == WsTable::SLOTS && t.n == 0);
    """)
