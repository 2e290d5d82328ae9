"""GEMM launches whose tiles are cut along K (mk_gemm, all three arithmetics).

Sizes whose tiles do not fill the GPU are split: all of them, or those of the
last round.  Operands too large for 32-bit offsets within a tile take the kernels
that the usual ones fall back to.  Edges: one tile with a long K, K that is not a multiple of a step
or of the slices, odd sizes and leading dimensions, a last round of few tiles,
beta != 0 (C is read by the reduction only).  Against float64 torch.

Tolerances: the partial sums of a slice and their sum have the same bound as
one long sum, K u |A||B|; on Gaussian operands the relative 2-norm error stays
below sqrt(K) u for u the unit roundoff of the accumulation (2^-53, 2^-24),
plus for the mixed arithmetics the rounding of the operands (2^-24; 2^-16 for
hi + lo bf16, whose lo * lo product is dropped).
"""
import math

import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def mk():
    import torch
    assert torch.cuda.is_available(), "GPU tests need a ROCm device"
    import mpskit_amd
    mpskit_amd.load()
    return mpskit_amd


def bound(prec, K):
    return {"fp64": 4 * math.sqrt(K) * 2.0 ** -53, "fp32": 4 * (math.sqrt(K) * 2.0 ** -24 + 2.0 ** -24),
            "bf16x3": 4 * (math.sqrt(K) * 2.0 ** -24 + 2.0 ** -16)}[prec]


@pytest.mark.parametrize("M,N,K", [(64, 64, 4096), (1, 1, 5000), (130, 70, 4100), (129, 1, 1031), (777, 1001, 3001),
                                   (1024, 1024, 2048), (640, 512, 8190), (2176, 2048, 1026), (5120, 2048, 520),
                                   # odd row counts and K: pairs that straddle the end of a tile, a tile of one row
                                   (2, 3, 5), (65, 63, 3), (1, 1, 1), (127, 129, 17), (129, 65, 1025),
                                   # K split over the waves of a workgroup, and just past its line
                                   (31, 33, 253), (31, 33, 257), (98, 162, 128), (130, 70, 130), (129, 257, 33), (193, 129, 129), (1153, 1025, 257)])
@pytest.mark.parametrize("prec", ["fp64", "fp32", "bf16x3"])
def test_split_gemm_matches_torch(mk, M, N, K, prec):
    import torch
    T = mk.tensors
    g = torch.Generator(device="cuda")
    g.manual_seed(M + 3 * N + 7 * K)
    for ta, tb, alpha, beta in ((False, False, 1.0, 0.0), (True, False, -0.5, 2.0), (False, True, 2.0, -1.0),
                                (True, True, 1.0, 1.0)):
        A = T.randn((K, M) if ta else (M, K), g)
        B = T.randn((N, K) if tb else (K, N), g)
        C = T.randn((M, N), g)
        ref = alpha * ((A.t() if ta else A) @ (B.t() if tb else B)) + beta * C
        scale = float(torch.linalg.vector_norm(ref))
        print("split gemm", M, N, K, prec, ta, tb, flush=True)
        out = mk.gemm(A, B, C, alpha=alpha, beta=beta, transa=ta, transb=tb, precision=prec)
        assert float(torch.linalg.vector_norm(out - ref)) <= bound(prec, K) * scale


@pytest.mark.parametrize("M,K", [(9_000_001, 17), (9_000_000, 18), (8_000_000, 19), (16_000_000, 16)])
def test_tall_operand(mk, M, K):
    """A Krylov basis times the coefficients of its Ritz vectors: columns so long that the K step past the
    last one would end beyond 2 GiB from the tile's first row (K = 16 has none)."""
    import torch
    T = mk.tensors
    g = torch.Generator(device="cuda")
    g.manual_seed(K)
    A, B = T.randn((M, K), g), T.randn((K, 5), g)
    print("tall gemm", M, K, flush=True)
    out, ref = mk.gemm(A, B), A @ B
    assert float(torch.linalg.vector_norm(out - ref)) <= bound("fp64", K) * float(torch.linalg.vector_norm(ref))


def mk_gemm(mk, A, lda, B, ldb, C, M, N, K, ta, tb, prec):
    """C = -0.5 op(A) op(B) + 2 C through the C ABI, with leading dimensions of any length."""
    import ctypes
    from mpskit_amd._lib import PREC_NAMES, check, load
    pa, pb, pc = (ctypes.c_void_p(t.data_ptr()) for t in (A, B, C))
    check(load().mk_gemm(mk.derivatives.default_context().handle, int(ta), int(tb), M, N, K, -0.5, pa, lda, pb, ldb, 2.0,
                         pc, M, PREC_NAMES[prec]))


@pytest.mark.parametrize("ta,tb,K,lda,ldb", [(False, False, 1031, 1 << 18, 1031), (True, False, 1031, 2_200_000, 1040),
                                             (False, True, 520, 131, 1 << 19), (True, True, 514, 520, 530_001)])
def test_fp64_past_the_32_bit_offsets(mk, ta, tb, K, lda, ldb):
    """Operands whose tiles span 2 GiB and more run on the branching kernel, whole and cut along K."""
    import torch
    M, N = 130, 70
    g = torch.Generator(device="cuda")
    g.manual_seed(K)
    # column-major with leading dimensions lda, ldb: the columns are rows of the torch tensors
    A = torch.full((M if ta else K, lda), float("nan"), dtype=torch.float64, device="cuda")
    B = torch.full((K if tb else N, ldb), float("nan"), dtype=torch.float64, device="cuda")
    a, b = A[:, :K if ta else M], B[:, :N if tb else K]
    a.normal_(generator=g)
    b.normal_(generator=g)
    C = mk.tensors.randn((M, N), g)
    ref = -0.5 * ((a if ta else a.t()) @ (b if tb else b.t())) + 2.0 * C
    print("branching fp64 gemm", ta, tb, K, lda, ldb, flush=True)
    mk_gemm(mk, A, lda, B, ldb, C, M, N, K, ta, tb, "fp64")
    assert float(torch.linalg.vector_norm(C - ref)) <= bound("fp64", K) * float(torch.linalg.vector_norm(ref))


@pytest.mark.parametrize("prec,K", [("bf16x3", 4_200_003), ("fp32", 2_100_005)])
@pytest.mark.parametrize("M,N", [(70, 9), (129, 40)])
def test_mixed_past_the_32_bit_offsets(mk, prec, K, M, N):
    """Operands of which 256 rows span 2 GiB and more run on the register-staged kernel, cut along K."""
    import torch
    g = torch.Generator(device="cuda")
    g.manual_seed(K)
    # rows of K entries on both sides (transposed storage of A)
    A, B = (torch.randn((n, K), dtype=torch.float64, device="cuda", generator=g) for n in (M, N))
    C = mk.tensors.randn((M, N), g)
    ref = -0.5 * (A @ B.t()) + 2.0 * C
    print("register-staged mixed gemm", prec, M, N, K, flush=True)
    mk_gemm(mk, A, K, B, K, C, M, N, K, True, False, prec)
    assert float(torch.linalg.vector_norm(C - ref)) <= bound(prec, K) * float(torch.linalg.vector_norm(ref))


def test_split_gemm_repeats_bitwise(mk):
    """The slices are added in a fixed order, and an unordered second stream has a workspace of its own."""
    import torch
    T = mk.tensors
    A, B = T.randn((1000, 3000)), T.randn((3000, 500))
    first = mk.gemm(A, B).clone()
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    outs = []
    for _ in range(3):
        outs.append(mk.gemm(A, B))
        with torch.cuda.stream(s):
            outs.append(mk.gemm(A, B))
    torch.cuda.synchronize()
    for o in outs:
        assert torch.equal(o, first)


def test_split_gemm_on_many_streams(mk):
    """A long-lived context splits on each of many streams, and for new ones once older ones are idle: the
    result is that of the split launch, bit for bit."""
    import torch
    T = mk.tensors
    A, B = T.randn((500, 3000)), T.randn((3000, 400))
    first = mk.gemm(A, B).clone()
    torch.cuda.synchronize()
    streams = [torch.cuda.Stream() for _ in range(24)]
    for s in streams[:12]:
        with torch.cuda.stream(s):
            out = mk.gemm(A, B)
        s.synchronize()
        assert torch.equal(out, first)
    for s in streams[12:]:
        with torch.cuda.stream(s):
            for _ in range(1100):
                out = mk.gemm(A, B, out)
        s.synchronize()
        assert torch.equal(out, first)


def test_workspaces_are_given_back(mk):
    """The streams' workspaces and the Krylov workspace (26 columns of 2^20 doubles and more at D = 512)."""
    import torch
    T = mk.tensors
    W, D = T.from_numpy(mk.models.tfim_bulk(1.0)), 512
    GL, GR = T.randn((D, 3, D)) / D, T.randn((D, 3, D)) / D
    GL, GR = (T.as_colmajor(0.5 * (E + E.permute(2, 1, 0))) for E in (GL, GR))
    op = mk.prepare_operator(mk.JordanMPO_AC2_Hamiltonian(GL, W, W, GR))
    A, B, x = T.randn((500, 3000)), T.randn((3000, 400)), T.randn((D, 2, D, 2))
    first, e = mk.gemm(A, B).clone(), op.eigsolve(x, krylovdim=20, maxiter=1, tol=1e-3)[0]
    torch.cuda.synchronize()
    before = torch.cuda.mem_get_info()[0]
    op.ctx.release_workspaces()
    after = torch.cuda.mem_get_info()[0]
    print("given back", (after - before) >> 20, "MiB", flush=True)
    assert after - before >= (64 << 20) + 20 * 8 * 4 * D * D
    op.ctx.release_workspaces()
    assert torch.equal(mk.gemm(A, B), first)
    assert op.eigsolve(x, krylovdim=20, maxiter=1, tol=1e-3)[0] == e


def test_split_gemm_not_split_under_capture(mk):
    """A captured call takes no shared workspace; replays agree with the eager result."""
    import torch
    T = mk.tensors
    A, B, C = T.randn((500, 3000)), T.randn((3000, 400)), T.empty((500, 400))
    ref = mk.gemm(A, B).clone()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        mk.gemm(A, B, C)
    for _ in range(3):
        C.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert float(torch.linalg.vector_norm(C - ref)) <= bound("fp64", 3000) * float(torch.linalg.vector_norm(ref))
        mk.gemm(A, B)
