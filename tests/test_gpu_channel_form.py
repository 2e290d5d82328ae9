"""Generic derivative operators applied as x GR, MPO step, GL (the channel form),
at sizes past the line where the operator switches to it, against float64 torch.

Edges: unequal bonds on all four environment legs, odd sizes (rows of the mixed
operands end in padding), MPO bonds that differ left, middle and right, d1 !=
d2, input counts at and between the register sizes of the MPO step (8, 16, 20,
32), alpha / beta, the allocation-free apply whose intermediates need chunks,
and the A / AA parts of Jordan operators.

Tolerances: two products and a short sum; relative 2-norm error below
4 sqrt(K) u of the accumulation (2^-53, 2^-24) plus twice the operand rounding
(2^-24, 2^-16) in the mixed arithmetics.
"""
import math

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

PRECS = ("fp64", "fp32", "bf16x3")


@pytest.fixture(scope="module")
def mk():
    import torch
    assert torch.cuda.is_available(), "GPU tests need a ROCm device"
    import mpskit_amd
    mpskit_amd.load()
    return mpskit_amd


def bound(prec, K):
    return {"fp64": 4 * math.sqrt(K) * 2.0 ** -53, "fp32": 8 * (math.sqrt(K) * 2.0 ** -24 + 2.0 ** -24),
            "bf16x3": 8 * (math.sqrt(K) * 2.0 ** -24 + 2.0 ** -16)}[prec]


def rnd(mk, shape, seed):
    import torch
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return mk.tensors.randn(shape, g)


def ac2(GL, W1, W2, GR, x):
    import torch
    z = torch.tensordot(GL, x, ([2], [0]))
    z = torch.tensordot(z, W1, ([1, 2], [0, 2]))
    z = torch.tensordot(z, W2, ([4, 2], [0, 2]))
    return torch.tensordot(z, GR, ([1, 4], [0, 1])).permute(0, 1, 3, 2)


def ac(GL, W, GR, x):
    import torch
    z = torch.tensordot(GL, x, ([2], [0]))
    z = torch.tensordot(z, W, ([1, 2], [0, 2]))
    return torch.tensordot(z, GR, ([1, 3], [0, 1]))


def rel(a, b):
    import torch
    return float(torch.linalg.vector_norm(a - b) / torch.linalg.vector_norm(b))


@pytest.mark.parametrize("dims", [(200, 215, 3, 2, 4, 2, 5, 231, 205), (301, 301, 5, 2, 5, 2, 5, 301, 301),
                                  (333, 280, 2, 3, 3, 2, 2, 300, 260), (400, 400, 8, 2, 8, 2, 8, 390, 390),
                                  (260, 260, 4, 2, 4, 2, 4, 264, 264), (350, 350, 2, 2, 2, 2, 2, 350, 350)])
def test_two_site(mk, dims):
    Da, Df, wl, d1, wm, d2, wr, Di, Dc = dims
    GL, GR = rnd(mk, (Da, wl, Df), 1), rnd(mk, (Di, wr, Dc), 2)
    W1, W2 = rnd(mk, (wl, d1, d1, wm), 3), rnd(mk, (wm, d2, d2, wr), 4)
    x, y0 = rnd(mk, (Df, d1, Di, d2), 5), rnd(mk, (Da, d1, Dc, d2), 6)
    op = mk.prepare_operator(mk.MPO_AC2_Hamiltonian(GL, W1, W2, GR), precisions=PRECS)
    ref = ac2(GL, W1, W2, GR, x)
    for prec in PRECS:
        print("channel form", dims, prec, flush=True)
        assert rel(op(x, precision=prec), ref) < bound(prec, max(wl * Df, Di))
        y = y0.clone(memory_format=__import__("torch").preserve_format)
        op(x, precision=prec, out=y, alpha=-0.5, beta=2.0)
        assert rel(y, -0.5 * ref + 2.0 * y0) < bound(prec, max(wl * Df, Di))


@pytest.mark.parametrize("dims", [(520, 500, 5, 2, 5, 515, 505), (701, 701, 3, 2, 4, 640, 690), (450, 450, 8, 3, 8, 450, 450)])
def test_one_site(mk, dims):
    Da, Df, wl, d, wr, Di, Dc = dims
    GL, GR, W = rnd(mk, (Da, wl, Df), 1), rnd(mk, (Di, wr, Dc), 2), rnd(mk, (wl, d, d, wr), 3)
    x = rnd(mk, (Df, d, Di), 5)
    op = mk.prepare_operator(mk.MPO_AC_Hamiltonian(GL, W, GR), precisions=PRECS)
    ref = ac(GL, W, GR, x)
    for prec in PRECS:
        print("channel form", dims, prec, flush=True)
        assert rel(op(x, precision=prec), ref) < bound(prec, max(wl * Df, Di))


@pytest.mark.parametrize("js", [[1.0, 0.24], [1.0, 0.5, 0.3]])
def test_jordan_parts(mk, js):
    """J1-J2 (A part of the one-site operator) and a three-neighbour chain (AA part of the two-site one)."""
    import torch
    T = mk.tensors
    W = T.from_numpy(mk.models.heisenberg_range_bulk(js))
    w, Dl, Dr = W.shape[0], 333, 350
    GL, GR = rnd(mk, (Dl, w, Dl), 1) / 18.0, rnd(mk, (Dr, w, Dr), 2) / 18.0
    GL, GR = T.as_colmajor(GL), T.as_colmajor(GR)
    GLi, GRi = GL.clone(), GR.clone()
    GLi[:, 0, :] = torch.eye(Dl, dtype=torch.float64, device="cuda")
    GRi[:, -1, :] = torch.eye(Dr, dtype=torch.float64, device="cuda")
    x2, x1 = rnd(mk, (Dl, 2, Dr, 2), 3), rnd(mk, (Dl, 2, Dr), 4)
    for op, x, ref in ((mk.JordanMPO_AC2_Hamiltonian(GL, W, W, GR), x2, ac2(GLi, W, W, GRi, x2)),
                       (mk.JordanMPO_AC_Hamiltonian(GL, W, GR), x1, ac(GLi, W, GRi, x1))):
        p = mk.prepare_operator(op, precisions=PRECS)
        for prec in PRECS:
            assert rel(p(x, precision=prec), ref) < bound(prec, 4 * w * Dl), (js, prec)


def test_noalloc_chunks(mk):
    """wl = wr = 5 around wm = 3: the fused form's scratch fits the fixed array, the channel form's does not."""
    import torch
    from mpskit_amd._lib import FP64, check, load
    D = 1100
    GL, GR = rnd(mk, (D, 5, D), 1), rnd(mk, (D, 5, D), 2)
    W1, W2 = rnd(mk, (5, 2, 2, 3), 3), rnd(mk, (3, 2, 2, 5), 4)
    x = rnd(mk, (D, 2, D, 2), 5)
    op = mk.prepare_operator(mk.MPO_AC2_Hamiltonian(GL, W1, W2, GR))
    y = mk.tensors.empty(op.y_shape)
    ref = op(x)
    check(load().mk_apply_noalloc(op.handle, mk.tensors.ptr(x), mk.tensors.ptr(y), 1.0, 0.0, FP64))
    torch.cuda.synchronize()
    assert rel(y, ref) < bound("fp64", 5 * D)
    assert np.isfinite(float(torch.sum(y)))
