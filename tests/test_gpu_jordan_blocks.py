"""Jordan operators applied by output block (the D x D blocks that are not zero)
against float64 torch contractions of the same environments and MPO tensors.

Edges: odd and unequal bonds (rows and K runs of the mixed operands end in
padding), sizes below one tile, first and last sites of a chain (one MPO row or
column), chains whose blocks are half empty (Ising), full (XXZ), longer-ranged
(J1-J2, three neighbours, exponential decay), a chain of on-site terms only,
MPO tensors without a zero block (eight products an output block beside the channel
form's), spin 1 for one site, alpha / beta, and batches of uneven bonds.

Tolerances: sums of at most 9 products of length D (of w D the channel form's) and
a short physical sum; 2-norm error, relative to the size of a random sum of the same n = 4 D terms
(the sum of their absolute values over sqrt(n); the result itself may cancel at
the smallest sizes), below 8 sqrt(4 D) u of the accumulation (2^-53, 2^-24)
plus twice the operand rounding (2^-24, 2^-16) in the mixed arithmetics.
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


def bound(prec, D):
    s = 8 * math.sqrt(4 * D)
    return {"fp64": s * 2.0 ** -53, "fp32": s * 2.0 ** -24 + 2.0 ** -23, "bf16x3": s * 2.0 ** -24 + 2.0 ** -14}[prec]


def rnd(mk, shape, seed):
    import torch
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return mk.tensors.randn(shape, g)


def close(a, b, tol, size):
    import torch
    return float(torch.linalg.vector_norm(a - b)) <= tol * size


def onsite(d=2):
    W = np.zeros((2, d, d, 2))
    W[0, :, :, 0] = W[1, :, :, 1] = np.eye(d)
    W[0, :, :, 1] = np.arange(d * d).reshape(d, d) - 1.5
    return W


def spin1():
    """Spin-1 Heisenberg chain with a single-ion term (w = 5, d = 3)."""
    s = 1.0 / math.sqrt(2.0)
    sp = 2 * s * np.array([[0, 1, 0], [0, 0, 1], [0, 0, 0.0]])
    sz = np.diag([1.0, 0.0, -1.0])
    W = np.zeros((5, 3, 3, 5))
    W[0, :, :, 0] = W[4, :, :, 4] = np.eye(3)
    for k, (c, b) in enumerate([(0.5 * sp, sp.T), (0.5 * sp.T, sp), (sz, sz)]):
        W[0, :, :, k + 1], W[k + 1, :, :, 4] = c, b
    W[0, :, :, 4] = 0.3 * sz @ sz
    return W


def chain(mk, name):
    m = mk.models
    return {"tfim": lambda: m.tfim_bulk(0.7), "xxz": lambda: m.xxz_bulk(0.5), "j1j2": lambda: m.j1j2_bulk(),
            "three": lambda: m.heisenberg_range_bulk([1.0, 0.5, 0.3]), "exp": lambda: m.exp_ising_bulk(),
            "onsite": onsite, "spin1": spin1}[name]()


def envs(mk, Dl, wl, Dr, wr):
    """Random levels, and the same with the identities a Jordan operator assumes."""
    import torch
    T = mk.tensors
    GL, GR = rnd(mk, (Dl, wl, Dl), 1), rnd(mk, (Dr, wr, Dr), 2)
    GLi, GRi = GL.clone(), GR.clone()
    GLi[:, 0, :] = torch.eye(Dl, dtype=torch.float64, device="cuda")
    GRi[:, -1, :] = torch.eye(Dr, dtype=torch.float64, device="cuda")
    return T.as_colmajor(GL), T.as_colmajor(GR), GLi, GRi


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


def check(op, x, y0, f, D):
    """f(g): the reference with g applied to every operand."""
    import torch
    ref = f(lambda t: t)
    size = float(torch.linalg.vector_norm(f(torch.abs))) / math.sqrt(4 * D)
    size2 = 0.5 * size + 2.0 * float(torch.linalg.vector_norm(y0))
    for prec in PRECS:
        y = op(x, precision=prec)
        assert close(y, ref, bound(prec, D), size), prec
        y = y0.clone(memory_format=torch.preserve_format)
        op(x, precision=prec, out=y, alpha=-0.5, beta=2.0)
        assert close(y, -0.5 * ref + 2.0 * y0, bound(prec, D), size2), prec


@pytest.mark.parametrize("name", ["tfim", "xxz", "j1j2", "three", "exp", "onsite"])
@pytest.mark.parametrize("Dl,Dr", [(1, 1), (5, 3), (17, 40), (64, 64), (131, 77), (300, 301)])
def test_two_site(mk, name, Dl, Dr):
    T = mk.tensors
    W = chain(mk, name)
    for site, (W1, W2) in {"bulk": (W, W), "first": (W[:1], W), "last": (W, W[..., -1:]), "both": (W[:1], W[..., -1:])}.items():
        GL, GR, GLi, GRi = envs(mk, Dl, W1.shape[0], Dr, W2.shape[3])
        W1d, W2d = T.from_numpy(W1), T.from_numpy(W2)
        x, y0 = rnd(mk, (Dl, 2, Dr, 2), 3), rnd(mk, (Dl, 2, Dr, 2), 4)
        print("blocks", name, Dl, Dr, site, flush=True)
        op = mk.prepare_operator(mk.JordanMPO_AC2_Hamiltonian(GL, W1d, W2d, GR), precisions=PRECS)
        check(op, x, y0, lambda g: ac2(g(GLi), g(W1d), g(W2d), g(GRi), g(x)), max(Dl, Dr))


@pytest.mark.parametrize("name", ["tfim", "xxz", "j1j2", "exp", "onsite", "spin1"])
@pytest.mark.parametrize("Dl,Dr", [(1, 1), (5, 3), (64, 64), (131, 77), (300, 301)])
def test_one_site(mk, name, Dl, Dr):
    T = mk.tensors
    Wb = chain(mk, name)
    d = Wb.shape[1]
    for site, W in {"bulk": Wb, "first": Wb[:1], "last": Wb[..., -1:], "only": Wb[:1, :, :, -1:]}.items():
        GL, GR, GLi, GRi = envs(mk, Dl, W.shape[0], Dr, W.shape[3])
        Wd = T.from_numpy(W)
        x, y0 = rnd(mk, (Dl, d, Dr), 3), rnd(mk, (Dl, d, Dr), 4)
        print("blocks", name, Dl, Dr, site, flush=True)
        op = mk.prepare_operator(mk.JordanMPO_AC_Hamiltonian(GL, Wd, GR), precisions=PRECS)
        check(op, x, y0, lambda g: ac(g(GLi), g(Wd), g(GRi), g(x)), max(Dl, Dr))


def dense(w, d=2):
    """A Jordan tensor with every block of A, B, C and D full."""
    W = np.random.default_rng(w).standard_normal((w, d, d, w))
    W[1:, :, :, 0] = W[-1, :, :, :] = 0.0
    W[0, :, :, 0] = W[-1, :, :, -1] = np.eye(d)
    return W


@pytest.mark.parametrize("w", [3, 5])
@pytest.mark.parametrize("Dl,Dr", [(33, 20), (120, 131), (200, 215), (301, 264)])
def test_full_blocks(mk, w, Dl, Dr):
    """Below and past the sizes where the channel form takes over; the allocation-free apply too."""
    import torch
    from mpskit_amd._lib import PREC_NAMES, check as ok, load
    T = mk.tensors
    Wb = dense(w)
    sites = {"bulk": (Wb, Wb), "first": (Wb[:1], Wb), "last": (Wb, Wb[..., -1:])}
    for site, (W1, W2) in sites.items():
        GL, GR, GLi, GRi = envs(mk, Dl, W1.shape[0], Dr, W2.shape[3])
        W1d, W2d = T.from_numpy(W1), T.from_numpy(W2)
        x, y0 = rnd(mk, (Dl, 2, Dr, 2), 3), rnd(mk, (Dl, 2, Dr, 2), 4)
        print("full blocks", w, Dl, Dr, site, flush=True)
        op = mk.prepare_operator(mk.JordanMPO_AC2_Hamiltonian(GL, W1d, W2d, GR), precisions=PRECS)
        f = lambda g: ac2(g(GLi), g(W1d), g(W2d), g(GRi), g(x))   # noqa: E731
        check(op, x, y0, f, max(Dl, Dr))
        ref, size = f(lambda t: t), float(torch.linalg.vector_norm(f(torch.abs))) / math.sqrt(4 * max(Dl, Dr))
        for prec in PRECS:
            y = y0.clone(memory_format=torch.preserve_format)
            ok(load().mk_apply_noalloc(op.handle, T.ptr(x), T.ptr(y), 1.0, 0.0, PREC_NAMES[prec]))
            torch.cuda.synchronize()
            assert close(y, ref, bound(prec, max(Dl, Dr)), size), prec
    GL, GR, GLi, GRi = envs(mk, Dl, w, Dr, w)
    Wd, x, y0 = T.from_numpy(Wb), rnd(mk, (Dl, 2, Dr), 3), rnd(mk, (Dl, 2, Dr), 4)
    op = mk.prepare_operator(mk.JordanMPO_AC_Hamiltonian(GL, Wd, GR), precisions=PRECS)
    check(op, x, y0, lambda g: ac(g(GLi), g(Wd), g(GRi), g(x)), max(Dl, Dr))


@pytest.mark.parametrize("name", ["tfim", "xxz", "j1j2", "exp", "onsite"])
@pytest.mark.parametrize("Dl,Dr", [(210, 203), (193, 260)])
def test_mixed_arithmetic_is_used(mk, name, Dl, Dr):
    """The smallest applies run in FP64 whatever is asked for (64 x 64 is one); past that line each arithmetic is
    its own, on runs of K with every kind of padding."""
    import torch
    T = mk.tensors
    W = T.from_numpy(chain(mk, name))
    for D1, D2, small in ((Dl, Dr, False), (64, 64, True)):
        GL, GR, GLi, GRi = envs(mk, D1, W.shape[0], D2, W.shape[3])
        x2, x1 = rnd(mk, (D1, 2, D2, 2), 3), rnd(mk, (D1, 2, D2), 3)
        for H, x, f in ((mk.JordanMPO_AC2_Hamiltonian(GL, W, W, GR), x2, lambda g: ac2(g(GLi), g(W), g(W), g(GRi), g(x2))),
                        (mk.JordanMPO_AC_Hamiltonian(GL, W, GR), x1, lambda g: ac(g(GLi), g(W), g(GRi), g(x1)))):
            op = mk.prepare_operator(H, precisions=PRECS)
            print("mixed", name, D1, D2, x.dim(), flush=True)
            check(op, x, torch.zeros_like(x), f, max(D1, D2))
            y = {p: op(x, precision=p) for p in PRECS}
            if small and name in ("tfim", "onsite"):
                assert torch.equal(y["bf16x3"], y["fp64"]) and torch.equal(y["fp32"], y["fp64"])
            if not small:
                n64 = float(torch.linalg.vector_norm(y["fp64"]))
                for p in ("fp32", "bf16x3"):   # off by a few roundings of the operands, not by those of FP64
                    assert 1e-9 < float(torch.linalg.vector_norm(y[p] - y["fp64"])) / n64 < 1e-4, p
                assert not torch.equal(y["fp32"], y["bf16x3"])


@pytest.mark.parametrize("name", ["tfim", "xxz", "onsite"])
def test_batch_of_uneven_bonds(mk, name):
    import torch
    T = mk.tensors
    W = T.from_numpy(chain(mk, name))
    ops, xs, refs = [], [], []
    for i, (Dl, Dr) in enumerate([(33, 47), (96, 96), (130, 129), (8, 200)]):
        GL, GR, GLi, GRi = envs(mk, Dl, W.shape[0], Dr, W.shape[3])
        ops.append(mk.prepare_operator(mk.JordanMPO_AC2_Hamiltonian(GL, W, W, GR), precisions=PRECS))
        xs.append(rnd(mk, (Dl, 2, Dr, 2), 10 + i))
        refs.append(ac2(GLi, W, W, GRi, xs[-1]))
    b = mk.BatchedDerivative(ops)
    assert b.grouped
    for prec in PRECS:
        for y, ref in zip(b.unpack(b.apply(b.pack(xs), precision=prec)), refs):
            assert close(y, ref, bound(prec, 200), float(torch.linalg.vector_norm(ref))), prec
