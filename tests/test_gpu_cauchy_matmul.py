"""Cauchy-product matmul kernel vs the CPU oracle (GPU).

``a @ b`` on PolyTensors inside plain_range() runs C_k = sum_{i+j=k} A_i B_j in
one MFMA launch; the oracle forms the reference's (K+1)(K+2)/2 matmuls
(/root/reference/src/polytensors/_plain.py:118-128) in float64. Per-order
tolerance max|got - want| / max|want|: 1e-10 float64, 1e-4 float32 (fp32 MFMA,
no TF32 anywhere).
"""

import pytest
import torch
import torch.nn.functional as F

import oracle
from polytensors_amd import PolyTensor, _ops
from tests.jets import rel_err

pytestmark = pytest.mark.gpu

TOL = {torch.float64: 1e-10, torch.float32: 1e-4}


def _series(shape, degree, seed, dtype):
    g = torch.Generator().manual_seed(seed)
    return [(torch.randn(shape, generator=g, dtype=torch.float64) * 0.5 ** k).to(dtype) for k in range(degree + 1)]


def _poly(cs):
    return PolyTensor(tuple(c.cuda() for c in cs))


def _check(got, want, dtype):
    assert len(got) == len(want)
    for k, (a, b) in enumerate(zip(got, want)):
        err = rel_err(a.cpu(), b)
        assert err <= TOL[dtype], f"order {k}: {err:.3e}"


@pytest.mark.parametrize("m,kd,n", [(64, 64, 64), (128, 256, 192), (100, 70, 90), (1, 33, 5), (257, 129, 65),
                                    (31, 3, 200), (64, 1, 64)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("degree", [1, 4])
def test_matches_oracle(monkeypatch, m, kd, n, dtype, degree):
    calls = []
    original = _ops.cauchy_matmul
    monkeypatch.setattr(_ops, "cauchy_matmul", lambda *a, **k: calls.append(1) or original(*a, **k))
    A, B = _series((m, kd), degree, 1, dtype), _series((kd, n), degree, 2, dtype)
    with torch.no_grad(), PolyTensor.plain_range():
        c = _poly(A) @ _poly(B)
    assert calls == [1] and c.shape == (m, n) and c.degree == degree
    _check(c.coeffs, oracle.matmul([a.double() for a in A], [b.double() for b in B]), dtype)


@pytest.mark.parametrize("degree", [0, 2, 3, 5, 6, 7, 8])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
def test_every_degree(degree, dtype):
    A, B = _series((96, 80), degree, 3, dtype), _series((80, 112), degree, 4, dtype)
    with torch.no_grad(), PolyTensor.plain_range():
        c = torch.matmul(_poly(A), _poly(B))
    _check(c.coeffs, oracle.matmul([a.double() for a in A], [b.double() for b in B]), dtype)


@pytest.mark.parametrize("side", ["left", "right"])
def test_plain_operand_uses_one_order(side):
    degree, dtype = 4, torch.float32
    A, B = _series((70, 48), degree, 5, dtype), _series((48, 66), degree, 6, dtype)
    with torch.no_grad(), PolyTensor.plain_range():
        if side == "left":
            c = A[0].cuda() @ _poly(B)
            want = oracle.matmul([A[0].double()], [b.double() for b in B])
        else:
            c = _poly(A) @ B[0].cuda()
            want = oracle.matmul([a.double() for a in A], [B[0].double()])
    _check(c.coeffs, want, dtype)


def test_batched_and_broadcast():
    degree, dtype = 3, torch.float32
    A = _series((2, 3, 40, 24), degree, 7, dtype)
    B = _series((24, 56), degree, 8, dtype)
    Bb = _series((2, 3, 24, 56), degree, 9, dtype)
    with torch.no_grad(), PolyTensor.plain_range():
        c1 = _poly(A) @ _poly(B)
        c2 = _poly(A) @ _poly(Bb)
        c3 = torch.bmm(_poly([a.reshape(6, 40, 24) for a in A]), _poly([b.reshape(6, 24, 56) for b in Bb]))
    _check(c1.coeffs, oracle.matmul([a.double() for a in A], [b.double() for b in B]), dtype)
    _check(c2.coeffs, oracle.matmul([a.double() for a in A], [b.double() for b in Bb]), dtype)
    _check([c.reshape(2, 3, 40, 56) for c in c3.coeffs], oracle.matmul([a.double() for a in A], [b.double() for b in Bb]),
           dtype)


@pytest.mark.parametrize("bias", [False, True])
def test_linear_uses_transposed_weight(bias):
    degree, dtype = 3, torch.float32
    X = _series((5, 7, 48), degree, 10, dtype)
    W = _series((40, 48), degree, 11, dtype)
    b = torch.randn(40, generator=torch.Generator().manual_seed(12)).to(dtype)
    with torch.no_grad(), PolyTensor.plain_range():
        y = F.linear(_poly(X), _poly(W), b.cuda() if bias else None)
    want = oracle.matmul([x.double() for x in X], [w.double().t() for w in W])
    if bias:
        want = [want[0] + b.double()] + want[1:]
    _check(y.coeffs, want, dtype)


@pytest.mark.parametrize("plain_b", [False, True])
def test_matmul_by_transposed_view(plain_b):
    # x @ W.t() with W contiguous [n, k]: the kernel reads W in place (its transposed-B mode)
    degree, dtype = 2, torch.float32
    X = _series((3, 33, 48), degree, 15, dtype)
    W = _series((40, 48), 0 if plain_b else degree, 16, dtype)
    with torch.no_grad(), PolyTensor.plain_range():
        w = W[0].cuda().t() if plain_b else PolyTensor(tuple(c.cuda().t() for c in W))
        y = _poly(X) @ w
    want = oracle.matmul([x.double() for x in X], [c.double().t() for c in W])
    _check(y.coeffs, want, dtype)


def test_vector_operands():
    degree, dtype = 2, torch.float64
    A, v = _series((30, 20), degree, 13, dtype), _series((20,), degree, 14, dtype)
    with torch.no_grad(), PolyTensor.plain_range():
        c = _poly(A) @ _poly(v)
        d = _poly(v) @ _poly([a.t().contiguous() for a in A])
    _check(c.coeffs, oracle.matmul([a.double() for a in A], [x.double() for x in v]), dtype)
    _check(d.coeffs, oracle.matmul([x.double() for x in v], [a.double().t() for a in A]), dtype)


def test_known_answer_real_analog():
    # /root/reference/tests/test_dispatch.py:63-70 with real directions: a = (I, J), b = (2I, 2J), J = ones(2, 2)
    eye, ones = torch.eye(2, dtype=torch.float64), torch.ones(2, 2, dtype=torch.float64)
    a = PolyTensor((eye.cuda(), ones.cuda()), degree=2)
    b = PolyTensor(((2 * eye).cuda(), (2 * ones).cuda()), degree=2)
    with torch.no_grad(), PolyTensor.plain_range():
        c = a @ b
    assert torch.equal(c.coeffs[0].cpu(), 2 * eye)
    assert torch.equal(c.coeffs[1].cpu(), 4 * ones)
    assert torch.equal(c.coeffs[2].cpu(), 4 * ones)     # J @ 2J = 4J


def test_full_size_config_sampled_rows():
    # benchmark config 2: A, B [5, 4096, 4096] fp32, coefficient k scaled by 0.5^k. Rows of C are checked
    # on a seeded sample; the full product's linearity is checked through C(A + A') = C(A) + C(A').
    degree, n = 4, 4096
    g = torch.Generator(device="cuda").manual_seed(1)
    A = [torch.randn(1, n, n, generator=g, device="cuda") * 0.5 ** k for k in range(degree + 1)]
    B = [torch.randn(1, n, n, generator=g, device="cuda") * 0.5 ** k for k in range(degree + 1)]
    C = _ops.cauchy_matmul(A, B, degree, False)
    rows = torch.randperm(n, generator=torch.Generator().manual_seed(2))[:8]
    want = oracle.matmul([a[0][rows].cpu().double() for a in A], [b[0].cpu().double() for b in B])
    _check([c[0][rows.cuda()] for c in C], want, torch.float32)
    A2 = [a.flip(-1) for a in A]
    lhs = _ops.cauchy_matmul([x + y for x, y in zip(A, A2)], B, degree, False)
    rhs = C + _ops.cauchy_matmul(A2, B, degree, False)
    for k in range(degree + 1):
        assert rel_err(lhs[k].cpu(), rhs[k].cpu()) <= 1e-5


# An ordinary operand on either side: the order-by-order products, at the edges of their tiles (64, 128
# and 256 rows or columns), contractions around its chunks (16 floats, 32 halves) and its four-chunk
# ring, single rows, batches, and row lengths the 16-byte loads do not take.
# Tolerance: each order against float64 of the stored inputs, relative to its largest value: one
# rounding of the result in the storage type, and float32 sums of k terms (below 1e-5 here).
@pytest.mark.parametrize("dtype,tol", [(torch.float32, 1e-5), (torch.bfloat16, 2.0 ** -8), (torch.float16, 2.0 ** -11 + 1e-5)])
@pytest.mark.parametrize("m,k,n,batch,degree", [
    (1, 8, 8, (), 1), (64, 16, 64, (), 2), (65, 72, 136, (), 3), (128, 128, 128, (), 8), (129, 160, 264, (), 2),
    (257, 64, 256, (3,), 1), (255, 1000, 513, (), 2), (40, 15, 33, (2,), 2), (520, 256, 3000, (), 4), (2, 4104, 72, (), 3)])
def test_ordinary_operand_products(dtype, tol, m, k, n, batch, degree):
    g = torch.Generator().manual_seed(m + k + n)
    A = [torch.randn(*batch, m, k, generator=g).to(dtype) for _ in range(degree + 1)]
    W = (torch.randn(n, k, generator=g) / k ** 0.5).to(dtype)
    B = [torch.randn(*batch, k, n, generator=g).to(dtype) for _ in range(degree + 1)]
    L = (torch.randn(m, k, generator=g) / k ** 0.5).to(dtype)
    with torch.no_grad(), PolyTensor.plain_range():
        x, y = (PolyTensor(tuple(c.cuda() for c in s)) for s in (A, B))
        got = {"x @ W^T": x @ W.cuda().t(), "x @ W": x @ W.cuda().t().contiguous(), "L @ y": L.cuda() @ y,
               "linear": torch.nn.functional.linear(x, W.cuda())}
    right, left = W.double().t(), L.double()
    for name, out in got.items():
        for o in range(degree + 1):
            want = left @ B[o].double() if name == "L @ y" else A[o].double() @ right
            err = (out.coeffs[o].cpu().double() - want).abs().max() / want.abs().max()
            assert err <= tol, (name, o, err)


# Series by series with rows that are no whole 16-byte vectors, or that start at any element: operands
# copied with padded rows, outputs written at any element, at the edges of the tiles and with operands
# shared over a batch. Tolerances as above; the sums hold up to (K + 1) k terms.
@pytest.mark.parametrize("dtype,tol", [(torch.float32, 1e-5), (torch.float64, 1e-13), (torch.bfloat16, 2.0 ** -8)])
@pytest.mark.parametrize("m,k,n,batch_a,batch_b,offset", [
    (1, 1, 1, (), (), 0), (64, 31, 65, (), (), 1), (257, 33, 259, (2,), (), 0), (300, 65, 511, (), (3,), 3),
    (65, 128, 64, (), (), 1), (40, 250, 9, (2,), (2,), 0)])
def test_rows_that_no_vector_divides(dtype, tol, m, k, n, batch_a, batch_b, offset):
    g, degree = torch.Generator().manual_seed(m + k + n), 3
    A = [torch.randn(*batch_a, m, k, generator=g, dtype=torch.float64).to(dtype) for _ in range(degree + 1)]
    B = [torch.randn(*batch_b, k, n, generator=g, dtype=torch.float64).to(dtype) for _ in range(degree + 1)]

    def placed(c):   # on the device, `offset` elements past an aligned address
        buffer = torch.zeros(c.numel() + offset, dtype=dtype, device="cuda")
        buffer[offset:] = c.flatten().cuda()
        return buffer[offset:].view(c.shape)

    with torch.no_grad(), PolyTensor.plain_range():
        out = PolyTensor(tuple(placed(c) for c in A)) @ PolyTensor(tuple(placed(c) for c in B))
    want = oracle.matmul([c.double() for c in A], [c.double() for c in B])
    for o in range(degree + 1):
        err = (out.coeffs[o].cpu().double() - want[o]).abs().max() / want[o].abs().max()
        assert err <= tol, (o, err)


# A linear layer's bias added by the kernel (an ordinary vector without a graph) on each kernel: order by
# order, series weights, float64; columns the 16-byte stores do not divide; real and complex directions;
# through addmm under wrapper autograd. A bias the kernel does not take (a series, another dtype) is added after.
@pytest.mark.parametrize("dtype,tol", [(torch.float32, 1e-5), (torch.float64, 1e-13), (torch.bfloat16, 2.0 ** -8)])
@pytest.mark.parametrize("m,k,n", [(1, 8, 3), (130, 72, 65), (64, 40, 264)])
@pytest.mark.parametrize("weight", ["plain", "series", "complex"])
def test_linear_bias(dtype, tol, m, k, n, weight):
    if weight == "complex" and dtype == torch.bfloat16:
        pytest.skip("no complex bfloat16")
    g, degree = torch.Generator().manual_seed(m + n), 3
    draw = lambda *shape: torch.randn(*shape, generator=g, dtype=torch.float64).to(dtype)   # noqa: E731
    X, W = [draw(2, m, k) for _ in range(degree + 1)], [draw(n, k) for _ in range(degree + 1)]
    if weight == "complex":
        X = X[:1] + [torch.complex(c, draw(2, m, k)) for c in X[1:]]
    b = draw(n)
    x = PolyTensor(tuple(c.cuda() for c in X))
    w = PolyTensor(tuple(c.cuda() for c in W)) if weight == "series" else W[0].cuda()
    up = lambda cs: [c.to(torch.complex128 if c.is_complex() else torch.float64) for c in cs]   # noqa: E731
    if weight == "series":
        want = oracle.matmul(up(X), [c.t() for c in up(W)])
    else:
        want = [c @ up(W)[0].t().to(c.dtype) for c in up(X)]
    want[0] = want[0] + b.double()
    with PolyTensor.plain_range():
        with torch.no_grad():
            outs = [F.linear(x, w, b.cuda()), F.linear(x, w, PolyTensor.constant(b.cuda(), degree))]
            if weight != "complex":
                outs.append(F.linear(x, w, b.cuda().double()))   # another dtype: promoted, as torch's add
        xg = PolyTensor(tuple(c.cuda() for c in X), requires_grad=True)
        outs.append(F.linear(xg, w, b.cuda()))
    for out in outs:
        for o in range(degree + 1):
            err = (out.coeffs[o].detach().cpu().to(want[o].dtype) - want[o]).abs().max() / want[o].abs().max()
            assert err <= 2 * tol, (o, err)   # (twice: the separate addition rounds again)


# Rows that whole cache lines would pad past the kernels' 1 GiB a matrix, and whole vectors do not: padded to
# vectors. Products and the gradient of the ordinary operand, on the first and last rows.
@pytest.mark.parametrize("rows,k", [(1_800_000, 257)])
def test_padded_rows_stay_below_the_limit(rows, k):
    n = 8
    g = torch.Generator(device="cuda").manual_seed(0)
    X = [torch.randn(rows, k, generator=g, device="cuda", dtype=torch.bfloat16) for _ in range(2)]
    w = torch.randn(k, n, generator=g, device="cuda", dtype=torch.bfloat16).requires_grad_()
    cot = [torch.randn(rows, n, generator=g, device="cuda", dtype=torch.bfloat16) for _ in range(2)]
    with PolyTensor.plain_range(), PolyTensor.coefficient_autograd():
        y = PolyTensor(tuple(X)) @ w
    (dw,) = torch.autograd.grad(y.coeffs, [w], cot)
    for o in range(2):
        for part in (slice(0, 300), slice(rows - 300, rows)):
            want = X[o][part].float() @ w.detach().float()
            assert (y.coeffs[o].detach()[part].float() - want).abs().max() <= 2.0 ** -8 * want.abs().max()
    want = sum(sum(x[i:i + 65536].T.double() @ c[i:i + 65536].double() for i in range(0, rows, 65536))
               for x, c in zip(X, cot))
    # float32 sums of 3.6 million terms of magnitude one, rounded to bfloat16
    assert (dw.double() - want).abs().max() <= 2.0 ** -7 * want.abs().max()


# float32 rows of no whole vectors, either side of the size from which they are copied with padded rows.
@pytest.mark.parametrize("m,n,k", [(257, 259, 255), (300, 1001, 301)])
@pytest.mark.parametrize("plain", [True, False])
def test_float_rows_padded_by_size(m, n, k, plain):
    degree, tol = 3, 1e-5
    A, B = _series((m, k), degree, 1, torch.float32), _series((k, n), degree, 2, torch.float32)
    if plain:
        B = B[:1]
    b = B[0].cuda() if plain else PolyTensor(tuple(c.cuda() for c in B))
    with torch.no_grad(), PolyTensor.plain_range():
        got = PolyTensor(tuple(c.cuda() for c in A)) @ b
    up = lambda cs: [c.double() for c in cs]   # noqa: E731
    want = [c @ up(B)[0] for c in up(A)] if plain else oracle.matmul(up(A), up(B))
    for o in range(degree + 1):
        assert (got.coeffs[o].cpu().double() - want[o]).abs().max() <= tol * want[o].abs().max(), o


# 16-bit products of few tiles, whose workgroups split the contraction in two: below and from 16 chunks of 32,
# an odd number of them, halves that end inside a term of a sum, ragged sides. Sums in float32, rounded once.
@pytest.mark.parametrize("dtype,tol", [(torch.bfloat16, 2.0 ** -8), (torch.float16, 2.0 ** -10)])
@pytest.mark.parametrize("m,n,k,terms", [(1, 8, 480, 1), (3, 130, 512, 1), (130, 65, 520, 2), (257, 129, 1001, 3),
                                         (64, 264, 168, 3), (128, 128, 33, 9), (40, 40, 2056, 4)])
def test_split_contraction(dtype, tol, m, n, k, terms):
    g = torch.Generator().manual_seed(k)
    draw = lambda *shape: (torch.randn(*shape, generator=g, dtype=torch.float64)).to(dtype)   # noqa: E731
    A, B = [draw(1, m, k) for _ in range(terms)], [draw(1, k, n) for _ in range(terms)]
    cu = lambda xs: [x.cuda() for x in xs]   # noqa: E731
    flip = lambda xs: [x.transpose(1, 2).contiguous() for x in xs]   # noqa: E731
    want = sum(a.double() @ b.double() for a, b in zip(A, B))
    for a, b, ta, tb in ((A, B, False, False), (A, flip(B), False, True), (flip(A), B, True, False)):
        got = _ops.matmul_order_sum(cu(a), cu(b), ta, tb).cpu().double()
        assert (got - want).abs().max() <= tol * want.abs().max(), (ta, tb)
    for trans_b in (False, True):
        got = _ops.cauchy_matmul(cu(A), cu(flip(B[:1]) if trans_b else B[:1]), terms - 1, trans_b).cpu().double()
        for o in range(terms):
            want_o = A[o].double() @ B[0].double()
            assert (got[o] - want_o).abs().max() <= tol * want_o.abs().max(), (o, trans_b)


# Products with an ordinary operand on both sides of the rule that sends them order by order: small matrices in
# batches, short contractions on large sides (the wide 16-bit tiles to degree 4, the narrow ones past it), both
# operands ordinary, and long contractions at the edges of the order-by-order tiles. Against float64 of the stored
# inputs, relative to the largest value: one rounding to the storage type, float32 sums of k terms of magnitude one.
@pytest.mark.parametrize("dtype,tol", [(torch.float32, 1e-5), (torch.bfloat16, 2.0 ** -8), (torch.float16, 2.0 ** -11 + 1e-5)])
@pytest.mark.parametrize("m,k,n,batch,degree", [
    (16, 16, 16, 300, 8), (1, 8, 300, 40, 1), (65, 24, 33, 17, 5), (300, 8, 264, 2, 4), (257, 40, 513, 1, 6),
    (70, 16, 64, 1, 0), (129, 1000, 264, 1, 3), (200, 4096, 65, 2, 8), (1, 1024, 640, 1, 2), (520, 513, 260, 3, 1)])
def test_ordinary_operand_routes(dtype, tol, m, k, n, batch, degree):
    g = torch.Generator().manual_seed(m + k + n)
    A = [torch.randn(batch, m, k, generator=g).to(dtype) for _ in range(degree + 1)]
    B = [(torch.randn(batch, k, n, generator=g) / k ** 0.5).to(dtype) for _ in range(degree + 1)]
    cu = lambda xs: [x.cuda() for x in xs]   # noqa: E731
    for a, b in ((A, B[:1]), (A[:1], B), (A[:1], B[:1]), (A, [B[0][:1]])):
        for trans_b in (False, True):
            got = _ops.cauchy_matmul(cu(a), cu([x.transpose(1, 2).contiguous() for x in b] if trans_b else b), degree, trans_b)
            for o in range(degree + 1):
                if o >= max(len(a), len(b)):
                    assert not got[o].any()
                    continue
                want = a[o if len(a) > 1 else 0].double() @ b[o if len(b) > 1 else 0].double()
                err = (got[o].cpu().double() - want).abs().max() / want.abs().max()
                assert err <= tol, (len(a), len(b), trans_b, o, err)


# More tiles than a launch along one dimension holds (2^32 threads): one row each of 65535 matrices by a shared one.
@pytest.mark.parametrize("dtype,tol", [(torch.bfloat16, 2.0 ** -8), (torch.float32, 1e-5)])
def test_many_small_matrices(dtype, tol):
    batch, k, n, degree = 65535, 8, 4096, 8
    g = torch.Generator(device="cuda").manual_seed(0)
    A = [torch.randn(batch, 1, k, generator=g, device="cuda").to(dtype) for _ in range(degree + 1)]
    b = torch.randn(1, k, n, generator=g, device="cuda").to(dtype)
    got = _ops.cauchy_matmul(A, [b], degree, False)
    for o in range(degree + 1):
        for part in (slice(0, 300), slice(30000, 30300), slice(batch - 300, batch)):
            want = A[o][part, 0].double() @ b[0].double()
            err = (got[o][part, 0].double() - want).abs().max() / want.abs().max()
            assert err <= tol, (o, err)


# float32 rows of no whole vectors from 2^28 multiply-adds: contractions either side of 128, and few multiply-adds
# for an element, where they are read as they are.
@pytest.mark.parametrize("m,n,k", [(520, 1025, 127), (515, 1025, 129), (5, 4097, 4097), (31, 1025, 4097)])
def test_float_rows_by_contraction_and_reuse(m, n, k):
    degree, tol = 3, 1e-5
    A, B = _series((m, k), degree, 1, torch.float32), _series((k, n), degree, 2, torch.float32)
    with torch.no_grad(), PolyTensor.plain_range():
        left, right = _poly(A) @ B[0].cuda(), A[0].cuda() @ _poly(B)
    for o in range(degree + 1):
        for got, want in ((left, A[o].double() @ B[0].double()), (right, A[0].double() @ B[o].double())):
            assert (got.coeffs[o].cpu().double() - want).abs().max() <= tol * want.abs().max(), o
