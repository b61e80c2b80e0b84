"""The wide A^T B products of three bf16 parts (tcc_dense_tn, tcc_gcn_relu_grad):
the edges of the blocks and of the 32-row steps, values that do not survive a
split, and whole numbers, against float64.

An element's error is bounded by its sum of |a b|: the three part products left
out come to at most 2^-24 of each product (for a and b in [1, 2) the middle
parts are at most 2^-8 and the low parts 2^-17), a step's six additions of 32
products each lose at most one unit in the last place, 2^-23, of it, and the
additions of steps and splits (at most 35 steps here) half a unit: below 2^-18
in all."""

import pytest
import torch

pytestmark = pytest.mark.gpu

BOUND = 2.0**-18


def _check(C, A, B):
    A, B = A.double().cpu(), B.double().cpu()
    want, mag = A.t() @ B, A.abs().t() @ B.abs()
    assert ((C.double().cpu() - want).abs() <= BOUND * mag).all()


@pytest.mark.parametrize("K", [1, 31, 32, 33, 65, 1100])
@pytest.mark.parametrize("M,N", [(17, 300), (64, 129), (65, 256), (112, 257), (113, 255), (129, 130), (300, 200),
                                 (200, 40)])
def test_edges(gpu, K, M, N):
    from tcc_amd import swtcf

    g = torch.Generator(device="cuda").manual_seed(K + M)
    A = torch.randn(K, M, generator=g, device="cuda")
    B = torch.randn(K, N, generator=g, device="cuda")
    C = swtcf.dense_tn(A, B)
    _check(C, A, B)
    assert torch.equal(swtcf.dense_tn(A, B), C)
    # rows of another stride and alignment
    Aw = torch.randn(K, M + 3, generator=g, device="cuda")
    Bw = torch.randn(K, N + 5, generator=g, device="cuda")
    _check(swtcf.dense_tn(Aw[:, 1: M + 1], Bw[:, 3: N + 3]), Aw[:, 1: M + 1], Bw[:, 3: N + 3])
    # whole numbers are exact
    Ai = torch.randint(-60, 61, (K, M), generator=g, device="cuda").float()
    Bi = torch.randint(-200, 201, (K, N), generator=g, device="cuda").float()
    assert torch.equal(swtcf.dense_tn(Ai, Bi).double(), Ai.double().t() @ Bi.double())


@pytest.mark.parametrize("bits", [(24, 1), (1, 24), (12, 12), (17, 7), (8, 16)])
def test_every_part_counts(gpu, bits):
    """One product a sum, of whole numbers of 24 significant bits in all, which
    the middle and low parts hold most of: exact in both operands' parts."""
    from tcc_amd import swtcf

    def whole(shape, n):  # odd numbers of n bits
        return (torch.randint(1 << (n - 1), 1 << n, shape, generator=g) | 1).float()

    g = torch.Generator().manual_seed(bits[0])
    K, M, N = 300, 130, 270
    A, B = whole((K, M), bits[0]), whole((K, N), bits[1])
    B[torch.arange(K).unsqueeze(1) != torch.arange(N)] = 0.0  # row k is column k's only one
    assert torch.equal(swtcf.dense_tn(A.cuda(), B.cuda()).double().cpu(), A.double().t() @ B.double())
    A, B = whole((K, M), bits[1]), whole((K, N), bits[0])
    A[torch.arange(K).unsqueeze(1) != torch.arange(M)] = 0.0
    assert torch.equal(swtcf.dense_tn(A.cuda(), B.cuda()).double().cpu(), A.double().t() @ B.double())
    AX, W1 = whole((500, 100), bits[0]), whole((100, 200), bits[1])
    for one in (0, 57, 99):
        X = torch.zeros_like(AX)
        X[:, one] = AX[:, one]
        H, _ = swtcf.gcn_relu_forward(X.cuda(), W1.cuda(), torch.ones(200, 1).cuda())
        assert torch.equal(H.double().cpu(), X.double() @ W1.double())


def _special(kind, A, B):
    K = A.shape[0]
    if kind == "inf":
        A[K // 2, 3] = float("inf")
    elif kind == "inf in the last row":
        B[K - 1, 5] = float("-inf")
    elif kind == "nan":
        B[K // 3, 40] = float("nan")
    elif kind == "nan of low bits":  # rounds to an infinity if its bits are only cut
        A.view(torch.int32)[K // 3, 7] = 0x7F800001
    elif kind == "largest":  # rounds up to an infinity in 8 bits
        A[::7] = torch.finfo(torch.float32).max * torch.sign(A[::7])
        B *= 1e-30
    elif kind == "tiny":
        A *= 1e-36
        B *= 1e10
    elif kind == "tiny columns":
        A[:, 5] *= 1e-37
        B[:, 9] *= 1e-38


KINDS = ["inf", "inf in the last row", "nan", "nan of low bits", "largest", "tiny", "tiny columns"]


@pytest.mark.parametrize("kind", KINDS)
def test_values_past_a_split(gpu, kind):
    from tcc_amd import swtcf

    K, M, N = 77, 100, 70
    g = torch.Generator().manual_seed(5)
    A, B = torch.randn(K, M, generator=g), torch.randn(K, N, generator=g)
    _special(kind, A, B)
    got = swtcf.dense_tn(A.cuda(), B.cuda()).double().cpu()
    A, B = A.double(), B.double()
    want = A.t() @ B
    assert torch.equal(torch.isnan(got), torch.isnan(want))
    assert torch.equal(torch.isinf(got), torch.isinf(want))
    inf = torch.isinf(want)
    assert torch.equal(got[inf], want[inf])
    mag = A.abs().t() @ B.abs()
    ok = torch.isfinite(want)
    # subnormal products lose at most half of the smallest number each
    assert ((got - want)[ok].abs() <= BOUND * mag[ok] + K * 2.0**-126).all()


def _hide(A, B, k, e, step):
    """Row k of A becomes 2^e and a fraction, and in every `step`th column of B
    only row k is left, of 2^100: there the small elements are the result,
    though their columns hold ordinary ones too."""
    A[k] = (1 + torch.rand(A.shape[1], generator=torch.Generator().manual_seed(1))) * 2.0**e
    B[:, ::step] = 0.0
    B[k, ::step] = 2.0**100 * (1 + B[k + 1, 1].abs())


@pytest.mark.parametrize("small", ["A", "B"])
@pytest.mark.parametrize("e", [-109, -112, -120, -133, -140])
def test_small_elements_among_ordinary_ones(gpu, e, small):
    from tcc_amd import swtcf

    for K, M, N in ((40, 64, 257), (70, 100, 256), (1100, 300, 300)):
        g = torch.Generator().manual_seed(K)
        A, B = torch.randn(K, M, generator=g), torch.randn(K, N, generator=g)
        _hide(*((A, B) if small == "A" else (B, A)), K // 2, e, 7)
        _check(swtcf.dense_tn(A.cuda(), B.cuda()), A, B)


@pytest.mark.parametrize("C", [1, 2, 3, 8])
@pytest.mark.parametrize("e", [-109, -115, -140])
def test_relu_gradient_small_elements(gpu, e, C):
    """One row of dOut1, and one of AX, too small to split."""
    from tcc_amd import swtcf

    K, F, Hd = 300, 113, 258
    for small in ("AX", "dOut1"):
        g = torch.Generator().manual_seed(3)
        AX, G, W2 = (torch.randn(s, generator=g) for s in ((K, F), (K, C), (Hd, C)))
        H = torch.rand(K, Hd, generator=g) + 0.5
        if small == "AX":
            AX[9] = (1 + torch.rand(F, generator=g)) * 2.0**e
            G[9] = 2.0**100
            H[:, ::5] = 0.0  # in these columns of dOut1 only row 9 is left
            H[9] = 1.0
        else:
            G[9] = (1 + torch.rand(C, generator=g)) * 2.0**e
            W2 = W2.abs()
            AX[:, ::5] = 0.0
            AX[9, ::5] = 2.0**100
        dW1, _ = swtcf.gcn_relu_grad(AX.cuda(), H.cuda(), G.cuda(), W2.cuda())
        # the kernel's own dOut1, a sum of C rounded products
        d = torch.where(H > 0, G.double() @ W2.double().t(), torch.zeros((), dtype=torch.float64))
        dmag = torch.where(H > 0, G.double().abs() @ W2.double().abs().t(), torch.zeros((), dtype=torch.float64))
        want, mag = AX.double().t() @ d, AX.double().abs().t() @ dmag
        # below 2^-126 each of the C additions of dOut1 rounds to a multiple of
        # 2^-149, by half of it at most
        sub = AX.double().abs().sum(0).unsqueeze(1) * (C * 2.0**-149)
        assert ((dW1.double().cpu() - want).abs() <= 2 * BOUND * mag + sub).all(), small


@pytest.mark.parametrize("C", [1, 2, 3, 8])
@pytest.mark.parametrize("K", [33, 1100])
def test_relu_gradient_edges(gpu, K, C):
    """dW1 and dW2 with an infinity in G's and H's last row, and without."""
    from tcc_amd import swtcf

    F, Hd = 113, 258
    g = torch.Generator().manual_seed(K + C)
    AX, G, W2 = (torch.randn(s, generator=g) for s in ((K, F), (K, C), (Hd, C)))
    H = torch.randn(K, Hd, generator=g).relu_()
    for special in (False, True):
        if special:
            G[K - 1, C - 1] = float("inf")
            H[K - 1, 2] = float("inf")
            H[K - 1, 3:] += 0.5
            H[K - 1, :2] = 0.25
        dW1, dW2 = swtcf.gcn_relu_grad(AX.cuda(), H.cuda(), G.cuda(), W2.cuda())
        d = (G.double() @ W2.double().t()).where(H > 0, torch.zeros((), dtype=torch.float64))
        dmag = (G.double().abs() @ W2.double().abs().t()).where(H > 0, torch.zeros((), dtype=torch.float64))
        for got, want, mag in ((dW1, AX.double().t() @ d, AX.double().abs().t() @ dmag),
                               (dW2, H.double().t() @ G.double(), H.double().abs().t() @ G.double().abs())):
            got = got.double().cpu()
            fin = torch.isfinite(want)
            assert torch.equal(torch.isfinite(got), fin)
            assert torch.equal(torch.isinf(got), torch.isinf(want))
            # d itself is a sum of C rounded products
            assert ((got - want)[fin].abs() <= 2 * BOUND * mag[fin]).all()
        assert special or bool(torch.isfinite(dW1).all())


@pytest.mark.parametrize("C", [1, 2, 4])
@pytest.mark.parametrize("K", [1, 63, 64, 65, 20_000])
@pytest.mark.parametrize("F,Hd", [(3, 5), (32, 256), (33, 255), (64, 32), (65, 33), (97, 130), (100, 256), (128, 100)])
def test_relu_forward_edges(gpu, K, F, Hd, C):
    """H and H W2 at the edges of the forward's steps and blocks, with rows and
    columns too small to split and (in the last pass) an infinity and a NaN."""
    from tcc_amd import swtcf

    g = torch.Generator(device="cuda").manual_seed(K + F + C)
    for special in range(3):
        AX = torch.randn(K, F + 1, generator=g, device="cuda")[:, :F] if special == 1 else \
            torch.randn(K, F, generator=g, device="cuda")
        W1, W2 = torch.randn(F, Hd, generator=g, device="cuda"), torch.randn(Hd, C, generator=g, device="cuda")
        if special == 1:
            AX[K // 2] *= 1e-33
            W1[:, Hd // 2] *= 1e-34
        if special == 2:
            AX[K - 1, F // 2] = float("inf")
            AX[0, 0] = float("nan")
        H, XW = swtcf.gcn_relu_forward(AX, W1, W2)
        pre = AX.double() @ W1.double()
        want = torch.where(pre < 0, torch.zeros_like(pre), pre)
        fin = torch.isfinite(want)
        assert torch.equal(torch.isnan(H), torch.isnan(want)) and torch.equal(torch.isinf(H), torch.isinf(want))
        mag = AX.double().abs() @ W1.double().abs()
        assert ((H.double() - want)[fin].abs() <= BOUND * mag[fin] + F * 2.0**-126).all()
        xw, xmag = H.double() @ W2.double(), H.double().abs() @ W2.double().abs()
        ok = torch.isfinite(xw)
        assert torch.equal(torch.isfinite(XW), ok)
        assert ((XW.double() - xw)[ok].abs() <= Hd * 2.0**-23 * xmag[ok] + Hd * 2.0**-126).all()


@pytest.mark.parametrize("small", ["AX", "W1"])
@pytest.mark.parametrize("e", [-109, -112, -120, -133, -140])
@pytest.mark.parametrize("K,F,Hd", [(5, 20, 33), (700, 100, 256), (20_000, 128, 100)])
def test_relu_forward_small_elements(gpu, K, F, Hd, e, small):
    from tcc_amd import swtcf

    g = torch.Generator().manual_seed(K)
    AX, W1 = torch.randn(K, F, generator=g), torch.rand(F, Hd, generator=g) + 0.5
    if small == "AX":
        _hide(AX.t(), W1, F // 2, e, 7)
    else:
        _hide(W1, AX.t(), F // 2, e, 7)
    H, _ = swtcf.gcn_relu_forward(AX.cuda(), W1.cuda(), torch.ones(Hd, 1).cuda())
    want = (AX.double() @ W1.double()).clamp_min(0)
    mag = AX.double().abs() @ W1.double().abs()
    assert ((H.double().cpu() - want).abs() <= BOUND * mag).all()


@pytest.mark.parametrize("terms", [1, 2, 3])
def test_few_terms_are_fp32_products(gpu, terms):
    """Sums of one to three products are as fp32 MFMA gives them: exact
    products, each addition rounded to nearest."""
    from tcc_amd import swtcf

    g = torch.Generator(device="cuda").manual_seed(terms)
    A, B = torch.randn(terms, 130, generator=g, device="cuda"), torch.randn(terms, 257, generator=g, device="cuda")
    C = swtcf.dense_tn(A, B).double()
    assert ((C - A.double().t() @ B.double()).abs() <= terms * 2.0**-24 * (A.double().abs().t() @ B.double().abs())).all()
    AX, W1 = torch.randn(3000, terms, generator=g, device="cuda"), torch.randn(terms, 200, generator=g, device="cuda")
    H, _ = swtcf.gcn_relu_forward(AX, W1, torch.randn(200, 2, generator=g, device="cuda"))
    want, mag = (AX.double() @ W1.double()).clamp_min(0), AX.double().abs() @ W1.double().abs()
    assert ((H.double() - want).abs() <= terms * 2.0**-24 * mag).all()
