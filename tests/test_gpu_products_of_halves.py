"""Products of rows that hold values of very different size.  The hook they go through was that of products with two fp16 parts per value; it
multiplies as all products do, on three bf16 parts (csrc/gemm.hip), and what is asked for here holds for those."""
import pytest

import parity_cases as PC

pytestmark = pytest.mark.gpu


def _operands(m, n, k, tA, tB, gen):
    import torch
    A, B = torch.randn(m * k, device="cuda", generator=gen), torch.randn(n * k, device="cuda", generator=gen)
    return A, B, A.view(m, k) if tA else A.view(k, m).t(), B.view(n, k) if not tB else B.view(k, n).t()


def _product(m, n, k, tA, tB, A, B):
    import torch
    C = torch.full((m * n + 4,), 7.0, device="cuda")
    PC.pkg().capi.probe_product_of_halves(C, m, n, k, A, tA, B, tB)
    assert bool((C[m * n:] == 7.0).all())
    return C[:m * n].view(n, m).t().double()


def _bound(A, B):
    """Of a value 23 of 24 bits are kept, the product of the low parts is left out: 4 * 2^-23 per term, less than the (k + 2) * 2^-24 of fp32
    sums in any order.  Below 2^-10 of its row's peak a value is off by 2^-35 of that peak, which no value of the row exceeds."""
    a, b = A.double().abs(), B.double().abs()
    return ((A.shape[1] + 2) * 2.0 ** -24 * (a @ b.t()) +
            2.0 ** -35 * (a.amax(1, keepdim=True) * b.sum(1) + a.sum(1, keepdim=True) * b.amax(1)) + A.shape[1] * 2.0 ** -149)


# 64 x 64 tiles and 128 x 128 on eight waves (224 tiles and more), every orientation, lines of no multiple of four, k that ends one to
# three values into a tile, rows fewer than a vector
SIZES = [(700, 1000, 128), (701, 999, 129), (1030, 1031, 131), (3, 30000, 160), (2, 30001, 163), (29000, 3, 130), (2050, 1500, 382),
         (2050, 1795, 300), (2047, 1793, 257), (1936, 6000, 256), (515, 7200, 1025)]


@pytest.mark.parametrize("tA,tB", [(True, False), (False, False), (False, True)])
@pytest.mark.parametrize("m,n,k", SIZES)
@pytest.mark.parametrize("what", ["plain", "exponents", "zero rows", "late", "outliers", "tiny"])
def test_within_the_bound_of_fp32_sums(m, n, k, tA, tB, what):
    """Rows whose sample of 64 values tells nothing about the others: zeros throughout, zeros but for one value, one value 2^40 times as large
    as all others, beside a column that leaves it out."""
    import torch
    print("halves", m, n, k, tA, tB, what, flush=True)
    gen = torch.Generator(device="cuda").manual_seed(m + 7 * n + 31 * k)
    A, B, a, b = _operands(m, n, k, tA, tB, gen)
    at = k // 4 if k >= 300 else k - 1 if k % 32 else 40  # in neither tile that is looked at, where there is one
    if what == "exponents":
        A *= torch.exp2(torch.randint(-9, 10, A.shape, device="cuda", generator=gen).float())
        a *= torch.exp2(torch.randint(-30, 31, (m, 1), device="cuda", generator=gen).float())
        b *= torch.exp2(torch.randint(-30, 31, (n, 1), device="cuda", generator=gen).float())
    elif what == "zero rows":
        a[::3], b[::5] = 0.0, 0.0
    elif what == "late":
        a[m - 1], b[n - 1] = 0.0, 0.0
        a[m - 1, at], b[n - 1, k - 1] = 1e-25, 3e20
    elif what == "outliers":
        a[m // 2, at] *= 2.0 ** 40
        b[n - 1, at] = 0.0
    elif what == "tiny":
        a *= 2.0 ** -126
        b *= 2.0 ** 60
    C = _product(m, n, k, tA, tB, A, B)
    bound = _bound(a, b)
    if what == "outliers":  # where the outlier meets a zero, the others keep their bits
        rest = a.clone()
        rest[m // 2, at] = 0.0
        bound[:, n - 1] = _bound(rest, b)[:, n - 1]
    assert bool(((C - a.double() @ b.double().t()).abs() <= bound).all())


@pytest.mark.parametrize("m,n,k,tA,tB", [(700, 1000, 130, True, False), (2050, 1500, 382, False, True), (1030, 1031, 200, False, False)])
def test_infinite_and_missing_values(m, n, k, tA, tB):
    """As a sum of single terms has them; the sums beside them keep their bound."""
    import torch
    gen = torch.Generator(device="cuda").manual_seed(k)
    A, B, a, b = _operands(m, n, k, tA, tB, gen)
    a[0, 0], a[1, k - 1], a[m - 1, k // 2], b[n - 1, 1] = float("inf"), -float("inf"), float("nan"), float("inf")
    C = _product(m, n, k, tA, tB, A, B)
    assert bool(C[m - 1].isnan().all()) and bool((~C[:, n - 1].isfinite()).all())
    assert torch.equal(C[0, :n - 1].isposinf(), b[:n - 1, 0] > 0) and torch.equal(C[1, :n - 1].isneginf(), b[:n - 1, k - 1] > 0)
    inner = slice(2, m - 1), slice(0, n - 1)
    assert bool(((C - a.double() @ b.double().t()).abs()[inner] <= _bound(a[2:m - 1], b[:n - 1])).all())


@pytest.mark.parametrize("k", [128, 200, 382, 1024, 4000])
def test_no_further_from_64_bits_than_three_parts(k):
    import torch
    m, n = 520, 2100
    gen = torch.Generator(device="cuda").manual_seed(k)
    A, B, a, b = _operands(m, n, k, True, False, gen)
    for f in (lambda x: x, torch.sigmoid):
        bf = f(B)
        want = a.double() @ bf.view(n, k).double().t()
        other = torch.empty(m * n, device="cuda")
        PC.pkg().capi.matrix_product(other, m, n, k, A, True, bf, False, False)
        error = (_product(m, n, k, True, False, A, bf) - want).norm()
        assert error <= (other.view(n, m).t().double() - want).norm()
