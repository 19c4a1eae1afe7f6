"""mykfa_gemm against float64 products: each operand layout and result type at the edges of its
tiles (256, 128, 64), K remainders of a stage and of 8, one K stage and many, K splits, several
units per workgroup, padded columns, and an addend. Bounds: bf16 results within one rounding
(2^-8 of the value) plus the fp32 sum's own error; fp32 results within the sum's error, which for
k products of N(0, 1) values is below k 2^-24 of sqrt(k)."""

import pytest
import torch

from myk_llm_amd.gemm import gemm
from myk_llm_amd.muon import batched_newton_schulz_orthogonalize, batched_syrk
from oracle import muon as om

pytestmark = pytest.mark.gpu


def _padded(g, b, rows, cols, fill=0.0):
    """(b, rows, cols) N(0, 1) bf16 rows padded to a multiple of 8 with `fill`."""
    x = torch.full((b, rows, (cols + 7) // 8 * 8), fill, dtype=torch.bfloat16)
    x[..., :cols] = torch.randn(b, rows, cols, generator=g).to(torch.bfloat16)
    return x.cuda()


def _close(got, exp, k, bf16):
    bound = exp.abs() * (2.0 ** -8 if bf16 else 0) + k * 2.0 ** -24 * k ** 0.5 * 4 + 1e-30
    assert ((got.double() - exp).abs() <= bound).all(), ((got.double() - exp).abs() / bound).max()


@pytest.mark.parametrize("b, m, n, k", [
    (1, 1, 8, 8), (1, 64, 64, 64), (3, 65, 72, 63), (2, 129, 200, 129), (9, 257, 264, 328), (1, 1000, 2056, 72),
    (1, 2048, 16640, 192), (1, 256, 512, 4104), (2, 127, 130, 2000), (1, 300, 33, 8200), (7, 1024, 2048, 320),
    (1, 2500, 4000, 8200), (1, 2500, 7600, 8200)])  # K parts over two rounds, and a last round in quarters
def test_products_match_float64(b, m, n, k):
    print(f"gemm {b} x {m} x {n} x {k}", flush=True)
    g = torch.Generator().manual_seed(m + n + k)
    a, w = _padded(g, b, m, k), _padded(g, b, k, n)
    exp = a[..., :k].double() @ w[..., :n].double()
    n8 = (n + 7) // 8 * 8
    c = torch.full((b, m, n8), float("nan"), dtype=torch.bfloat16, device="cuda")
    gemm(a, w, c, m, n, k)
    _close(c[..., :n], exp, k, True)
    assert (c[..., n:] == 0).all()  # a row's pad is stored as zeros
    add = _padded(g, b, m, n)
    gemm(a, w, c, m, n, k, add=add, alpha=-0.5, beta=2.0)
    _close(c[..., :n], 2.0 * add[..., :n].double() - 0.5 * exp, k, True)
    wt = _padded(g, b, n, k)
    gemm(a, wt, c, m, n, k, b_transposed=True, alpha=2.0)
    _close(c[..., :n], 2.0 * (a[..., :k].double() @ wt[..., :k].double().transpose(1, 2).contiguous()), k, True)
    at = _padded(g, b, k, m, fill=float("nan"))  # columns past m reach no result
    acc = torch.randn(b, m, n8, device="cuda")
    old = acc.clone()
    prod = at[..., :m].double().transpose(1, 2).contiguous() @ w[..., :n].double()
    gemm(at, w, acc, m, n, k, a_transposed=True, beta=1.0)
    _close(acc[..., :n], prod + old[..., :n].double(), k, False)
    acc.fill_(float("nan"))
    gemm(at, w, acc, m, n, k, a_transposed=True)
    _close(acc[..., :n], prod, k, False)


@pytest.mark.parametrize("b, m, k", [(1, 8, 8), (5, 63, 65), (2, 129, 100), (30, 257, 640), (3, 132, 72)])
def test_symmetric_products(b, m, k):
    g = torch.Generator().manual_seed(m + k)
    x = torch.randn(b, m, k, generator=g).to(torch.bfloat16).cuda()
    out = batched_syrk(x)
    exp = x.double() @ x.double().transpose(1, 2).contiguous()
    _close(out, exp, k, True)
    assert torch.equal(out, out.transpose(1, 2))
    res = batched_syrk(x, bias=out, alpha=0.25, beta=-1.5)
    _close(res, 0.25 * exp - 1.5 * out.double(), k, True)
    assert torch.equal(res, res.transpose(1, 2))


@pytest.mark.parametrize("shape, steps, transposed", [((3, 130, 190), 5, None), ((2, 201, 77), 4, None), ((1, 8, 1024), 1, None),
                                                     ((2, 65, 64), 5, False), ((2, 96, 257), 3, True), ((4, 512, 512), 5, None)])
def test_newton_schulz_odd_shapes(shape, steps, transposed):
    """Against the oracle's float32 iteration: the bf16 roundings between the products, 2^-9
    relative each, grow at most by the quintic's slope (3.45) a step."""
    g = torch.Generator().manual_seed(steps)
    x = torch.randn(*shape, generator=g).to(torch.bfloat16)
    kept = x.clone()
    dev = x.cuda()
    got = batched_newton_schulz_orthogonalize(dev, steps, transposed)
    assert torch.equal(dev.cpu(), kept) and got.is_contiguous()
    exp = torch.stack([om.newton_schulz_reference(m, steps) for m in x.float()])
    err = (got.float().cpu() - exp).norm() / exp.norm()
    assert err <= 2.0 ** -9 * 3.45 * steps * 2, err


@pytest.mark.parametrize("m, n, k", [(50257, 1024, 65), (4136, 4096, 129), (4096, 4136, 1)])
def test_quarters_past_an_edge(m, n, k):
    """The last units of a product run as quarters, some of which begin past M or N, with one row of K in
    the last stage: they store nothing, and the others' results are whole."""
    print(f"quarters past an edge {m} x {n} x {k}", flush=True)
    g = torch.Generator().manual_seed(m + k)
    a, w = _padded(g, 1, k, m), _padded(g, 1, k, n)
    c = torch.full((1, m, (n + 7) // 8 * 8), float("nan"), device="cuda")
    gemm(a, w, c, m, n, k, a_transposed=True)
    _close(c[..., :n], a[..., :m].double().transpose(1, 2).contiguous() @ w[..., :n].double(), k, False)
    b = torch.full_like(c, float("nan"), dtype=torch.bfloat16)
    rows = a[..., :m].transpose(1, 2).contiguous()
    x = torch.zeros(1, m, (k + 7) // 8 * 8, dtype=torch.bfloat16, device="cuda")
    x[..., :k] = rows
    gemm(x, w, b, m, n, k)
    _close(b[..., :n], rows.double() @ w[..., :n].double(), k, True)


@pytest.mark.parametrize("m, n, k", [(70, 33, 72), (300, 33, 8200), (700, 2500, 4104), (4136, 4099, 136)])
def test_pads_are_zeros(m, n, k):
    """Every bf16 result but the symmetric one pads its rows with zeros: with B's pads not a number, with A's
    rows infinite against the rows that B has not, with an addend whose pads are not a number."""
    g = torch.Generator().manual_seed(m)
    a, w, wt = _padded(g, 1, m, k), _padded(g, 1, k, n, fill=float("nan")), _padded(g, 1, n, k)
    inf = a.clone()
    inf[0, 1::2, 3] = float("inf")
    n8 = (n + 7) // 8 * 8
    assert n8 > n
    for left, right, kw in ((a, w, {}), (inf, wt, {"b_transposed": True}), (a, w, {"add": _padded(g, 1, m, n, fill=float("nan")), "beta": 1.0})):
        c = torch.full((1, m, n8), 7.0, dtype=torch.bfloat16, device="cuda")
        gemm(left, right, c, m, n, k, **kw)
        assert (c[..., n:] == 0).all()
        assert not torch.isnan(c[0, 0, :n]).any()


def test_newton_schulz_of_more_matrices_than_a_grid_dimension():
    """Matrices of the first run, of the border and of the last one."""
    g = torch.Generator(device="cuda").manual_seed(0)
    x = torch.randn(65537, 8, 16, generator=g, device="cuda", dtype=torch.bfloat16)
    for steps in (1, 2):
        out = batched_newton_schulz_orthogonalize(x, steps)
        assert not torch.isnan(out).any()
        for b in (0, 32768, 65534, 65535, 65536):
            exp = om.newton_schulz_reference(x[b].float().cpu(), steps)
            err = (out[b].float().cpu() - exp).norm() / exp.norm()
            assert err <= 2.0 ** -9 * 3.45 * steps * 2, (b, err)
