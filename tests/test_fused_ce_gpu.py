"""Parity of the fused linear + cross-entropy (myk_llm_amd.fused_ce, csrc/fused_ce.hip) with
the CPU oracle (oracle/fused_ce.py) on identical seeded inputs.

- The CE row kernel against the float64 row oracle on the same logits: lse and ce within
  2e-5 relative (fp32 sums of fp32 exponentials), the in-place gradient within one storage
  ulp of each element, relative down to the type's subnormals (the target column adds the
  fp32 cancellation of softmax * scale' - scale); both the register-resident path
  (vocab <= 65536, multiple of 8) and the two-pass path (larger or unaligned rows), on
  N(0, 4^2) rows and on peaked rows whose probabilities reach far below fp16's range.
- The whole op against the reference's own test (tests/test_fused_ce.py:10-38), with its
  tolerances, and at the reference model's head shape (H = 1024, V = 65536).
"""

import sys

import numpy as np
import pytest
import torch

from _util import storage_ulp
from myk_llm_amd import _lib, fused_ce
from myk_llm_amd.fused_ce import _ce_rows, fused_linear_cross_entropy
from oracle import fused_ce as oc

pytestmark = pytest.mark.gpu


def _say(*a):
    print(*a, flush=True)
    sys.stdout.flush()


@pytest.mark.parametrize("rows,vocab,dtype,z,spread", [
    (64, 1000, torch.bfloat16, 0.0, 4.0),
    (37, 4096, torch.bfloat16, 1e-3, 4.0),
    (16, 65536, torch.bfloat16, 1e-3, 4.0),
    (24, 12000, torch.bfloat16, 1e-3, 4.0),   # 32 columns per lane
    (8, 65536, torch.float16, 0.0, 4.0),
    (9, 100000, torch.bfloat16, 1e-4, 4.0),   # two-pass, 16-byte accesses
    (11, 1003, torch.bfloat16, 1e-3, 4.0),    # two-pass, element accesses
    (5, 8, torch.bfloat16, 0.0, 4.0),
    # peaked rows: probabilities far below fp16's normal range
    (16, 65536, torch.bfloat16, 1e-3, 8.0),   # some chunks hold p < 2^-63 (recomputed), most not
    (16, 65536, torch.bfloat16, 0.0, 20.0),   # nearly every chunk recomputed
    (16, 65536, torch.bfloat16, 1e-3, "dominant"),  # one logit 40 above N(0, 1) rows: p ~ 2^-58
])
def test_ce_rows_match_oracle(rows, vocab, dtype, z, spread):
    _say(f"ce rows {rows}x{vocab} {dtype} z={z} spread={spread}")
    g = torch.Generator().manual_seed(rows * 7 + vocab)
    if spread == "dominant":
        x = torch.randn(rows, vocab, generator=g)
        x[torch.arange(rows), torch.randint(0, vocab, (rows,), generator=g)] += 40.0
        x = x.to(dtype)
    else:
        x = (torch.randn(rows, vocab, generator=g) * spread).to(dtype)
    t = torch.randint(0, vocab, (rows,), generator=g)
    t[1::4] = -100
    scale = 1.0 / 123.0
    logits = x.cuda()
    ce = torch.empty(rows, device="cuda")
    lse = torch.empty(rows, device="cuda")
    _ce_rows(logits, t.cuda(), ce, lse, scale, z, -100)
    torch.cuda.synchronize()
    grad_ref, ce_ref, lse_ref = oc.ce_rows(x.double().numpy(), t.numpy(), scale, z)
    np.testing.assert_allclose(lse.cpu().double().numpy(), lse_ref, rtol=2e-5, atol=1e-6)
    np.testing.assert_allclose(ce.cpu().double().numpy(), ce_ref, rtol=2e-5, atol=2e-5)
    got = logits.float().cpu()
    ref = torch.tensor(grad_ref)
    # One storage ulp of the float64 value, relative everywhere down to a floor: fp16's
    # subnormal spacing (2^-24, all the type can hold there); for bf16, 2^-126, below which the
    # fp32 exponential itself flushes (as the reference's tl.exp does) and bf16 is subnormal.
    # The target column adds the fp32 cancellation of softmax * scale' - scale, as the
    # reference computes it: a few fp32 ulps of scale * (1 + 2 z |lse|).
    sub = 2.0 ** -24 if dtype == torch.float16 else 2.0 ** -126
    bound = storage_ulp(ref, dtype).double().clamp_min(sub)
    sup = torch.nonzero(t != -100)[:, 0]
    bound[sup, t[sup]] += 8 * 2.0 ** -24 * scale * (1 + 2 * z * torch.tensor(lse_ref).abs()[sup])
    err = (got.double() - ref).abs()
    _say(f"  grad max-abs {err.max().item():.3e}, max err/ulp {(err / storage_ulp(ref, dtype).double()).max():.3f}, "
         f"exact {(err == 0).double().mean().item() * 100:.2f}%")
    assert (err <= bound).all(), f"{(err > bound).sum().item()} gradient elements beyond one ulp"
    assert torch.equal(got[1::4], torch.zeros_like(got[1::4]))


def test_out_of_range_target_gives_nan_and_stays_in_bounds():
    x = torch.randn(3, 512).to(torch.bfloat16).cuda()
    guard = torch.full((2, 512), 7.0, dtype=torch.bfloat16, device="cuda")
    buf = torch.cat([x, guard])  # rows after the chunk must stay untouched
    t = torch.tensor([5, 512, -1], device="cuda")
    ce, lse = torch.empty(3, device="cuda"), torch.empty(3, device="cuda")
    _ce_rows(buf[:3], t, ce, lse, 1.0, 0.0, -100)
    torch.cuda.synchronize()
    assert torch.isfinite(ce[0]) and torch.isnan(ce[1]) and torch.isnan(ce[2])
    assert torch.equal(buf[3:], guard)


def test_deterministic():
    x = (torch.randn(32, 65536) * 3).to(torch.bfloat16).cuda()
    t = torch.randint(0, 65536, (32,)).cuda()
    outs = []
    for _ in range(3):
        lg = x.clone()
        ce, lse = torch.empty(32, device="cuda"), torch.empty(32, device="cuda")
        _ce_rows(lg, t, ce, lse, 0.01, 1e-3, -100)
        outs.append((lg, ce, lse))
    for o in outs[1:]:
        assert all(torch.equal(a, b) for a, b in zip(o, outs[0]))


@pytest.mark.parametrize("z_loss", [0.0, 1e-3])
def test_matches_reference_loss_and_gradients(z_loss):
    """tests/test_fused_ce.py:10-38, its shapes, seeds and tolerances."""
    torch.manual_seed(0)
    n, h, v = 300, 64, 1000
    hidden = torch.randn(n, h).cuda().requires_grad_(True)
    weight = (0.1 * torch.randn(v, h)).cuda().requires_grad_(True)
    targets = torch.randint(0, v, (n,)).cuda()
    targets[::7] = -100
    normalizer = 123.0
    loss, ce_sum, z_sum = fused_linear_cross_entropy(hidden, weight, targets, normalizer, z_loss, chunk_size=128)
    loss.backward()
    grads = hidden.grad.clone(), weight.grad.clone()

    hc = hidden.detach().cpu().requires_grad_(True)
    wc = weight.detach().cpu().requires_grad_(True)
    ref, ce_ref = oc.loss_reference(hc, wc, targets.cpu(), normalizer, z_loss)
    ref.backward()
    torch.testing.assert_close(loss.cpu(), ref, rtol=1e-3, atol=1e-3)
    torch.testing.assert_close(ce_sum.cpu(), ce_ref.detach(), rtol=1e-3, atol=1e-2)
    torch.testing.assert_close(grads[0].cpu(), hc.grad, rtol=2e-2, atol=2e-4)
    torch.testing.assert_close(grads[1].cpu(), wc.grad, rtol=2e-2, atol=2e-4)
    valid = targets.cpu() != -100
    logits = hc.detach().bfloat16().float() @ wc.detach().bfloat16().float().t()
    z_ref = torch.logsumexp(logits, -1)[valid].square().sum()
    torch.testing.assert_close(z_sum.cpu(), z_ref, rtol=1e-3, atol=1e-2)


def test_model_head_shape():
    """The reference model's head (hidden 1024, tied 64K vocabulary, configs/model/200m.yaml)
    on 4096 tokens in 2048-token chunks (train/config.py:79), bf16 hidden as under autocast:
    loss and gradients against the fp32 reference of tests/test_fused_ce.py:27-33."""
    _say("fused CE at H=1024, V=65536, 4096 tokens")
    g = torch.Generator().manual_seed(11)
    n, h, v = 4096, 1024, 65536
    hidden = torch.randn(n, h, generator=g).to(torch.bfloat16)
    weight = (0.05 * torch.randn(v, h, generator=g))
    targets = torch.randint(0, v, (n,), generator=g)
    targets[::9] = -100
    normalizer = float((targets != -100).sum())
    hd, wd = hidden.cuda().requires_grad_(True), weight.cuda().requires_grad_(True)
    loss, ce_sum, _ = fused_linear_cross_entropy(hd, wd, targets.cuda(), normalizer, 1e-4)
    loss.backward()
    torch.cuda.synchronize()
    # reference on the GPU in fp32 (bf16-rounded operands, exact in fp32), chunked by rows
    wb = wd.detach().bfloat16().float()
    hb = hd.detach().float()
    ce_tot, z_tot = 0.0, 0.0
    gh = torch.empty(n, h, device="cuda")
    gw = torch.zeros(v, h, device="cuda")
    for s0 in range(0, n, 1024):
        lg = (hb[s0:s0 + 1024] @ wb.t()).double()
        tt = targets[s0:s0 + 1024].cuda()
        valid = tt != -100
        lse = torch.logsumexp(lg, -1)
        ce = torch.where(valid, lse - lg.gather(1, tt.clamp_min(0)[:, None])[:, 0], 0.0)
        ce_tot += ce.sum().item()
        z_tot += (lse[valid] ** 2).sum().item()
        p = torch.softmax(lg, -1) * (1 + 2e-4 * lse)[:, None]
        p[valid.nonzero()[:, 0], tt[valid]] -= 1.0
        p[~valid] = 0
        p = (p / normalizer).float()
        gh[s0:s0 + 1024] = p @ wb
        gw += p.t() @ hb[s0:s0 + 1024]
    ref_loss = (ce_tot + 1e-4 * z_tot) / normalizer
    _say(f"  loss {loss.item():.6f} vs {ref_loss:.6f}; ce_sum {ce_sum.item():.3f} vs {ce_tot:.3f}")
    assert abs(loss.item() - ref_loss) <= 1e-3 * abs(ref_loss)
    assert abs(ce_sum.item() - ce_tot) <= 1e-3 * abs(ce_tot)
    for got, ref, name in ((hd.grad, gh, "d hidden"), (wd.grad, gw, "d weight")):
        err = (got.float() - ref).abs().max().item()
        _say(f"  {name}: max-abs {err:.3e} (max |ref| {ref.abs().max().item():.3e})")
        # the reference's gradient tolerance (tests/test_fused_ce.py:37-38) scaled to the
        # gradient's magnitude (1 / normalizer here, vs 1 / 123 there)
        torch.testing.assert_close(got.float(), ref, rtol=2e-2, atol=2e-2 * ref.abs().max().item())


@pytest.mark.parametrize("rows, vocab, stride", [(5, 1001, 1008), (3, 4095, 4096), (2, 7, 8), (4, 65535, 65544), (3, 32003, 32008)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_rows_with_a_vocabulary_tail(rows, vocab, stride, dtype):
    """Padded rows whose vocabulary is no multiple of 8 against the streaming kernel's elementwise
    result on unpadded rows (the same formula; one rounding of the 16-bit result apart), ignored
    and last-column targets included; the pad columns stay untouched."""
    g = torch.Generator().manual_seed(vocab)
    x = (4 * torch.randn(rows, vocab, generator=g)).to(dtype).cuda()
    targets = torch.randint(0, vocab, (rows,), generator=g).cuda()
    targets[0], targets[-1] = vocab - 1, -100
    padded = torch.full((rows, stride), 7.0, dtype=dtype, device="cuda")
    padded[:, :vocab] = x
    plain = torch.empty(rows * (vocab | 1) + rows, dtype=dtype, device="cuda").as_strided((rows, vocab), (vocab | 1, 1))
    plain.copy_(x)
    got, exp = (torch.empty(2, rows, device="cuda") for _ in range(2))
    fused_ce._ce_rows(padded[:, :vocab], targets, got[0], got[1], 0.5, 1e-3, -100)
    fused_ce._ce_rows(plain, targets, exp[0], exp[1], 0.5, 1e-3, -100)
    torch.testing.assert_close(got, exp, rtol=1e-5, atol=1e-5)
    ulp = 2.0 ** (-7 if dtype == torch.bfloat16 else -10)
    torch.testing.assert_close(padded[:, :vocab].float(), plain.float(), rtol=ulp, atol=2.0 ** -24)
    assert (padded[:, vocab:] == 7).all()


@pytest.mark.parametrize("tokens, width, vocab, chunk, keep", [(100, 72, 1003, 33, 1 << 30), (100, 72, 1003, 33, 1), (517, 64, 264, 128, 2 * 264 * 2 * 128),
                                                              (100, 72, 1003, None, 1 << 30)])
@pytest.mark.parametrize("dtypes", [(torch.float32, torch.float32), (torch.bfloat16, torch.bfloat16), (torch.float16, torch.float32)])
def test_kept_chunks_and_dtypes(monkeypatch, tokens, width, vocab, chunk, keep, dtypes):
    """One pass and several, the last one shorter, give the reference's loss and gradients; passes too
    large for the device's memory are taken back for passes of the default's tokens (here `chunk`; without one
    the call names 40)."""
    monkeypatch.setattr(fused_ce, "_KEEP_BYTES", keep)
    named = {"chunk_size": 40 if chunk is None else fused_ce._Unset(chunk)}
    real, refused, passes = fused_ce.gemm, [], []

    def scarce(a, b, c, m, n, k, **kw):
        if kw.get("a_transposed") and tokens > 500 and k > chunk:  # no memory for the larger passes
            refused.append(k)
            raise torch.OutOfMemoryError("planted")
        if kw.get("a_transposed"):
            passes.append(k)
        real(a, b, c, m, n, k, **kw)

    monkeypatch.setattr(fused_ce, "gemm", scarce)
    g = torch.Generator().manual_seed(tokens)
    hidden = torch.randn(tokens, width, generator=g).to(torch.bfloat16).to(dtypes[0]).cuda().requires_grad_()
    weight = (0.1 * torch.randn(vocab, width, generator=g)).to(torch.bfloat16).to(dtypes[1]).cuda().requires_grad_()
    targets = torch.randint(0, vocab, (tokens,), generator=g).cuda()
    targets[::7] = -100
    n = float((targets != -100).sum())
    loss, ce_sum, z_sum = fused_ce.fused_linear_cross_entropy(hidden, weight, targets, n, 1e-3, **named)
    (3.0 * loss).backward()
    assert refused == ([176] if tokens > 500 else [])
    assert passes == ([128] * 4 + [5] if tokens > 500 else [40, 40, 20] if chunk is None else [100] if keep > 1 else [33, 33, 33, 1])
    h, w = (x.detach().double().requires_grad_() for x in (hidden, weight))
    logits = h @ w.t()
    lse = torch.logsumexp(logits, -1)
    valid = targets != -100
    ce = (lse - logits.gather(1, targets.clamp_min(0)[:, None])[:, 0])[valid].sum()
    z = lse[valid].square().sum()
    exp = (ce + 1e-3 * z) / n
    (3.0 * exp).backward()
    for got, want in ((loss, exp), (ce_sum, ce), (z_sum, z)):
        torch.testing.assert_close(got.double(), want, rtol=2e-3, atol=0)
    for got, want in ((hidden.grad, h.grad), (weight.grad, w.grad)):
        assert got.dtype in dtypes
        err = (got.double() - want).norm() / want.norm()
        assert err < 1e-2, err  # bf16 logits and gradients: 2^-8 each


@pytest.mark.parametrize("shape", [(1000, 1024), (1000, 256), (1000, 512, 1), (512,)])
def test_weight_of_another_width_is_refused(shape):
    hidden = torch.randn(40, 512, dtype=torch.bfloat16, device="cuda")
    weight = torch.randn(*shape, dtype=torch.bfloat16, device="cuda")
    with pytest.raises(RuntimeError, match="shape|size|dim|2D|matri"):
        fused_linear_cross_entropy(hidden, weight, torch.zeros(40, dtype=torch.int64, device="cuda"), 40.0)


def _flat_view(x, offset):
    """x's values in a view that starts `offset` elements into a flat buffer."""
    flat = torch.zeros(offset + x.numel(), dtype=x.dtype, device=x.device)
    return flat[offset:].view(x.shape).copy_(x)


def _far_rows(x):
    """x's rows so far apart that a tile of 256 spans more than 2 GiB."""
    step = (1 << 22) + (1 << 15)
    return torch.empty(step * (x.shape[0] - 1) + x.shape[1], dtype=x.dtype, device=x.device).as_strided(x.shape, (step, 1)).copy_(x)


@pytest.mark.parametrize("tokens, hidden_as, weight_as", [
    (30, lambda x: x, lambda w: _flat_view(w, 1)), (30, lambda x: _flat_view(x, 3), lambda w: w),
    (1, lambda x: x.new_zeros(1, 65).as_strided((1, 64), (65, 1)).copy_(x), lambda w: w), (30, _far_rows, lambda w: w),
    (30, lambda x: x.t().contiguous().t(), lambda w: w.t().contiguous().t())])
def test_layouts_that_the_products_do_not_read(tokens, hidden_as, weight_as):
    """The same bits as for plain tensors: such layouts are copied, not refused."""
    g = torch.Generator().manual_seed(tokens)
    hidden = torch.randn(tokens, 64, generator=g).to(torch.bfloat16).cuda()
    weight = (0.1 * torch.randn(300, 64, generator=g)).to(torch.bfloat16).cuda()
    targets = torch.randint(0, 300, (tokens,), generator=g).cuda()
    results = []
    for h, w in ((hidden, weight), (hidden_as(hidden), weight_as(weight))):
        h, w = h.detach().requires_grad_(), w.detach().requires_grad_()
        loss, ce_sum, z_sum = fused_linear_cross_entropy(h, w, targets, float(tokens), 1e-3)
        results.append((loss, ce_sum, z_sum, *torch.autograd.grad(loss, (h, w))))
    assert all(torch.equal(a, b) for a, b in zip(*results))


@pytest.mark.parametrize("rows, vocab", [(7, 1003), (5, 32003), (3, 65535)])
@pytest.mark.parametrize("aligned", [True, False])
def test_gradients_of_a_vocabulary_tail_are_rounded_once(rows, vocab, aligned):
    """Rows whose vocabulary 8 does not divide, padded to aligned rows or not: the gradient off the target
    column is the fp32 value rounded once, half a bf16 ulp and the fp32 error itself, which is the exponent's:
    |x - lse| log2(e) below 64 in fp32 and the sum of the row, together below 2^-17 of the value (2^-9 ulp)."""
    g = torch.Generator().manual_seed(vocab)
    x = (3 * torch.randn(rows, vocab, generator=g)).to(torch.bfloat16)
    stride = (vocab + 7) // 8 * 8 if aligned else vocab
    logits = torch.empty(rows, stride, dtype=torch.bfloat16, device="cuda")[:, :vocab].copy_(x)
    targets = torch.randint(0, vocab, (rows,), generator=g)
    ce, lse = torch.empty(rows, device="cuda"), torch.empty(rows, device="cuda")
    _ce_rows(logits, targets.cuda(), ce, lse, 1.0 / 7, 1e-3, -100)
    ref = torch.tensor(oc.ce_rows(x.double().numpy(), targets.numpy(), 1.0 / 7, 1e-3)[0])
    err = (logits.cpu().double() - ref).abs() / storage_ulp(ref, torch.bfloat16).double()
    err[torch.arange(rows), targets] = 0
    _say(f"rows of {vocab}, aligned {aligned}: {err.max().item():.4f} ulp")
    assert err.max() <= 0.5 + 2.0 ** -9


def test_chunk_size_bounds_the_memory():
    """Forward and backward of 8192 tokens in chunks of 256: the d logits in memory are those of 256 tokens,
    beside the results, the bf16 weight and the fp32 partials of the products."""
    tokens, width, vocab = 8192, 256, 32000
    hidden = torch.randn(tokens, width, device="cuda").requires_grad_()
    weight = (0.05 * torch.randn(vocab, width, device="cuda")).requires_grad_()
    targets = torch.randint(0, vocab, (tokens,), device="cuda")

    def peak(**kw):
        torch.cuda.synchronize()
        torch.cuda.reset_peak_memory_stats()
        before = torch.cuda.memory_allocated()
        loss = fused_linear_cross_entropy(hidden, weight, targets, float(tokens), **kw)[0]
        torch.autograd.grad(loss, (hidden, weight))
        return torch.cuda.max_memory_allocated() - before

    small, default = peak(chunk_size=256), peak()
    _say(f"peak {small >> 20} MiB in chunks of 256, {default >> 20} MiB by default")
    results = 2 * tokens * width * 4 + vocab * width * (2 + 4 + 4)
    assert small <= results + 256 * vocab * 2 * 2 + (32 << 20)
    assert default >= tokens * vocab * 2


def test_compiled_calls_break_the_graph():
    """Under torch.compile the call runs as it is, its default and a named chunk_size alike."""
    hidden = torch.randn(64, 64, dtype=torch.bfloat16, device="cuda").requires_grad_()
    weight = torch.randn(300, 64, dtype=torch.bfloat16, device="cuda").requires_grad_()
    targets = torch.randint(0, 300, (64,), device="cuda")
    for kw in ({}, {"chunk_size": 32}):
        def step():
            return fused_linear_cross_entropy(hidden * 2, weight, targets, 64.0, **kw)[0]
        assert torch.equal(torch.compile(step, backend="eager")(), step())


def _twice_as_far(x):
    y = x.new_empty(*x.shape[:-1], 2 * x.shape[-1])[..., ::2]
    return y.copy_(x)


@pytest.mark.parametrize("unpack", [lambda x: x.t().contiguous().t(), _twice_as_far, lambda x: _flat_view(x, 1),
                                    lambda x: x.double(), lambda x: x.cpu().cuda()])
def test_saved_gradients_may_come_back_in_another_layout(unpack):
    """A hook on saved tensors may hand the stored gradients back strided, unaligned or in another type."""
    g = torch.Generator().manual_seed(3)
    hidden = torch.randn(30, 64, generator=g).to(torch.bfloat16).cuda().requires_grad_()
    weight = (0.1 * torch.randn(300, 64, generator=g)).cuda().requires_grad_()
    targets = torch.randint(0, 300, (30,), generator=g).cuda()
    exp = torch.autograd.grad(3.0 * fused_linear_cross_entropy(hidden, weight, targets, 30.0)[0], (hidden, weight))
    with torch.autograd.graph.saved_tensors_hooks(lambda x: x, unpack):
        loss = 3.0 * fused_linear_cross_entropy(hidden, weight, targets, 30.0)[0]
    got = torch.autograd.grad(loss, (hidden, weight))
    for a, b in zip(got, exp):
        assert a.dtype == b.dtype
        # one rounding of a bf16 product (none of a float64 one)
        torch.testing.assert_close(a.float(), b.float(), rtol=2.0 ** -8, atol=0)


def test_upstream_gradients_of_other_kinds():
    """A mapped upstream gradient maps the gradients, a dual one gives them its tangent."""
    hidden = torch.randn(30, 64, device="cuda").to(torch.bfloat16).requires_grad_()
    weight = (0.1 * torch.randn(300, 64, device="cuda")).requires_grad_()
    loss = fused_linear_cross_entropy(hidden, weight, torch.randint(0, 300, (30,), device="cuda"), 30.0)[0]
    (exp,) = torch.autograd.grad(loss, weight, torch.tensor(1.0, device="cuda"), retain_graph=True)
    factors = torch.tensor([1.0, 2.0, -0.5], device="cuda")
    (mapped,) = torch.autograd.grad(loss, weight, factors, retain_graph=True, is_grads_batched=True)
    assert torch.equal(mapped, factors[:, None, None] * exp)
    with torch.autograd.forward_ad.dual_level():
        up = torch.autograd.forward_ad.make_dual(torch.tensor(1.0, device="cuda"), torch.tensor(4.0, device="cuda"))
        (dual,) = torch.autograd.grad(loss, weight, up)
        primal, tangent = torch.autograd.forward_ad.unpack_dual(dual)
        assert torch.equal(primal, exp) and tangent is not None and torch.equal(tangent, 4.0 * exp)


def test_an_ignored_token_with_infinities_has_no_gradient():
    """With a vocabulary that 8 does not divide, rows of the d logits have pads, which are read back."""
    hidden = torch.randn(40, 64, device="cuda").to(torch.bfloat16)
    hidden[7, 5] = float("inf")
    hidden.requires_grad_()
    weight = torch.randn(1003, 64, device="cuda").to(torch.bfloat16).requires_grad_()
    targets = torch.randint(0, 1003, (40,), device="cuda")
    targets[7] = -100
    loss = fused_linear_cross_entropy(hidden, weight, targets, 39.0)[0]
    (grad,) = torch.autograd.grad(loss, hidden)
    assert torch.isfinite(loss) and torch.isfinite(grad).all() and (grad[7] == 0).all()
