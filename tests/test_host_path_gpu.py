"""The native host path against the Python one it stands in for: the same bits for every form that
it accepts, and the same answer from autograd where it is looked at from outside (hooks on saved
tensors, a second backward, gradients of gradients, mapped and forward-mode gradients)."""

import ctypes

import pytest
import torch

from myk_llm_amd import flash_attn as fa
from myk_llm_amd import flash_attn_func, flash_attn_varlen_func, flash_attn_with_kvcache

pytestmark = pytest.mark.gpu


class _Recorded:
    """The extension, noting for each call whether it took it."""

    def __init__(self):
        self.mod, self.took = fa._native(), []

    def _note(self, r):
        self.took.append(r is not NotImplemented)
        return r

    def attention(self, *a):
        return self._note(self.mod.attention(*a))

    def kvcache(self, *a):
        return self._note(self.mod.kvcache(*a))


def _both(monkeypatch, call, native=None):
    """The call's results as it is, and with the Python path alone. native: whether the first is one that the
    extension takes."""
    with monkeypatch.context() as m:
        recorded = _Recorded()
        m.setattr(fa, "_host", recorded)
        got = call()
        assert native is None or (recorded.took and all(t == native for t in recorded.took)), recorded.took
    with monkeypatch.context() as m:
        m.setattr(fa, "_host", fa._NoHost)
        return got, call()


def _same(got, exp):
    assert len(got) == len(exp)
    for a, b in zip(got, exp):
        assert (a is None) == (b is None) and (a is None or (a.shape == b.shape and a.dtype == b.dtype and torch.equal(a, b)))
        assert a is None or (a.requires_grad == b.requires_grad and a.stride() == b.stride())


def _qkv(g, lead, hq, hk, d, dtype, form):
    def make(h):
        if form == "sliced":  # one of a wider projection's parts
            x = torch.randn(*lead, h + 2, d, generator=g)[..., 1:1 + h, :]
            return x.to(dtype).cuda()
        if form == "heads_first":
            return torch.randn(*lead[:-1], h, lead[-1], d, generator=g).to(dtype).cuda().transpose(-3, -2)
        if form == "unaligned":  # not what the kernels read: copied by the Python path
            return torch.randn(*lead, h, d + 3, generator=g).to(dtype).cuda()[..., 3:]
        return torch.randn(*lead, h, d, generator=g).to(dtype).cuda()

    return make(hq), make(hk), make(hk)


@pytest.mark.parametrize("form", ["plain", "sliced", "heads_first", "unaligned"])
@pytest.mark.parametrize("packed", [False, True])
@pytest.mark.parametrize("d, dtype, needs", [(64, torch.bfloat16, "qkv"), (128, torch.float16, "qkv"), (32, torch.bfloat16, "k"),
                                             (64, torch.bfloat16, "")])
@pytest.mark.parametrize("with_lse", [False, True])
def test_attention_bits(monkeypatch, form, packed, d, dtype, needs, with_lse):
    g = torch.Generator().manual_seed(d)
    q, k, v = _qkv(g, (150,) if packed else (2, 75), 4, 2, d, dtype, form)
    for n, x in (("q", q), ("k", k), ("v", v)):
        x.requires_grad_(n in needs)
    cu = torch.tensor([0, 31, 150], dtype=torch.int32, device="cuda")
    dout = torch.randn(4, q.shape[-3] if packed else 75, d, generator=g).to(dtype).cuda().transpose(0, 1)
    dout = dout if packed else dout.expand(2, 75, 4, d)

    def call():
        kw = dict(causal=True, window_size=(40, 0), softmax_scale=0.2, return_softmax_lse=with_lse)
        r = flash_attn_varlen_func(q, k, v, cu, cu, 119, 119, **kw) if packed else flash_attn_func(q, k, v, **kw)
        out = r[0] if with_lse else r
        ins = [x for x in (q, k, v) if x.requires_grad]
        return (*(r if with_lse else (r,)), *(torch.autograd.grad(out, ins, dout) if ins else ()))

    _same(*_both(monkeypatch, call, native=form != "unaligned"))


@pytest.mark.parametrize("nq, lens, with_lse", [(1, [0, 200], False), (16, [3, 77], True), (17, [0, 200], True), (40, [250, 1], False)])
@pytest.mark.parametrize("index", [torch.int32, torch.int64])
def test_kvcache_bits(monkeypatch, nq, lens, with_lse, index):
    g = torch.Generator().manual_seed(nq)
    q, k, v = _qkv(g, (2, nq), 8, 2, 64, torch.bfloat16, "plain")
    caches = torch.randn(2, 2, 256, 2, 64, generator=g).to(torch.bfloat16).cuda()
    cl = torch.tensor(lens, dtype=index, device="cuda")

    def call():
        kc, vc = caches[0].clone(), caches[1].clone()
        r = flash_attn_with_kvcache(q, kc, vc, k, v, cache_seqlens=cl, causal=True, return_softmax_lse=with_lse)
        return (*(r if with_lse else (r,)), kc, vc)

    _same(*_both(monkeypatch, call, native=index == torch.int32))


def _error(call):
    try:
        call()
    except Exception as e:  # noqa: BLE001
        return type(e)
    return None


def test_refusals_and_autograd_from_outside(monkeypatch):
    g = torch.Generator().manual_seed(1)
    q, k, v = (x.requires_grad_() for x in _qkv(g, (2, 40), 4, 2, 64, torch.bfloat16, "plain"))
    grad = torch.randn(2, 40, 4, 64, generator=g).to(torch.bfloat16).cuda()

    def second_backward():
        out = flash_attn_func(q, k, v)
        out.backward(grad)
        out.backward(grad)

    def changed_in_place():
        x = q.clone()
        out = flash_attn_func(x, k, v)
        x.mul_(2)
        out.backward(grad)

    def mapped():
        out = flash_attn_func(q, k, v)
        torch.autograd.grad(out, q, torch.stack([grad, grad]), is_grads_batched=True)

    def functional():
        torch.func.grad(lambda x: flash_attn_func(x, k, v).float().sum())(q.detach())

    def forward_mode():
        with torch.autograd.forward_ad.dual_level():
            flash_attn_func(torch.autograd.forward_ad.make_dual(q.detach(), grad), k, v)

    def wrong_heads():
        flash_attn_func(q[:, :, :3], k, v)

    def wrong_dtype():
        flash_attn_func(q, k.half(), v)

    def host_keys():
        flash_attn_func(q, k.cpu(), v)

    for call in (second_backward, changed_in_place, mapped, functional, forward_mode, wrong_heads, wrong_dtype, host_keys):
        got, exp = _both(monkeypatch, lambda call=call: _error(call))
        assert got is exp and got is not None, (call.__name__, got, exp)

    def hooked():
        seen = []
        with torch.autograd.graph.saved_tensors_hooks(lambda x: (seen.append(tuple(x.shape)), x * 1)[1], lambda x: x):
            out = flash_attn_func(q, k, v, causal=True)
        return (torch.tensor(len(seen)), *torch.autograd.grad(out, (q, k, v), grad))

    def twice():
        out = flash_attn_func(q, k, v)
        return torch.autograd.grad(out, (q, k, v), grad, create_graph=True)

    def unused():
        out, lse = flash_attn_func(q, k, v, return_softmax_lse=True)
        return (*torch.autograd.grad(out.float().sum(), (q,), retain_graph=True), torch.tensor(out.requires_grad),
                torch.tensor(lse.requires_grad))

    for call in (hooked, twice, unused):
        _same(*_both(monkeypatch, call, native=True))


@pytest.mark.parametrize("packed", [False, True])
def test_stored_ds_backward_holds_its_gradients_once(monkeypatch, packed):
    """Where the backward is planned in Python the native one keeps nothing beside it: the same peak."""
    g = torch.Generator().manual_seed(0)
    n = 2048
    q, k, v = (x.requires_grad_() for x in _qkv(g, (n,) if packed else (1, n), 16, 4, 128, torch.bfloat16, "plain"))
    dout = torch.randn(q.shape, generator=g).to(torch.bfloat16).cuda()
    cu = torch.tensor([0, 500, n], dtype=torch.int32, device="cuda")

    def call():
        out = flash_attn_varlen_func(q, k, v, cu, cu, n, n, causal=True) if packed else flash_attn_func(q, k, v, causal=True)
        torch.cuda.synchronize()
        torch.cuda.reset_peak_memory_stats()
        before = torch.cuda.memory_allocated()
        grads = torch.autograd.grad(out, (q, k, v), dout)
        torch.cuda.synchronize()
        return torch.cuda.max_memory_allocated() - before, grads

    (got, a), (exp, b) = _both(monkeypatch, call, native=True)
    _same(a, b)
    assert got <= exp, (got, exp)


def test_launches_run_without_the_interpreter_lock(monkeypatch):
    """The entry that the native path asks for the number of decode splits is replaced by the interpreter's own
    question whether this thread holds its lock; what it answers arrives at the next entry."""
    g = torch.Generator().manual_seed(0)
    q, k, v = _qkv(g, (2, 3), 4, 2, 64, torch.bfloat16, "plain")
    caches = torch.zeros(2, 2, 64, 2, 64, dtype=torch.bfloat16, device="cuda")
    lens = torch.zeros(2, dtype=torch.int32, device="cuda")
    held = []

    def size(*args):
        held.append(args[-1])
        return 16

    entries = {"decode_num_splits": ctypes.pythonapi.PyGILState_Check,
               "decode_workspace_size": ctypes.CFUNCTYPE(ctypes.c_size_t, *[ctypes.c_int32] * 5)(size),
               "decode": ctypes.CFUNCTYPE(ctypes.c_int, *[ctypes.c_void_p] * 2, ctypes.c_size_t, ctypes.c_void_p)(lambda *a: 0)}
    lib = fa._lib.lib()
    monkeypatch.setattr(fa, "_host", None)
    mod = fa._native()
    try:
        mod.setup(*(ctypes.cast(entries.get(n) or getattr(lib, f"mykfa_{n}"), ctypes.c_void_p).value for n in fa._HOST_ENTRIES),
                  fa._lib.check, fa._backward_launch)
        flash_attn_with_kvcache(q, *caches, k, v, cache_seqlens=lens)
        flash_attn_func(q, k, v)
        flash_attn_func(q.requires_grad_(), k, v)
    finally:
        fa._host = None
        fa._native()
    assert held == [0, 0, 0]


def test_errors_of_the_library_and_of_hooks_reach_the_caller(monkeypatch):
    g = torch.Generator().manual_seed(0)
    q, k, v = (x.requires_grad_() for x in _qkv(g, (1, 40), 4, 2, 64, torch.bfloat16, "plain"))

    def not_a_scale():
        flash_attn_func(q, k, v, softmax_scale=float("nan"))

    def not_a_scale_without_gradients():
        with torch.no_grad():
            not_a_scale()

    def hook():
        def pack(x):
            raise LookupError("no room")
        with torch.autograd.graph.saved_tensors_hooks(pack, lambda x: x):
            flash_attn_func(q, k, v)

    for call, kind in ((not_a_scale, fa._lib.MykfaError), (not_a_scale_without_gradients, fa._lib.MykfaError), (hook, LookupError)):
        got, exp = _both(monkeypatch, lambda call=call: _error(call))
        assert got is exp is kind
    assert torch.isfinite(flash_attn_func(q, k, v)).all()
