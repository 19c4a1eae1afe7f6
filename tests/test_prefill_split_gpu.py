"""The forward with split keys (few query blocks, long caches) against the oracle: sequences of
no key, of one part and of many, partial tiles, windows, every head_dim, a negative scale, and
the smallest and largest query counts that take it."""

import pytest
import torch

from _util import assert_close, assert_lse
from myk_llm_amd import flash_attn_func, flash_attn_with_kvcache
from oracle.attention import kvcache_reference, reference_with_lse

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nq, heads, kv_heads, d, lens, window, scale, dtype", [
    (17, 16, 4, 128, [0, 1, 1400], (-1, -1), None, torch.bfloat16),
    (33, 8, 2, 64, [255, 256, 257, 2015], (-1, -1), None, torch.float16),
    (130, 4, 4, 64, [2040, 63], (-1, -1), None, torch.bfloat16),
    (64, 6, 2, 128, [1900], (1500, 0), None, torch.bfloat16),
    (40, 3, 1, 32, [2000, 0], (-1, -1), -0.2, torch.bfloat16),
    (100, 5, 5, 16, [1500], (-1, 7), None, torch.float16),
    (31, 8, 1, 256, [1000, 30], (-1, -1), None, torch.bfloat16),
])
def test_split_keys_match_oracle(nq, heads, kv_heads, d, lens, window, scale, dtype):
    print(f"split keys nq={nq} H={heads}/{kv_heads} D={d} lens={lens}", flush=True)
    g = torch.Generator().manual_seed(nq)
    b, cap = len(lens), 2200
    mk = lambda *s: torch.randn(*s, generator=g).to(dtype)  # noqa: E731
    q, kc, vc, kn, vn = mk(b, nq, heads, d), mk(b, cap, kv_heads, d), mk(b, cap, kv_heads, d), mk(b, nq, kv_heads, d), mk(b, nq, kv_heads, d)
    cl = torch.tensor(lens, dtype=torch.int32)
    causal = window[1] <= 0
    exp, exp_lse, _, _ = kvcache_reference(q.float(), kc.float(), vc.float(), kn.float(), vn.float(), cl, causal,
                                           window, scale)
    out, lse = flash_attn_with_kvcache(q.cuda(), kc.cuda(), vc.cuda(), kn.cuda(), vn.cuda(), cache_seqlens=cl.cuda(),
                                       causal=causal, window_size=window, softmax_scale=scale, return_softmax_lse=True)
    assert_close(out, exp)
    assert_lse(lse, exp_lse)


@pytest.mark.parametrize("sq, sk, heads", [(1792, 1792, 16), (1793, 1793, 16), (1024, 1024, 16), (700, 1111, 8)])
def test_dense_batches_around_the_rule(sq, sk, heads):
    """One causal sequence on both sides of the most rows that are split, and Lq != Lk."""
    g = torch.Generator().manual_seed(sq)
    mk = lambda *s: torch.randn(*s, generator=g).to(torch.bfloat16)  # noqa: E731
    q, k, v = mk(1, sq, heads, 64), mk(1, sk, heads // 4, 64), mk(1, sk, heads // 4, 64)
    out, lse = flash_attn_func(q.cuda(), k.cuda(), v.cuda(), causal=True, return_softmax_lse=True)
    exp, exp_lse = reference_with_lse(q, k, v, True, (-1, -1))
    assert_close(out, exp)
    assert_lse(lse, exp_lse)


@pytest.mark.parametrize("nq, heads, kv_heads, d, lens, cap, dtype", [
    (389, 16, 4, 128, [0], 8192, torch.bfloat16),     # eight slots a block, one or two parts
    (100, 8, 2, 64, [0, 300, 2, 900], 8192, torch.bfloat16),
    (40, 4, 4, 32, [8160], 8192, torch.float16),      # keys past the capacity are dropped
    (500, 2, 1, 256, [17], 4096, torch.bfloat16),
])
def test_short_prompts_into_large_caches(nq, heads, kv_heads, d, lens, cap, dtype):
    print(f"short prompt nq={nq} H={heads}/{kv_heads} D={d} lens={lens} cap={cap}", flush=True)
    g = torch.Generator().manual_seed(nq)
    b = len(lens)
    mk = lambda *s: torch.randn(*s, generator=g).to(dtype)  # noqa: E731
    q, kc, vc, kn, vn = mk(b, nq, heads, d), mk(b, cap, kv_heads, d), mk(b, cap, kv_heads, d), mk(b, nq, kv_heads, d), mk(b, nq, kv_heads, d)
    cl = torch.tensor(lens, dtype=torch.int32)
    exp, exp_lse, exp_k, exp_v = kvcache_reference(q.float(), kc.float(), vc.float(), kn.float(), vn.float(), cl, True, (-1, -1))
    for index in (torch.int32, torch.int64):  # (int64 lengths: the Python path)
        kd, vd, seq = kc.cuda(), vc.cuda(), cl.to(index).cuda()
        out, lse = flash_attn_with_kvcache(q.cuda(), kd, vd, kn.cuda(), vn.cuda(), cache_seqlens=seq, causal=True,
                                           return_softmax_lse=True)
        assert_close(out, exp)
        assert_lse(lse, exp_lse)
        assert torch.equal(kd.cpu().float(), exp_k.float()) and torch.equal(vd.cpu().float(), exp_v.float())
        assert torch.equal(seq.cpu(), cl.to(index))


@pytest.mark.parametrize("index", [torch.int32, torch.int64])  # the native path, the Python one
def test_no_memory_for_the_parts(index):
    """Where the device has no room for the partials the keys stay whole."""
    g = torch.Generator(device="cuda").manual_seed(0)
    mk = lambda *s: torch.randn(*s, generator=g, device="cuda").to(torch.bfloat16)  # noqa: E731
    q, kc, vc, kn, vn = mk(1, 389, 16, 128), mk(1, 8192, 4, 128), mk(1, 8192, 4, 128), mk(1, 389, 4, 128), mk(1, 389, 4, 128)
    lens = torch.tensor([6000], dtype=index, device="cuda")
    call = lambda: flash_attn_with_kvcache(q, kc, vc, kn, vn, cache_seqlens=lens, causal=True)  # noqa: E731
    exp = call()
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    total = torch.cuda.get_device_properties(0).total_memory
    filler = []
    torch.cuda.set_per_process_memory_fraction((torch.cuda.memory_reserved() + (24 << 20)) / total)
    try:
        room = torch.empty(4 << 20, dtype=torch.uint8, device="cuda")  # for O and the LSE
        try:
            while True:  # no 10 MB in one piece are left, and so no 26, the partials, with the room's 4
                filler.append(torch.empty(10 << 20, dtype=torch.uint8, device="cuda"))
        except torch.OutOfMemoryError:
            del room
        before = torch.cuda.memory_stats()["num_ooms"]
        got = call()
    finally:
        torch.cuda.set_per_process_memory_fraction(1.0)
    assert torch.cuda.memory_stats()["num_ooms"] > before
    assert_close(got, exp)
    del got, filler
    assert torch.equal(call(), exp)
