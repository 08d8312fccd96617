"""Prefill launches that split a kv head's query heads into sets with row tiles of their own: a row's arithmetic does not
depend on the rows beside it, so a grouped call equals, bit for bit, the call over a cache with every kv head repeated for
each of its query heads (groups of one head, nothing packed), and is close to float64."""
import numpy as np
import pytest
import torch

import gi_attn
from attn_common import assert_close, reference_f64

pytestmark = pytest.mark.gpu

# (n, pos0, n_heads, n_kv): groups of 2, 3, 4, 6 and 8, split or whole, rows that end inside a wave and inside a tile
SHAPES = [(16, 0, 12, 2), (17, 100, 12, 2), (33, 0, 16, 2), (57, 300, 8, 4), (64, 0, 9, 3), (100, 700, 12, 2), (129, 0, 32, 8), (500, 0, 6, 1)]


@pytest.mark.parametrize("n,pos0,n_heads,n_kv", SHAPES)
@pytest.mark.parametrize("fmt,hd", [("f16", 64), ("f16", 128), ("f16", 256), ("i8", 64), ("i8", 128), ("i8", 256), ("q4", 256), ("f32", 96), ("f32", 128)])
def test_sets_equal_the_call_with_repeated_heads(gpu, n, pos0, n_heads, n_kv, fmt, hd):
    print("[case] sets", n, pos0, n_heads, n_kv, fmt, hd, flush=True)
    G, ctx = n_heads // n_kv, pos0 + n
    gen = torch.Generator(device=gpu).manual_seed(9800 + n + hd)
    q = torch.randn((n, n_heads * hd), device=gpu, generator=gen)
    empty = torch.empty(0, dtype=torch.uint8, device=gpu)  # (no cut in f32 either)
    rep = lambda *ts: [t.repeat_interleave(G, 1).contiguous() for t in ts]
    if fmt == "q4":
        kc, vc = (torch.randint(0, 256, (ctx, n_kv, 128), device=gpu, dtype=torch.uint8, generator=gen) for _ in range(2))
        ks, vs = ((0.2 + 0.15 * torch.rand((ctx, n_kv, 8), device=gpu, generator=gen)).half() for _ in range(2))
        for staged in (True, False):
            got = gi_attn.prefill_q4(q, kc, vc, ks, vs, pos0, n_heads, n_kv, staged=staged)
            want = gi_attn.prefill_q4(q, *rep(kc, vc, ks, vs), pos0, n_heads, n_heads, staged=staged)
            assert torch.equal(got, want), staged
        return
    if fmt == "i8":
        kc, vc = (torch.randint(-127, 128, (ctx, n_kv, hd), device=gpu, dtype=torch.int8, generator=gen) for _ in range(2))
        ks, vs = (0.01 + 0.01 * torch.rand((ctx, n_kv), device=gpu, generator=gen) for _ in range(2))
        for staged in (True, False):
            got = gi_attn.prefill(q, kc, vc, pos0, n_heads, n_kv, hd=hd, k_scale=ks, v_scale=vs, staged=staged)
            kr, vr, ksr, vsr = rep(kc, vc, ks, vs)
            want = gi_attn.prefill(q, kr, vr, pos0, n_heads, n_heads, hd=hd, k_scale=ksr, v_scale=vsr, staged=staged)
            assert torch.equal(got, want), staged
        return
    kc, vc = (torch.randn((ctx, n_kv, hd), device=gpu, generator=gen).half() for _ in range(2))
    got = gi_attn.prefill(q, kc, vc, pos0, n_heads, n_kv, hd=hd, f32=fmt == "f32", workspace=empty)
    want = gi_attn.prefill(q, *rep(kc, vc), pos0, n_heads, n_heads, hd=hd, f32=fmt == "f32", workspace=empty)
    assert torch.equal(got, want)
    k, v = (t.view(torch.int16).cpu().numpy().view(np.uint16).reshape(ctx, -1) for t in (kc, vc))
    r = n - 1
    tol = dict(max_abs=2e-5, rel_l2=2e-5) if fmt == "f32" else {}
    assert_close(got[r:].cpu().numpy(), reference_f64(q[r:].cpu().numpy(), k, v, pos0 + r, n_heads, n_kv, hd=hd), what="last row", **tol)


def test_packed_rows_past_the_product_form(gpu):
    # 2048 tokens of 1024 heads on one kv head: n * G * G reaches 2^31, where a packed row's token takes a division
    n, heads, hd = 2048, 1024, 64
    print("[case] packed rows, division", n, heads, flush=True)
    gen = torch.Generator(device=gpu).manual_seed(9890)
    q = torch.randn((n, heads * hd), device=gpu, generator=gen).half()
    kc, vc = (torch.randn((n, 1, hd), device=gpu, generator=gen).half() for _ in range(2))
    got = gi_attn.prefill(q, kc, vc, 0, heads, 1, hd=hd)
    want = gi_attn.prefill(q, *(t.repeat_interleave(heads, 1).contiguous() for t in (kc, vc)), 0, heads, heads, hd=hd)
    torch.cuda.synchronize()
    assert torch.equal(got, want) and torch.isfinite(got).all()
