"""The two launch forms of the cache write (one head per wave for a few tokens, four for many) and its two rotations (the
lane swap for whole heads rotated in halves, the LDS row otherwise): a batch in the second form against its tokens one by
one in the first, which must agree bit for bit, and the rotation against float64."""
import numpy as np
import pytest
import torch

import gi_attn

pytestmark = pytest.mark.gpu


def caches(fmt, cap, n_kv, hd, dev):
    if fmt == "f16":
        return [torch.zeros((cap, n_kv, hd), dtype=torch.float16, device=dev) for _ in "kv"] + [None, None]
    if fmt == "i8":
        return [torch.zeros((cap, n_kv, hd), dtype=torch.int8, device=dev) for _ in "kv"] + \
               [torch.zeros((cap, n_kv), device=dev) for _ in "kv"]
    return [torch.zeros((cap, n_kv, 128), dtype=torch.uint8, device=dev) for _ in "kv"] + \
           [torch.zeros((cap, n_kv, 8), dtype=torch.float16, device=dev) for _ in "kv"]


def write(fmt, qkv, c, pos, heads, n_kv, hd, **kw):
    if fmt == "q4":
        gi_attn.qk_norm_rope_q4(qkv, *c, pos, heads, n_kv, **kw)
    else:
        gi_attn.qk_norm_rope(qkv, c[0], c[1], pos, heads, n_kv, hd=hd, k_scale=c[2], v_scale=c[3], **kw)


@pytest.mark.parametrize("fmt,hd,heads,n_kv,rope_dim,neox,norm", [
    ("f16", 64, 9, 3, 64, True, True), ("f16", 128, 8, 2, 128, True, False), ("i8", 128, 32, 8, 128, True, True),
    ("i8", 128, 8, 2, 64, True, True), ("f16", 128, 8, 2, 128, False, True), ("f16", 96, 4, 4, 96, True, True),
    ("i8", 256, 16, 2, 256, True, True), ("q4", 256, 16, 2, 256, True, True), ("q4", 256, 4, 1, 64, True, True),
])
def test_batch_equals_tokens_and_float64(gpu, fmt, hd, heads, n_kv, rope_dim, neox, norm):
    print("[case] rope forms", fmt, hd, heads, n_kv, rope_dim, neox, norm, flush=True)
    n, pos0, base = 300, 1234, 1e6
    gen = torch.Generator(device=gpu)
    gen.manual_seed(hd + rope_dim)
    x = torch.randn((n, (heads + 2 * n_kv) * hd), generator=gen, device=gpu)
    kw = dict(rope_dim=rope_dim, neox=neox, base=base)
    if norm:
        kw.update(qn=torch.rand(hd, generator=gen, device=gpu) + 0.5, kn=torch.rand(hd, generator=gen, device=gpu) + 0.5)
    a, b = x.clone(), x.clone()
    ca, cb = (caches(fmt, pos0 + n, n_kv, hd, gpu) for _ in range(2))
    write(fmt, a, ca, pos0, heads, n_kv, hd, **kw)
    toks = [0, 1, 151, 299]
    for t in toks:
        write(fmt, b[t:t + 1], cb, pos0 + t, heads, n_kv, hd, **kw)
    torch.cuda.synchronize()
    for t in toks:
        assert torch.equal(a[t], b[t]), t
        for u, v in zip(ca, cb):
            assert u is None or torch.equal(u[pos0 + t], v[pos0 + t]), t
    if fmt == "q4":
        return  # (rotated rows: the transform's own tests)
    y = x.cpu().numpy().astype(np.float64).reshape(n, -1, hd)[:, :heads + n_kv]
    if norm:
        y /= np.sqrt((y ** 2).mean(-1, keepdims=True) + 1e-6)
        y[:, :heads] *= kw["qn"].cpu().numpy()
        y[:, heads:] *= kw["kn"].cpu().numpy()
    i = np.arange(rope_dim // 2)
    ang = np.arange(pos0, pos0 + n)[:, None] * base ** (-2.0 * i / rope_dim)
    c, s = np.cos(ang)[:, None], np.sin(ang)[:, None]
    lo, hi = (i, i + rope_dim // 2) if neox else (2 * i, 2 * i + 1)
    z = y.copy()
    z[..., lo], z[..., hi] = y[..., lo] * c - y[..., hi] * s, y[..., lo] * s + y[..., hi] * c
    got = a.cpu().numpy().reshape(n, -1, hd)[:, :heads + n_kv]
    # the f32 angle of a position below 1534 is off by up to 1534 * 2^-23 * 1.5 = 2.7e-4 of a radian at |y| <= 8
    assert np.abs(got - z).max() <= 2.2e-3


@pytest.mark.parametrize("hd,rope_dim,neox", [(64, 64, True), (128, 128, True), (128, 128, False), (128, 64, True),
                                              (256, 256, True), (96, 96, True)])
def test_rotated_pair_rounds_one_product(gpu, hd, rope_dim, neox):
    """Every way of pairing gives a = round(p c - round(q s)) and b = round(q c + round(p s)), to the bit (a 64-bit mantissa
    holds the unrounded sums to well below f32's half step). Head 0's pairs are (1, 0) and come out as the pair's (c, s)."""
    print("[case] rope pair", hd, rope_dim, neox, flush=True)
    n, heads, n_kv, pos0 = 70, 8, 1, 4321
    gen = torch.Generator(device=gpu)
    gen.manual_seed(hd)
    x = torch.randn((n, (heads + 2 * n_kv) * hd), generator=gen, device=gpu)
    half = rope_dim // 2
    i = np.arange(half)
    ia, ib = (i, i + half) if neox else (2 * i, 2 * i + 1)
    x[:, :hd] = 0
    x[:, torch.as_tensor(ia, device=gpu)] = 1
    y = x.clone()
    c = caches("f16", pos0 + n, n_kv, hd, gpu)
    write("f16", y, c, pos0, heads, n_kv, hd, rope_dim=rope_dim, neox=neox, base=1e6)
    xs = x.cpu().numpy().reshape(n, -1, hd)[:, 1:heads + n_kv]
    ys = y.cpu().numpy().reshape(n, -1, hd)
    co, si = ys[:, :1, ia], ys[:, :1, ib]
    ld = np.longdouble
    p, q = xs[..., ia], xs[..., ib]
    a = (ld(p) * ld(co) - ld(q * si)).astype(np.float32)
    b = (ld(q) * ld(co) + ld(p * si)).astype(np.float32)
    got = ys[:, 1:heads + n_kv]
    assert np.array_equal(got[..., ia], a)
    assert np.array_equal(got[..., ib], b)
