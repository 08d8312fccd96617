"""The prefill entry points of one cache each (gi_attn_prefill, _i8, _q4, _f32, and _i8_ws / _q4_ws), called directly: bit
for bit what gi_attn_prefill_ws gives without a workspace, cut in a workspace with room, and close to float64. NaN and
infinities pass the merge of a cut launch as they pass an uncut one."""
import numpy as np
import pytest
import torch

import gi_attn
from attn_common import (assert_close, make_inputs, make_inputs_i8, make_inputs_q4, reference_f64, reference_f64_i8,
                         reference_f64_q4)

pytestmark = pytest.mark.gpu


def dev(x, gpu, *shape):
    x = np.ascontiguousarray(x)
    if x.dtype == np.uint16:
        return torch.from_numpy(x.view(np.int16)).to(gpu).view(torch.float16).view(*shape)
    return torch.from_numpy(x).to(gpu).view(*shape)


def ptrs(*ts):
    return [None if t is None else t.data_ptr() for t in ts]


# (n, pos0, n_heads, n_kv, hd): one tile and many, short and long enough to be cut with room
@pytest.mark.parametrize("n,pos0,n_heads,n_kv", [(16, 0, 8, 2), (130, 40, 6, 2), (40, 1500, 8, 2)])
@pytest.mark.parametrize("fmt,hd", [("f16", 64), ("f16", 128), ("f16", 256), ("i8", 64), ("i8", 128), ("i8", 256), ("q4", 256), ("f32", 80),
                                    ("f32", 128), ("f32i8", 64), ("f32i8", 112)])
def test_entry_points_called_directly(gpu, fmt, hd, n, pos0, n_heads, n_kv):
    print("[case] entry", fmt, hd, n, pos0, n_heads, n_kv, flush=True)
    lib, ctx, row = gi_attn.load_library(), pos0 + n, n_heads * hd
    seed = 9000 + n + hd
    if fmt == "q4":
        q, k, v, ks, vs = make_inputs_q4(seed, n, ctx, n_heads, n_kv)
        cache = [dev(x, gpu, ctx, n_kv, 128) for x in (k, v)] + [dev(x, gpu, ctx, n_kv, 8) for x in (ks, vs)]
        strides, want = (n_kv * 128, 128, n_kv * 8, 8), reference_f64_q4(q, k, v, ks, vs, pos0, n_heads, n_kv)
    elif fmt.endswith("i8"):
        q, k, v, ks, vs = make_inputs_i8(seed, n, ctx, n_heads, n_kv, hd=hd)
        cache = [dev(x, gpu, ctx, n_kv, hd) for x in (k, v)] + [dev(x, gpu, ctx, n_kv) for x in (ks, vs)]
        strides, want = (n_kv * hd, hd, n_kv, 1), reference_f64_i8(q, k, v, ks, vs, pos0, n_heads, n_kv, hd=hd)
    else:
        q, k, v = make_inputs(seed, n, ctx, n_heads, n_kv, hd=hd)
        cache = [dev(x, gpu, ctx, n_kv, hd) for x in (k, v)] + [None, None]
        strides, want = (n_kv * hd, hd, 0, 0), reference_f64(q, k, v, pos0, n_heads, n_kv, hd=hd)
    qt = torch.from_numpy(q).to(gpu)
    code = 2 if fmt == "q4" else 1 if fmt.endswith("i8") else 0
    f32 = fmt.startswith("f32")
    tail = (pos0, n, n_heads, n_kv)
    scale = float(hd) ** -0.5

    def run(call):
        out = torch.full((n, row), float("nan"), device=gpu)
        gi_attn._check(call((gi_attn._stream(), qt.data_ptr(), gi_attn.GI_F32, row), (out.data_ptr(), gi_attn.GI_F32, row, *tail)))
        torch.cuda.synchronize()
        return out

    def any_entry(ws=None, flags=0):
        size = 0 if ws is None else ws.numel()
        return run(lambda a, o: lib.gi_attn_prefill_ws(*a, *ptrs(*cache), code, flags | (2 if f32 else 0), *strides, *o, hd, scale,
                                                       None if ws is None else ws.data_ptr(), size))

    if f32:
        got = run(lambda a, o: lib.gi_attn_prefill_f32(*a, *ptrs(*cache), code, *strides, *o, hd, scale))
    elif fmt == "q4":
        got = run(lambda a, o: lib.gi_attn_prefill_q4(*a, *ptrs(*cache), *strides, *o, scale))
    elif fmt == "i8":
        got = run(lambda a, o: lib.gi_attn_prefill_i8(*a, *ptrs(*cache), *strides, *o, hd, scale))
    else:
        got = run(lambda a, o: lib.gi_attn_prefill(*a, *ptrs(*cache[:2]), *strides[:2], *o, hd, scale))
    tol = dict(max_abs=2e-5, rel_l2=2e-5) if f32 else {}
    assert_close(got.cpu().numpy(), want, what=fmt, **tol)
    assert torch.equal(any_entry(), got)
    part = lib.gi_attn_prefill_scratch_bytes(*tail, hd, code, 2 if f32 else 0)
    assert (part > 0) == (ctx >= 1024 or (f32 and ctx > 192))
    room = lib.gi_attn_prefill_workspace_bytes(ctx, n_kv, hd, code) if code and not f32 else 0
    ws = torch.empty(room + part, dtype=torch.uint8, device=gpu)
    if code and not f32:
        entry = lib.gi_attn_prefill_q4_ws if fmt == "q4" else lib.gi_attn_prefill_i8_ws
        extra = (scale,) if fmt == "q4" else (hd, scale)
        exact = run(lambda a, o: entry(*a, *ptrs(*cache), *strides, *o, *extra, ws.data_ptr(), room))
        assert torch.equal(exact, got)
        cut = run(lambda a, o: entry(*a, *ptrs(*cache), *strides, *o, *extra, ws.data_ptr(), room + part))
        assert torch.equal(cut, any_entry(ws, gi_attn.GI_PREFILL_WIDEN))
    else:
        cut = any_entry(ws)
    assert_close(cut.cpu().numpy(), want, what=fmt + " with room", **tol)
    if part > 0 and not f32:
        assert not torch.equal(cut, got)  # (another reference maximum per slice)


@pytest.mark.parametrize("hd", [64, 96, 128, 256])
def test_nan_and_infinities_through_the_merge(gpu, hd):
    # a NaN key that the last 20 tokens see (their rows NaN), infinite values in one dim each, one of them in the last slice
    # only and past most rows (its dim infinite for the last tokens): the cut launch as the uncut one
    n, pos0, n_heads, n_kv = 60, 1500, 4, 2
    print("[case] NaN and inf", hd, flush=True)
    ctx = pos0 + n
    gen = torch.Generator(device=gpu).manual_seed(9060 + hd)
    q = torch.randn((n, n_heads * hd), device=gpu, generator=gen)
    kc, vc = (torch.randn((ctx, n_kv, hd), device=gpu, generator=gen).half() for _ in range(2))
    vc[300, 0, 5] = float("inf")
    vc[ctx - 5, 0, 9] = float("-inf")
    kc[ctx - 20, 1] = float("nan")
    empty = torch.empty(0, dtype=torch.uint8, device=gpu)
    code = 2 if hd == 96 else 0
    assert gi_attn.load_library().gi_attn_prefill_scratch_bytes(pos0, n, n_heads, n_kv, hd, 0, code) > 0
    cut = gi_attn.prefill(q, kc, vc, pos0, n_heads, n_kv, hd=hd)
    whole = gi_attn.prefill(q, kc, vc, pos0, n_heads, n_kv, hd=hd, workspace=empty)
    torch.cuda.synchronize()
    heads = cut.view(n, n_heads, hd)
    assert torch.equal(cut.isnan(), whole.isnan()) and torch.equal(cut.isinf(), whole.isinf())
    assert torch.equal(cut[cut.isinf()], whole[whole.isinf()])
    assert heads[:, 0, 5].isinf().all() and heads[n - 20:, 2:].isnan().all() and not heads[:n - 20, 2:].isnan().any()
    fin = cut.isfinite()
    assert_close(cut[fin].cpu().numpy(), whole[fin].cpu().numpy(), what="finite outputs")


@pytest.mark.parametrize("hd", [64, 128, 256])
@pytest.mark.parametrize("stride", [1 << 23, 1 << 24])
def test_i8_scales_far_apart(gpu, hd, stride):
    # scales of one position 32 and 64 MiB from the next: a tile's 64 span 2 and 4 GiB, more than 32-bit offsets reach
    n, n_heads, n_kv = 70, 4, 2
    print("[case] far scales", hd, stride, flush=True)
    lib, row = gi_attn.load_library(), n_heads * hd
    q, k, v, ks, vs = make_inputs_i8(9100 + hd, n, n, n_heads, n_kv, hd=hd)
    qt, kt, vt = dev(q, gpu, n, row), dev(k, gpu, n, n_kv, hd), dev(v, gpu, n, n_kv, hd)
    near = [dev(x, gpu, n, n_kv) for x in (ks, vs)]
    far = [torch.empty((n - 1) * stride + n_kv, device=gpu) for _ in range(2)]
    for f, s in zip(far, near):
        f.as_strided((n, n_kv), (stride, 1)).copy_(s)

    def run(scales, sc_stride):
        out = torch.full((n, row), float("nan"), device=gpu)
        gi_attn._check(lib.gi_attn_prefill_i8(gi_attn._stream(), qt.data_ptr(), gi_attn.GI_F32, row, *ptrs(kt, vt, *scales), n_kv * hd, hd,
                                              sc_stride, 1, out.data_ptr(), gi_attn.GI_F32, row, 0, n, n_heads, n_kv, hd, hd ** -0.5))
        torch.cuda.synchronize()
        return out

    got = run(near, n_kv)
    assert_close(got.cpu().numpy(), reference_f64_i8(q, k, v, ks, vs, 0, n_heads, n_kv, hd=hd), what="near")
    assert torch.equal(run(far, stride), got)
