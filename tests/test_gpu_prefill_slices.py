"""Prefill launches cut along their keys (gi_attn_prefill_ws, the partials merged by gi_prefill_combine_*) and the packed
row tiles they share: short batches over long prefixes, against float64, and against the launch without a workspace, which
is never cut. Sizes at the edges: 16 and 17 key tiles, a last slice that only part of the rows sees, rows that end inside
a wave, inside a row tile and at its end, groups that do not divide a wave."""
import sys

import numpy as np
import pytest
import torch

import gi_attn
from attn_common import (assert_close, make_inputs, make_inputs_i8, make_inputs_q4, reference_f64, reference_f64_i8,
                         reference_f64_q4)

pytestmark = pytest.mark.gpu

SHAPES = [
    # (n, pos0, n_heads, n_kv, hd)
    (16, 16 * 64 - 16, 4, 4, 128),    # 16 tiles, one row per token and head
    (17, 16 * 64 - 16, 8, 1, 128),    # 17 tiles, the last one seen by the last token only
    (43, 2000, 6, 1, 128),            # G 6: 258 rows, two rows past a tile of 256
    (64, 4033, 8, 1, 128),
    (200, 3000, 32, 8, 128),
    (255, 1500, 9, 3, 64),
    (31, 9000, 9, 3, 64),
    (300, 5000, 16, 4, 128),          # over 4096 keys, 256 tokens or more
    (300, 5000, 8, 8, 64),
]


def dev(x, gpu, *shape):
    return torch.from_numpy(np.ascontiguousarray(x)).to(gpu).view(*shape)


def sliced(n, pos0, n_heads, n_kv, hd, fmt):
    return gi_attn.load_library().gi_attn_prefill_scratch_bytes(pos0, n, n_heads, n_kv, hd, fmt, 0) > 0


@pytest.mark.parametrize("n,pos0,n_heads,n_kv,hd", SHAPES)
@pytest.mark.parametrize("out_dtype", [torch.float32, torch.float16])
def test_sliced_prefill_f16(gpu, n, pos0, n_heads, n_kv, hd, out_dtype):
    print("[case] sliced prefill f16", n, pos0, n_heads, n_kv, hd, out_dtype, flush=True)
    assert sliced(n, pos0, n_heads, n_kv, hd, 0)
    q, k, v = make_inputs(9100 + n + hd, n, pos0 + n, n_heads, n_kv, hd=hd)
    qt = dev(q, gpu, n, n_heads * hd)
    kt, vt = (dev(x.view(np.int16), gpu, -1, n_kv, hd).view(torch.float16) for x in (k, v))
    got = gi_attn.prefill(qt, kt, vt, pos0, n_heads, n_kv, hd=hd, out_dtype=out_dtype)
    whole = torch.empty_like(got)
    code = gi_attn.GI_F16 if out_dtype == torch.float16 else gi_attn.GI_F32
    gi_attn._check(gi_attn.load_library().gi_attn_prefill(
        gi_attn._stream(), qt.data_ptr(), gi_attn.GI_F32, n_heads * hd, kt.data_ptr(), vt.data_ptr(), n_kv * hd, hd,
        whole.data_ptr(), code, n_heads * hd, pos0, n, n_heads, n_kv, hd, hd ** -0.5))
    torch.cuda.synchronize()
    # both round Q and P to f16 and differ in P's reference max per slice: within the bar of each from float64
    rows = sorted({0, 1, n // 2, n - 2, n - 1})
    for r in rows:
        want = reference_f64(q[r:r + 1], k, v, pos0 + r, n_heads, n_kv, hd=hd)
        assert_close(got[r:r + 1].float().cpu().numpy(), want, what=f"sliced row {r}")
    assert_close(got.float().cpu().numpy(), whole.float().cpu().numpy(), what="sliced against whole")


@pytest.mark.parametrize("n,pos0,n_heads,n_kv,hd", SHAPES)
def test_sliced_prefill_i8_same_for_both_stagings(gpu, n, pos0, n_heads, n_kv, hd):
    print("[case] sliced prefill i8", n, pos0, n_heads, n_kv, hd, flush=True)
    assert sliced(n, pos0, n_heads, n_kv, hd, 1)
    q, k, v, ks, vs = make_inputs_i8(9200 + n + hd, n, pos0 + n, n_heads, n_kv, hd=hd)
    qt = dev(q, gpu, n, n_heads * hd)
    kt, vt = (dev(x, gpu, -1, n_kv, hd) for x in (k, v))
    kst, vst = (dev(x, gpu, -1, n_kv) for x in (ks, vs))
    kw = dict(hd=hd, out_dtype=torch.float32, k_scale=kst, v_scale=vst)
    got = gi_attn.prefill(qt, kt, vt, pos0, n_heads, n_kv, staged=True, **kw)
    tile = gi_attn.prefill(qt, kt, vt, pos0, n_heads, n_kv, staged=False, **kw)
    torch.cuda.synchronize()
    assert torch.equal(got, tile)
    for r in sorted({0, 1, n // 2, n - 1}):
        want = reference_f64_i8(q[r:r + 1], k, v, ks, vs, pos0 + r, n_heads, n_kv, hd=hd)
        assert_close(got[r:r + 1].cpu().numpy(), want, what=f"sliced i8 row {r}")


def test_sliced_prefill_graph_replay(gpu):
    # the sliced launch and its merge captured together, replayed with new queries and eager work between the replays
    n, pos0, n_heads, n_kv = 40, 3000, 8, 2
    _, k, v = make_inputs(9300, 1, pos0 + n, n_heads, n_kv)
    kt, vt = (dev(x.view(np.int16), gpu, -1, n_kv, 128).view(torch.float16) for x in (k, v))
    q = torch.randn((n, n_heads * 128), device=gpu)
    out = torch.empty_like(q)
    gi_attn.prefill(q, kt, vt, pos0, n_heads, n_kv, out=out)
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        gi_attn.prefill(q, kt, vt, pos0, n_heads, n_kv, out=out)
    for r in range(3):
        q.copy_(torch.randn_like(q))
        want = gi_attn.prefill(q, kt, vt, pos0, n_heads, n_kv)
        torch.cuda.synchronize()
        out.zero_()
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want), f"replay {r}"


@pytest.mark.parametrize("n,pos0,n_heads,n_kv", [(16, 1008, 4, 4), (17, 1008, 16, 2), (50, 2500, 12, 2), (255, 1200, 8, 1),
                                                 (300, 4000, 16, 2)])
def test_sliced_prefill_h256_every_cache(gpu, n, pos0, n_heads, n_kv):
    # head size 256: f16, int8 and 4-bit, both stagings alike, rows at the edges of waves and of tiles of 64 and 128
    print("[case] sliced prefill h256", n, pos0, n_heads, n_kv, flush=True)
    hd = 256
    assert sliced(n, pos0, n_heads, n_kv, hd, 0)
    q, k, v = make_inputs(9400 + n, n, pos0 + n, n_heads, n_kv, hd=hd)
    qt = dev(q, gpu, n, n_heads * hd)
    kt, vt = (dev(x.view(np.int16), gpu, -1, n_kv, hd).view(torch.float16) for x in (k, v))
    got = gi_attn.prefill(qt, kt, vt, pos0, n_heads, n_kv, hd=hd)
    q8, k8, v8, ks, vs = make_inputs_i8(9500 + n, n, pos0 + n, n_heads, n_kv, hd=hd)
    q8t, kt, vt = dev(q8, gpu, n, n_heads * hd), dev(k8, gpu, -1, n_kv, hd), dev(v8, gpu, -1, n_kv, hd)
    kw = dict(hd=hd, k_scale=dev(ks, gpu, -1, n_kv), v_scale=dev(vs, gpu, -1, n_kv))
    got8, tile8 = (gi_attn.prefill(q8t, kt, vt, pos0, n_heads, n_kv, staged=s, **kw) for s in (True, False))
    q4, kc, vc, ks4, vs4 = make_inputs_q4(9600 + n, n, pos0 + n, n_heads, n_kv)
    t4 = [dev(q4, gpu, n, n_heads * hd), dev(kc, gpu, -1, n_kv, 128), dev(vc, gpu, -1, n_kv, 128)]
    t4 += [dev(np.ascontiguousarray(x).view(np.int16), gpu, -1, n_kv, 8).view(torch.float16) for x in (ks4, vs4)]
    got4, tile4 = (gi_attn.prefill_q4(*t4, pos0, n_heads, n_kv, staged=s) for s in (True, False))
    torch.cuda.synchronize()
    assert torch.equal(got8, tile8) and torch.equal(got4, tile4)
    for r in sorted({0, 1, n // 2, n - 1}):
        assert_close(got[r:r + 1].cpu().numpy(), reference_f64(q[r:r + 1], k, v, pos0 + r, n_heads, n_kv, hd=hd), what=f"row {r}")
        assert_close(got8[r:r + 1].cpu().numpy(), reference_f64_i8(q8[r:r + 1], k8, v8, ks, vs, pos0 + r, n_heads, n_kv, hd=hd),
                     what=f"i8 row {r}")
        assert_close(got4[r:r + 1].cpu().numpy(), reference_f64_q4(q4[r:r + 1], kc, vc, ks4, vs4, pos0 + r, n_heads, n_kv),
                     what=f"q4 row {r}")


@pytest.mark.parametrize("n,pos0,n_heads,n_kv,hd,i8", [(16, 240, 4, 4, 80, False), (17, 700, 6, 2, 96, True),
                                                       (130, 900, 4, 4, 96, False), (255, 200, 9, 3, 48, True),
                                                       (40, 3000, 8, 8, 112, False), (60, 1500, 8, 2, 16, False)])
def test_sliced_prefill_f32(gpu, n, pos0, n_heads, n_kv, hd, i8):
    # the f32 kernels: rows that end inside a wave of 16 and a tile of 128, hd / 16 fragments that do not fill a merge block
    print("[case] sliced prefill f32", n, pos0, n_heads, n_kv, hd, i8, flush=True)
    assert sliced(n, pos0, n_heads, n_kv, hd, int(i8))
    if i8:
        q, k, v, ks, vs = make_inputs_i8(9700 + n + hd, n, pos0 + n, n_heads, n_kv, hd=hd)
        kw = dict(k_scale=dev(ks, gpu, -1, n_kv), v_scale=dev(vs, gpu, -1, n_kv))
        kt, vt = dev(k, gpu, -1, n_kv, hd), dev(v, gpu, -1, n_kv, hd)
        want = reference_f64_i8(q, k, v, ks, vs, pos0, n_heads, n_kv, hd=hd)
    else:
        q, k, v = make_inputs(9700 + n + hd, n, pos0 + n, n_heads, n_kv, hd=hd)
        kw = {}
        kt, vt = (dev(x.view(np.int16), gpu, -1, n_kv, hd).view(torch.float16) for x in (k, v))
        want = reference_f64(q, k, v, pos0, n_heads, n_kv, hd=hd)
    got = gi_attn.prefill(dev(q, gpu, n, n_heads * hd), kt, vt, pos0, n_heads, n_kv, hd=hd, **kw)
    torch.cuda.synchronize()
    assert_close(got.cpu().numpy(), want, max_abs=2e-5, rel_l2=2e-5, what="sliced f32")


@pytest.mark.parametrize("fmt,hd", [("f16", 128), ("f16", 64), ("f16", 256), ("i8", 128), ("i8", 256), ("q4", 256), ("f32", 96)])
def test_chunked_prompt_with_a_short_last_chunk(gpu, fmt, hd):
    # a prompt of 1100 tokens in chunks of 512: the full chunks equal the whole prompt bit for bit; the last one, of 76
    # tokens, is cut along its keys and agrees within the bar, and equals it too where its workspace has no room
    n, chunk, n_heads, n_kv = 1100, 512, (16 if hd == 256 else 8), 2
    print("[case] short last chunk", fmt, hd, flush=True)
    gen = torch.Generator(device=gpu).manual_seed(9990 + hd)
    q = torch.randn((n, n_heads * hd), device=gpu, generator=gen)
    code = {"i8": 1, "q4": 2}.get(fmt, 0)
    if fmt == "q4":
        cache = [torch.randint(0, 256, (n, n_kv, 128), device=gpu, dtype=torch.uint8, generator=gen) for _ in range(2)]
        cache += [(0.2 + 0.15 * torch.rand((n, n_kv, 8), device=gpu, generator=gen)).half() for _ in range(2)]
        call = lambda x, pos, ws=None: gi_attn.prefill_q4(x, *cache, pos, n_heads, n_kv, workspace=ws)
    elif fmt == "i8":
        kv = [torch.randint(-127, 128, (n, n_kv, hd), device=gpu, dtype=torch.int8, generator=gen) for _ in range(2)]
        ks, vs = (0.01 + 0.01 * torch.rand((n, n_kv), device=gpu, generator=gen) for _ in range(2))
        call = lambda x, pos, ws=None: gi_attn.prefill(x, *kv, pos, n_heads, n_kv, hd=hd, k_scale=ks, v_scale=vs, workspace=ws)
    else:
        kv = [torch.randn((n, n_kv, hd), device=gpu, generator=gen).half() for _ in range(2)]
        call = lambda x, pos, ws=None: gi_attn.prefill(x, *kv, pos, n_heads, n_kv, hd=hd, f32=fmt == "f32", workspace=ws)
    whole = call(q, 0)
    for c0 in (0, 512):
        assert torch.equal(call(q[c0:c0 + chunk], c0), whole[c0:c0 + chunk]), c0
    tail = q[1024:].contiguous()
    assert gi_attn.load_library().gi_attn_prefill_scratch_bytes(1024, n - 1024, n_heads, n_kv, hd, code, 0) > 0
    got = call(tail, 1024)
    assert_close(got.cpu().numpy(), whole[1024:].cpu().numpy(), what="last chunk, cut")
    room = gi_attn.load_library().gi_attn_prefill_workspace_bytes(n, n_kv, hd, code)
    assert torch.equal(call(tail, 1024, torch.empty(room, dtype=torch.uint8, device=gpu)), whole[1024:])
