"""What a prefill call does with the workspace that its caller brings: over the int8 cache nothing but the widened keys up to
gi_attn_prefill_workspace_bytes (outputs bit for bit as without one), and launches cut along their keys beyond that."""
import ctypes

import numpy as np
import pytest
import torch

import gi_attn
from attn_common import assert_close, make_inputs_i8

pytestmark = pytest.mark.gpu


def dev(x, gpu, *shape):
    return torch.from_numpy(np.ascontiguousarray(x)).to(gpu).view(*shape)


def merges(fn):
    """Merge launches (of sliced prefills) that fn() makes."""
    torch.cuda.synchronize()
    gi_attn.kernel_timing(True)
    gi_attn.kernel_timing_read("prefill_combine")
    fn()
    gi_attn.kernel_timing(False)
    return gi_attn.kernel_timing_read("prefill_combine")[1]


I8_SHAPES = [(16, 1008, 4, 4, 64), (57, 6100, 32, 8, 128), (20, 2000, 9, 3, 64), (100, 1500, 16, 4, 128), (40, 1500, 8, 2, 256)]


@pytest.mark.parametrize("n,pos0,n_heads,n_kv,hd", I8_SHAPES)
def test_i8_workspace_up_to_the_widened_keys_changes_no_bit(gpu, n, pos0, n_heads, n_kv, hd):
    print("[case] i8 workspace", n, pos0, n_heads, n_kv, hd, flush=True)
    lib = gi_attn.load_library()
    need = lib.gi_attn_prefill_workspace_bytes(pos0 + n, n_kv, hd, 1)
    assert lib.gi_attn_prefill_scratch_bytes(pos0, n, n_heads, n_kv, hd, 1, 0) > 0  # a call with room would be cut
    _, k, v, ks, vs = make_inputs_i8(9900 + n + hd, 1, pos0 + n, n_heads, n_kv, hd=hd)
    qkv = torch.from_numpy(np.random.default_rng(9901 + n).standard_normal((n, (n_heads + 2 * n_kv) * hd), dtype=np.float32)).to(gpu)
    kt, vt, kst, vst = dev(k, gpu, -1, n_kv, hd), dev(v, gpu, -1, n_kv, hd), dev(ks, gpu, -1, n_kv), dev(vs, gpu, -1, n_kv)
    ptrs = [t.data_ptr() for t in (kt, vt, kst, vst)]
    row = qkv.shape[1]
    scale = 1.0 / ctypes.c_float(hd ** 0.5).value
    none = torch.empty((n, n_heads * hd), device=gpu)
    gi_attn._check(lib.gi_attn_prefill_i8(gi_attn._stream(), qkv.data_ptr(), gi_attn.GI_F32, row, *ptrs, n_kv * hd, hd, n_kv, 1,
                                          none.data_ptr(), gi_attn.GI_F32, n_heads * hd, pos0, n, n_heads, n_kv, hd, scale))
    q = qkv[:, :n_heads * hd]
    for nbytes in (need, need - 16, 4096):  # widened, and too small for it
        ws = torch.empty(nbytes, dtype=torch.uint8, device=gpu)
        if nbytes == need:
            got = gi_attn.prefill(q, kt, vt, pos0, n_heads, n_kv, hd=hd, scale=scale, k_scale=kst, v_scale=vst, workspace=ws)
            assert torch.equal(got, none)
        got = gi_attn.attention(qkv, kt, vt, pos0, n_heads, n_kv, hd=hd, k_scale=kst, v_scale=vst, workspace=ws)
        assert torch.equal(got, none), nbytes
    # beyond the widened keys the partials go, and the launch is cut
    part = lib.gi_attn_prefill_scratch_bytes(pos0, n, n_heads, n_kv, hd, 1, 0)
    ws = torch.empty(need + part, dtype=torch.uint8, device=gpu)
    out = torch.empty_like(none)
    for call in (lambda: gi_attn.prefill(q, kt, vt, pos0, n_heads, n_kv, hd=hd, scale=scale, k_scale=kst, v_scale=vst, workspace=ws, out=out),
                 lambda: gi_attn.attention(qkv, kt, vt, pos0, n_heads, n_kv, hd=hd, k_scale=kst, v_scale=vst, workspace=ws, out=out),
                 lambda: gi_attn.attention(qkv, kt, vt, pos0, n_heads, n_kv, hd=hd, k_scale=kst, v_scale=vst, out=out)):
        out.zero_()
        assert merges(call) == 1
        assert_close(out.cpu().numpy(), none.cpu().numpy(), what="cut")


# (n, pos0, n_heads, n_kv, hd, f32)
ANY_SHAPES = [(57, 3000, 16, 4, 128, False), (40, 2000, 9, 3, 64, False), (40, 1500, 8, 2, 256, False), (40, 1000, 8, 2, 96, False),
              (40, 1000, 8, 2, 128, True)]


@pytest.mark.parametrize("n,pos0,n_heads,n_kv,hd,f32", ANY_SHAPES)
def test_f16_and_f32_calls_take_the_workspace_they_are_given(gpu, n, pos0, n_heads, n_kv, hd, f32):
    # enough room: the launch is cut as with a scratch of its own, the same bits, and nothing is allocated; too small for
    # any cut, misaligned or empty: it is not cut, as the entry points without a workspace
    print("[case] given workspace", n, pos0, n_heads, n_kv, hd, f32, flush=True)
    lib = gi_attn.load_library()
    part = lib.gi_attn_prefill_scratch_bytes(pos0, n, n_heads, n_kv, hd, 0, gi_attn.GI_PREFILL_F32 if f32 else 0)
    assert part > 0
    gen = torch.Generator(device=gpu).manual_seed(9950 + hd)
    qkv = torch.randn((n, (n_heads + 2 * n_kv) * hd), device=gpu, generator=gen)
    kt, vt = (torch.randn((pos0 + n, n_kv, hd), device=gpu, generator=gen).half() for _ in range(2))
    q, scale = qkv[:, :n_heads * hd], 1.0 / ctypes.c_float(hd ** 0.5).value
    out, uncut = (torch.empty((n, n_heads * hd), device=gpu) for _ in range(2))
    args = (gi_attn._stream(), qkv.data_ptr(), gi_attn.GI_F32, qkv.shape[1], kt.data_ptr(), vt.data_ptr())
    tail = (n_kv * hd, hd)
    if f32:
        gi_attn._check(lib.gi_attn_prefill_f32(*args, None, None, 0, *tail, 0, 0, uncut.data_ptr(), gi_attn.GI_F32, n_heads * hd, pos0, n,
                                               n_heads, n_kv, hd, scale))
    else:
        gi_attn._check(lib.gi_attn_prefill(*args, *tail, uncut.data_ptr(), gi_attn.GI_F32, n_heads * hd, pos0, n, n_heads, n_kv, hd, scale))
    room = torch.empty(part + 16, dtype=torch.uint8, device=gpu)
    calls = (lambda ws: gi_attn.prefill(q, kt, vt, pos0, n_heads, n_kv, hd=hd, scale=scale, out=out, f32=f32, workspace=ws),
             lambda ws: gi_attn.attention(qkv, kt, vt, pos0, n_heads, n_kv, hd=hd, out=out, no_tc=f32, workspace=ws))
    for call in calls:
        call(None)
        own = out.clone()
        assert_close(own.cpu().numpy(), uncut.cpu().numpy(), what="cut")
        out.zero_()
        torch.cuda.synchronize()
        before = torch.cuda.memory_stats()["allocation.all.allocated"]
        assert merges(lambda: call(room)) == 1
        assert torch.cuda.memory_stats()["allocation.all.allocated"] == before
        assert torch.equal(out, own)
        for ws in (room[:4096], room[8:], room[:0]):
            out.zero_()
            assert merges(lambda: call(ws)) == 0
            assert torch.equal(out, uncut)
        with pytest.raises(gi_attn.GiAttnError, match="workspace must be a CUDA tensor"):
            call(torch.empty(part, dtype=torch.uint8))


@pytest.mark.parametrize("i8", [False, True])
def test_operator_writes_rows_side_by_side_into_any_out(gpu, i8):
    # attention() takes an out of any shape with n * n_heads * hd values: flat, or with the heads apart
    n, pos0, n_heads, n_kv, hd = 20, 40, 8, 2, 128
    print("[case] operator out", i8, flush=True)
    _, k, v, ks, vs = make_inputs_i8(9990, 1, pos0 + n, n_heads, n_kv, hd=hd)
    kt, vt, kst, vst = dev(k, gpu, -1, n_kv, hd), dev(v, gpu, -1, n_kv, hd), dev(ks, gpu, -1, n_kv), dev(vs, gpu, -1, n_kv)
    if not i8:
        kt, vt, kst, vst = kt.half(), vt.half(), None, None
    gen = torch.Generator(device=gpu).manual_seed(9991)
    qkv = torch.randn((n, (n_heads + 2 * n_kv) * hd), device=gpu, generator=gen)
    want = gi_attn.attention(qkv, kt, vt, pos0, n_heads, n_kv, hd=hd, k_scale=kst, v_scale=vst)
    for shape in ((n * n_heads * hd,), (n, n_heads, hd), (1, n * n_heads * hd)):
        out = torch.empty(shape, device=gpu)
        got = gi_attn.attention(qkv, kt, vt, pos0, n_heads, n_kv, hd=hd, k_scale=kst, v_scale=vst, out=out)
        assert got is out and torch.equal(out.view(n, -1), want), shape


def test_an_expanded_workspace_is_not_used(gpu):
    # one element, 2^28 by its shape: uncut, as with an empty one
    n, pos0, n_heads, n_kv, hd = 57, 3000, 16, 4, 128
    print("[case] expanded workspace", flush=True)
    gen = torch.Generator(device=gpu).manual_seed(9995)
    q = torch.randn((n, n_heads * hd), device=gpu, generator=gen)
    kt, vt = (torch.randn((pos0 + n, n_kv, hd), device=gpu, generator=gen).half() for _ in range(2))
    want = gi_attn.prefill(q, kt, vt, pos0, n_heads, n_kv, hd=hd, workspace=torch.empty(0, dtype=torch.uint8, device=gpu))
    ws = torch.empty(1, dtype=torch.uint8, device=gpu).expand(1 << 28)
    call = lambda: gi_attn.prefill(q, kt, vt, pos0, n_heads, n_kv, hd=hd, workspace=ws)
    assert merges(call) == 0 and torch.equal(call(), want)
