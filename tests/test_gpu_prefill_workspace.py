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
