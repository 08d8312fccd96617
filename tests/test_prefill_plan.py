"""The prefill's launch rules on the host: which calls are cut along their keys, how the rest are spread over the CUs, and
the packed rows' division. The plan and the division are the library's own headers, built into a small shared object."""
import ctypes
import os
import random
import subprocess

import pytest

import gi_attn

SHIM = r"""
#include "gi_prefill_plan.h"
#include "gi_prefill_rows.h"
extern "C" {
uint32_t row_mul(long long n, int group) { return gi_row_mul(n, group); }
int row_token(int row, uint32_t mul, int group) { return gi_row_token(row, mul, group); }
void plan(int pos0, int n, int n_heads, int n_kv, int hd, int kind, size_t room, int* out) {
    const PrefillPlan p = prefill_plan(pos0, n, n_heads, n_kv, hd, (PrefillKind)kind, room);
    out[0] = p.waves, out[1] = p.group, out[2] = p.tiles, out[3] = p.nslice, out[4] = p.rows;
}
size_t part_bytes(int nslice, int waves, int kind, int n, int n_heads, int n_kv, int hd) {
    return prefill_part_bytes(nslice, waves, (PrefillKind)kind, n, n_heads, n_kv, hd);
}
}
"""
STAGED, TILE, F32 = range(3)
ANY_ROOM = (1 << 64) - 1


@pytest.fixture(scope="module")
def host(tmp_path_factory):
    d = tmp_path_factory.mktemp("plan")
    (d / "shim.cpp").write_text(SHIM)
    csrc = os.path.join(os.path.dirname(gi_attn.__file__), "csrc")
    subprocess.run(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", "-I", csrc, str(d / "shim.cpp"), "-o", str(d / "shim.so")], check=True)
    lib = ctypes.CDLL(str(d / "shim.so"))
    i, sz = ctypes.c_int, ctypes.c_size_t
    lib.row_mul.argtypes, lib.row_mul.restype = [ctypes.c_longlong, i], ctypes.c_uint32
    lib.row_token.argtypes, lib.row_token.restype = [i, ctypes.c_uint32, i], i
    lib.plan.argtypes, lib.plan.restype = [i] * 6 + [sz, ctypes.POINTER(i)], None
    lib.part_bytes.argtypes, lib.part_bytes.restype = [i] * 7, sz
    return lib


def plan(host, pos0, n, heads, kv, hd, kind, room):
    """(waves, group, key tiles a slice, slices, workgroups of a slice)"""
    out = (ctypes.c_int * 5)()
    host.plan(pos0, n, heads, kv, hd, kind, room, out)
    waves, group, tiles, nslice, rows = out
    most = (16 if kind == F32 else 32) * waves
    assert rows == most if nslice > 1 or kind == F32 else rows in (most, most // 2, most // 4, most // 8) and rows >= 32
    return waves, group, tiles, nslice, heads // group * -(-n * group // rows)


def scratch(pos0, n, n_heads=32, n_kv=8, hd=128, fmt=0, flags=0):
    return gi_attn.load_library().gi_attn_prefill_scratch_bytes(pos0, n, n_heads, n_kv, hd, fmt, flags)


def test_short_spans_and_chunks_of_short_prompts_are_not_cut():
    for n, pos0 in ((16, 0), (64, 15 * 64 - 64), (256, 3840), (512, 3584), (4096, 0), (8192, 0), (8192, 65536)):
        assert scratch(pos0, n) == 0, (n, pos0)
    assert scratch(0, 0) == 0 and scratch(-1, 16) == 0 and scratch(0, 16, 32, 5) == 0 and scratch(0, 16, hd=72) == 0
    # a few tokens over a long prefix, a chunk over more than 4096 keys; the partials of at most 1024 workgroups
    for n, pos0, heads, kv in ((16, 1008, 4, 4), (57, 6000, 32, 8), (512, 15872, 32, 4), (16, 65520, 8, 1)):
        assert 0 < scratch(pos0, n, heads, kv) <= 1024 * 256 * 130 * 4, (n, pos0)


def test_widened_keys_only_above_one_row_tile():
    lib = gi_attn.load_library()
    widen = gi_attn.GI_PREFILL_WIDEN
    for n in (16, 64, 65, 300):
        want = lib.gi_attn_prefill_workspace_bytes(n, 8, 128, 1) if 4 * n > 256 else 0
        assert scratch(0, n, fmt=1, flags=widen) == want, n
    assert scratch(0, 20, 16, 2, 256, 2, widen) == lib.gi_attn_prefill_workspace_bytes(20, 2, 256, 2)


def test_packed_row_division_is_exact(host):
    # token of packed row r: a product while n * G * G < 2^31 (else a division, multiplier 0)
    rng = random.Random(3)
    for G in list(range(1, 70)) + [96, 128, 255]:
        n = ((1 << 31) - 1) // (G * G)  # the longest batch that the product serves
        m = host.row_mul(n, G)
        assert m and host.row_mul(n + 1, G) == 0
        top = n * G - 1
        rows = {0, 1, G - 1, G, G + 1, top, top - top % G, top - top % G - 1} | {rng.randrange(top + 1) for _ in range(300)}
        for r in rows:
            if 0 <= r <= top:
                assert host.row_token(r, m, G) == r // G == host.row_token(r, 0, G), (r, G)


def test_short_prompts_have_no_fewer_workgroups_than_heads_give(host):
    # one tile of rows a head is what a launch without packed rows would have; CUs idle in all of these
    for n in (16, 32, 57, 64, 128):
        for heads, kv, hd in ((32, 8, 128), (32, 4, 128), (16, 2, 256), (8, 4, 256), (9, 3, 64), (32, 8, 64)):
            for kind in (STAGED, TILE):
                waves, group, _, nslice, wgs = plan(host, 0, n, heads, kv, hd, kind, 0)
                assert nslice == 1 and heads // kv % group == 0
                assert heads <= wgs * 1.5 and wgs <= 256, (n, heads, kv, hd, kind, wgs)
        assert plan(host, 0, n, 32, 8, 96, F32, 0)[1] == 1
    # tiles of 32 rows where those of a workgroup's waves are few (64 rows at head size 256: 16 of them)
    assert plan(host, 0, 64, 16, 2, 256, STAGED, 0)[4] == 32 and plan(host, 0, 64, 32, 8, 128, STAGED, 0)[4] == 64
    assert plan(host, 0, 250, 32, 8, 128, TILE, 0)[4] == 256


def test_tiles_widened_in_the_prefill_are_planned_as_they_are_launched(host):
    # up to 256 rows a kv head no call stages widened keys: these plans rate the larger workgroup alone, which is what the
    # kernels have (with the smaller one rated too, 57 tokens at 6100 keys had 112 workgroups on 256 CUs)
    for n, pos0, heads, kv, hd in ((57, 6100, 32, 8, 128), (32, 16000, 32, 8, 128), (40, 16000, 9, 3, 64), (64, 6100, 32, 8, 64)):
        waves, group, _, nslice, wgs = plan(host, pos0, n, heads, kv, hd, TILE, ANY_ROOM)
        assert waves == 8 and group == heads // kv and nslice * wgs > 128, (n, pos0, nslice, wgs)
    # above, and at head size 256, the slices are those of the call that stages widened keys: the same bits from both
    for n, pos0, heads, kv, hd in ((65, 6100, 32, 8, 128), (200, 3000, 32, 8, 128), (400, 16000, 9, 3, 64), (16, 6100, 16, 2, 256),
                                   (200, 16000, 16, 2, 256)):
        tile, staged = (plan(host, pos0, n, heads, kv, hd, kind, ANY_ROOM) for kind in (TILE, STAGED))
        assert tile[0] == (4 if hd == 256 else 8) and tile[1:4] == staged[1:4], (n, pos0, tile, staged)


def test_an_uncut_launch_of_equal_workgroups_fills_whole_rounds(host):
    # workgroups of nearly one length (a long prefix), a few more of the smaller size than CUs: a second round as long as the
    # first, where the larger size takes one
    # (6000 tokens of 8/8 heads at 8000 are a tie, 317 and 313 us; at 16000 the sizes take 551 and 497)
    for n, pos0, heads, kv, hd in ((1500, 3000, 32, 8, 128), (4096, 16000, 9, 3, 64), (6000, 16000, 8, 8, 128)):
        waves, _, _, nslice, wgs = plan(host, pos0, n, heads, kv, hd, STAGED, 0)
        assert waves == 8 and nslice == 1 and wgs <= 256, (n, pos0, waves, wgs)
    assert plan(host, 0, 1024, 32, 8, 128, STAGED, 0)[0] == 4  # unequal ones even out
    assert plan(host, 0, 2000, 32, 8, 128, STAGED, 0)[0] == 4  # (44 us, 53 with 8 waves)
    assert plan(host, 1000, 512, 32, 8, 128, STAGED, 0)[0] == 4  # one round of either


def test_a_plan_fits_its_room(host):
    rng = random.Random(5)
    cut = 0
    for _ in range(3000):
        kind = rng.randrange(3)
        hd = rng.choice((16, 48, 64, 80, 96, 112, 128) if kind == F32 else (64, 128, 256))
        kv = rng.choice((1, 2, 3, 4, 8, 16))
        heads = kv * rng.choice((1, 2, 3, 4, 6, 7, 8, 16))
        n, pos0 = int(2 ** rng.uniform(4, 12)), int(2 ** rng.uniform(0, 17)) - 1
        whole = plan(host, pos0, n, heads, kv, hd, kind, ANY_ROOM)
        need = host.part_bytes(whole[3], whole[0], kind, n, heads, kv, hd)
        assert need <= 1024 * (128 if hd == 256 or kind == F32 else 256) * (hd + 2) * 4  # a session's room for any call
        assert whole[3] <= 64 and whole[2] * whole[3] * 64 >= pos0 + n
        assert plan(host, pos0, n, heads, kv, hd, kind, need) == whole or whole[3] == 1
        assert plan(host, pos0, n, heads, kv, hd, kind, 0)[3] == 1
        if whole[3] > 1:
            cut += 1
            for room in (need - 1, need // 2, 4096):
                p = plan(host, pos0, n, heads, kv, hd, kind, room)
                assert host.part_bytes(p[3], p[0], kind, n, heads, kv, hd) <= room and p[2] * p[3] * 64 >= pos0 + n
                assert p[3] == 1 or p[1] == heads // kv  # (the merge takes whole groups)
    assert cut > 500
