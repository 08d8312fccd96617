"""The prefill's launch rules on the host: which calls are cut along their keys, and the packed rows' division."""
import random

import gi_attn


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


def test_packed_row_division_is_exact():
    # token of packed row r: the high word of 2 r * ceil(2^31 / G), used while n * G * G < 2^31
    rng = random.Random(3)
    for G in list(range(1, 70)) + [96, 128, 255]:
        m = ((1 << 31) + G - 1) // G
        top = (1 << 31) // (G * G) * G - 1  # the last row of the longest batch
        rows = {0, 1, G - 1, G, G + 1, top, top - top % G, top - top % G - 1} | {rng.randrange(top + 1) for _ in range(300)}
        for r in rows:
            if 0 <= r <= top:
                assert (2 * r * m) >> 32 == r // G, (r, G)
