"""Which way a call reaches the device (fa_sched_launch, the rule the launch itself asks), on the host."""
import ctypes
import os
import subprocess

import pytest

CUS = 256
REPO = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def launch(fa, B, H, Hk, S, Skv, D, causal=True, wl=-1, splits=1, sched=0, cus=CUS, strides=None):
    """(schedule, decoding kernel, streaming hint)"""
    p = fa.make_params(B, H, S, D, 0x1000, 0x2000, 0x3000, 0x4000, causal=causal, window_left=wl, n_kv_heads=0 if Hk == H else Hk,
                       S_kv=0 if Skv == S else Skv, split_num=splits, workspace_ptr=0x5000, workspace_bytes=1 << 62, sched=sched,
                       **(strides or {}))
    dec, nt = ctypes.c_int(-1), ctypes.c_int(-1)
    st = fa.lib().fa_sched_launch(ctypes.byref(p), cus, ctypes.byref(dec), ctypes.byref(nt))
    return st, dec.value, nt.value


def test_schedules_of_the_tile_kernels(fa):
    """At most one item per resident workgroup, fewer than eight, more; a named schedule; refusals."""
    assert launch(fa, 1, 4, 4, 512, 512, 64)[:2] == (fa.FA_SCHED_DISPATCH, 0)
    assert launch(fa, 4, 16, 16, 2048, 2048, 64)[:2] == (fa.FA_SCHED_PERSISTENT, 0)
    assert launch(fa, 2, 32, 32, 8192, 8192, 128)[:2] == (fa.FA_SCHED_QUEUE, 0)
    assert launch(fa, 2, 32, 32, 8192, 8192, 128, causal=False)[:2] == (fa.FA_SCHED_PERSISTENT, 0)
    assert launch(fa, 1, 40, 40, 512, 512, 64, sched=fa.FA_SCHED_QUEUE)[0] == fa.FA_SCHED_QUEUE
    assert launch(fa, 1, 4, 3, 512, 512, 64)[0] == fa.FA_ERR_LAYOUT


def small(fa, B, H, S, Skv, D, causal=True, wl=-1, wr=-1, splits=1, sched=0, cus=CUS, Hk=None, dropout=0.0, exact=False, dtype=0):
    """(waves of the kernel of 32-row blocks, parts of the first rows)"""
    p = fa.make_params(B, H, S, D, 0x1000, 0x2000, 0x3000, 0x4000, causal=causal, window_left=wl, window_right=wr, n_kv_heads=Hk or 0, sched=sched,
                       S_kv=0 if Skv == S else Skv, split_num=splits, workspace_ptr=0x5000, workspace_bytes=1 << 62, dropout_prob=dropout,
                       exact_first_rows=exact, dtype=dtype)
    parts = ctypes.c_int(-1)
    waves = fa.lib().fa_sched_small(ctypes.byref(p), cus, ctypes.byref(parts))
    if waves > 0:
        assert fa.lib().fa_sched_launch(ctypes.byref(p), cus, None, None) == fa.FA_SCHED_DISPATCH
    return waves, parts.value


def test_line_between_32_row_blocks_and_the_tile_kernels(fa):
    """Two blocks to a compute unit, four where a causal walk of 2048 queries and more is uneven; key splits, dropout, one and two key
    tiles on most units; whatever schedule is named, on other devices too."""
    for D in (64, 128):
        assert [small(fa, 1, h, 320, 320, D, causal=False)[0] for h in (1, 51, 52)] == [4, 4, 0]                  # 510 and 520 blocks
        assert [small(fa, 1, h, 500, 500, D, wl=100, exact=True)[0] for h in (32, 33)] == [4, 0]                   # 512 and 528
        assert [small(fa, 1, h, 2048, 2048, D, exact=True)[0] for h in (4, 8, 16, 17)] == [8, 4, 4, 0]             # 256, 512, 1024 and 1088
        assert [small(fa, 1, h, 2048, 2048, D, causal=False)[0] for h in (8, 9)] == [4, 0]
        assert [small(fa, 1, h, 2048, 2048, D, wl=2000, exact=True)[0] for h in (8, 9)] == [4, 0]
        assert [small(fa, 1, h, 128, 128, D, causal=False)[0] for h in (64, 65)] == [4, 0] and small(fa, 1, 100, 129, 129, D, causal=False)[0] == 4
        assert [small(fa, 1, h, 64, 64, D, causal=False)[0] for h in (128, 129)] == [4, 0] and small(fa, 1, 256, 64, 65, D, causal=False)[0] == 4
        assert [small(fa, 1, 100, s, 64, D, causal=False)[0] for s in (96, 97)] == [0, 0 if D == 128 else 4]
        assert small(fa, 1, 200, 64, 64, D, causal=False, wl=40)[0] == 4 and small(fa, 1, 200, 64, 64, D, causal=False, wl=64, wr=64)[0] == 0
        assert small(fa, 1, 4, 256, 2000, D, splits=2)[0] == 0 and small(fa, 1, 4, 256, 256, D, dropout=0.1)[0] == 0
        assert [small(fa, 1, 8, 256, 256, D, sched=n)[0] for n in range(4)] == [4] * 4
        assert [small(fa, 1, 16, 320, 320, D, causal=False, cus=c)[0] for c in (64, 80)] == [0, 4]
        # eight waves: at most a block to a compute unit, from 24 key tiles (64 keys each, 32 at head dimension 128) on
        n = 24 * (64 if D == 64 else 32)
        assert small(fa, 1, 4, 64, n - 1, D, causal=False)[0] == 8 and small(fa, 1, 4, 64, n - n // 24, D, causal=False)[0] == 4
        assert small(fa, 1, 4, 200, 5000, D, wl=n)[0] == 8 and small(fa, 1, 4, 200, 5000, D, wl=n // 2)[0] == 4
        assert small(fa, 1, 4, 1, 1000, D)[0] == 0 and small(fa, 1, 4, 8, 4, D, causal=False)[0] == 4              # (one is the decoding kernel's)
    assert small(fa, 1, 4, 256, 256, 96)[0] == fa.FA_ERR_HEAD_DIM


def test_parts_of_the_first_rows(fa):
    """Four per head beside 32-row blocks where a quarter of the slots more holds them (head dimension 128: eight, or where all are
    resident; 64 in bf16, two 128-row blocks: where those that have rows are), else the tile kernels; these in as many as fit into
    twice the slots (head dimension 64: 7/4); none where there are none."""
    assert [small(fa, 1, h, 256, 256, 64) for h in (40, 41, 53, 54)] == [(4, 4), (4, 4), (4, 4), (0, 8)]
    assert [small(fa, 1, h, 256, 256, 128) for h in (40, 41, 42, 43)] == [(4, 4), (4, 4), (4, 4), (0, 8)]
    assert [small(fa, 1, h, 256, 256, 64, dtype=1) for h in (42, 43)] == [(4, 4), (0, 8)] and small(fa, 1, 53, 257, 257, 64, dtype=1)[0] == 0
    assert [small(fa, 1, 60, s, k, 64, dtype=1)[0] for s, k in ((128, 129), (129, 129), (192, 192), (192, 208), (192, 207))] == [4, 0, 0, 4, 0]
    assert small(fa, 1, 44, 257, 257, 64, dtype=1) == (4, 4)
    assert [small(fa, 1, h, 256, 256, 128)[1] for h in (100, 180, 256, 257)] == [8, 2, 2, 0]
    assert small(fa, 1, 8, 2048, 2048, 64) == (4, 4) and small(fa, 1, 16, 2048, 2048, 64) == (4, 4) and small(fa, 1, 16, 4096, 4096, 64) == (0, 8)
    assert small(fa, 1, 8, 256, 256, 64, exact=True) == (4, 0) and small(fa, 1, 8, 256, 288, 64) == (4, 0) and small(fa, 1, 8, 256, 287, 64) == (4, 4)
    assert small(fa, 1, 8, 256, 256, 64, causal=False) == (4, 0) and small(fa, 1, 8, 256, 256, 64, causal=False, wr=0) == (4, 4)
    assert small(fa, 1, 8, 256, 200, 64) == (4, 0) and small(fa, 1, 8, 10, 20, 64, Hk=1) == (4, 0)                 # (a group's rows in one block)


@pytest.mark.parametrize("sched", [0, 1, 2, 3])
def test_decoding_takes_no_work_queue(fa, sched):
    """Causal decoding with as many items as would make the tile kernels balance through a queue, and with a queue asked for."""
    assert launch(fa, 64, 32, 32, 1, 2048, 128, splits=2, sched=sched)[:2] == (fa.FA_SCHED_DISPATCH, 1)
    assert launch(fa, 512, 16, 16, 1, 2048, 128, sched=sched)[:2] == (fa.FA_SCHED_DISPATCH, 1)


def test_decoding_grid_stays_below_2_to_the_32_threads(fa):
    """One 256-thread workgroup per K/V head and split: from 2^24 of them on the tile kernels take the call, and "auto"
    never splits a decoding call beyond that."""
    heads = 1 << 23
    assert launch(fa, heads // 8, 8, 8, 1, 1, 64, causal=False)[1] == 1
    assert launch(fa, heads // 8, 8, 8, 1, 512, 64, splits=2)[:2] == (fa.FA_SCHED_QUEUE, 0)
    assert launch(fa, heads // 8 - 1, 8, 8, 1, 512, 64, splits=2)[1] == 1
    assert launch(fa, heads // 4, 8, 8, 1, 1, 64, causal=False)[:2] == (fa.FA_SCHED_PERSISTENT, 0)
    for b in (heads // 8, heads // 24, heads // 9):
        p = fa.make_params(b, 8, 1, 64, causal=True, S_kv=4096)
        n = fa.lib().fa_fwd_auto_splits(ctypes.byref(p))
        assert n >= 1 and launch(fa, b, 8, 8, 1, 4096, 64, splits=n)[1] == 1


def test_short_keys_and_many_heads_take_the_tile_kernels(fa):
    """Head dimension 128, 17 to 32 rows, at most 192 keys, 1024 K/V heads and more, no mask or a packed block."""
    for S, Skv in ((17, 17), (32, 64), (32, 192), (20, 129)):
        assert launch(fa, 64, 16, 16, S, Skv, 128, causal=False)[1] == 0
    assert launch(fa, 128, 64, 8, 4, 104, 128)[1] == 0 and launch(fa, 128, 64, 8, 4, 104, 128, causal=False)[1] == 0
    assert launch(fa, 128, 64, 8, 4, 104, 128, wl=50)[1] == 0
    for args in ((64, 16, 16, 16, 64, 128), (64, 16, 16, 32, 193, 128), (64, 16, 16, 32, 64, 64), (63, 16, 16, 32, 64, 128)):
        assert launch(fa, *args, causal=False)[1] == 1
    assert launch(fa, 64, 16, 16, 32, 128, 128)[1] == 1
    p = fa.make_params(64, 16, 32, 128, causal=False, S_kv=64)
    assert fa.lib().fa_fwd_auto_splits(ctypes.byref(p)) == 1


def test_streaming_hint_counts_the_keys_that_are_read(fa):
    """More than 128 MB of K and V, behind a left window only its keys: B16, 8 K/V heads, D 128 read 64 KB per key."""
    def hint(Skv, wl):
        return launch(fa, 16, 32, 8, 2, Skv, 128, wl=wl, splits=4)[1:]
    assert hint(1953, -1) == (1, 0) and hint(1954, -1) == (1, 1)
    for Skv in (8192, 200000):
        assert hint(Skv, 128) == (1, 0) and hint(Skv, 1951) == (1, 0) and hint(Skv, 1952) == (1, 1) and hint(Skv, -1) == (1, 1)


def test_grid_of_the_merge_of_key_splits(tmp_path):
    """tests/c/check_combine_grid.c: every row covered, fewer than 2^32 threads."""
    exe = str(tmp_path / "check_combine_grid")
    subprocess.run(["gcc", "-O2", "-Wall", "-Wextra", "-I", os.path.join(REPO, "flash-attn-rtx5060_amd", "csrc"),
                    os.path.join(REPO, "tests", "c", "check_combine_grid.c"), "-o", exe], check=True)
    out = subprocess.run([exe], stdout=subprocess.PIPE, text=True)
    assert out.returncode == 0, out.stdout
