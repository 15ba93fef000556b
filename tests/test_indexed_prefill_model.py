"""CPU models of `indexed_prefill_kernel` (moespresso_amd/csrc/prefill_attn.hip), the kernel of every prefill call, and the rules
its generated code has to keep (hipcc compiles the source to gfx950 assembly; nothing runs on a GPU).

* rows: the ring rows and pool rows a workgroup asks for, tile by tile, against the reference's visit rules and the bounds of
  the tensors they address (indexed_attention_kernel.py:120-173 of the reference);
* key ranges: the ranges that a unit of a part-filled last round is cut into hold each of its tiles once;
* schedule: two tile buffers and one barrier a tile. Every wave runs the same program, so two waves' actions are ordered only
  where a barrier lies between them: an action's epoch is the number of barriers in front of it.
"""

import os
import re
import shutil

import numpy as np
import pytest

from moespresso_amd import _lib, build
from test_prefill_row_table_model import host_n_win, unit_rows

SOURCE = os.path.join(build.CSRC, "prefill_attn.hip")
TILE, LDS = 32, 80 * 1024
ROW_PITCH = 512 * 2 + 32
MAX_IDS = (LDS - 2 * TILE * ROW_PITCH - 64) // 4 // 64 * 64


def test_the_constants_are_those_of_the_kernel():
    text = open(SOURCE).read()
    for line in ("kTile = 32;", "kThreads = 256;", "kPitch = kD * 2 + 32;", "kOffIds = 2 * kTileBytes;", "kLdsBytes = 80 * 1024;",
                 "kMaxIds = (kLdsBytes - kOffIds - 64) / 4 / 64 * 64;", "kMaxRanges = 8;"):
        assert f"constexpr int {line}" in text, line
    assert 2 * TILE * ROW_PITCH + MAX_IDS * 4 + 4 <= LDS and 2 * LDS <= 160 * 1024


# ------------------------------------------------------------------------------------------------ rows

def tiles_of(t, ids, *, pos0, n_tokens, raw_cap, raw_start, window, ratio, n_pool):
    """[(base, [row or None] * 32)] of token t's tiles, as window_row and pool_row form them (base "ring" or "pool")."""
    hw = host_n_win(pos0, n_tokens, raw_cap, window)
    rows, visible, n_win = unit_rows(t, pos0=pos0, n_tokens=n_tokens, raw_cap=raw_cap, raw_start=raw_start, window=window,
                                     ratio=ratio, n_pool=n_pool, host_n_win=hw)
    stop = next((i for i, v in enumerate(ids) if v >= 0 and v >= visible), len(ids))
    wt = -(-n_win // TILE)
    out = []
    for tile in range(wt):
        slots = range(tile * TILE, (tile + 1) * TILE)
        out.append(("ring", [rows[s] if s < n_win else None for s in slots]))
    for tile in range(-(-stop // TILE)):
        slots = range(tile * TILE, (tile + 1) * TILE)
        read = [ids[g if g < MAX_IDS and g < len(ids) else 0] for g in slots]
        out.append(("pool", [i if g < stop and i >= 0 else None for g, i in zip(slots, read)]))
    return out, rows, visible, stop, wt


@pytest.mark.parametrize("seed", range(6))
def test_every_tile_row_lies_in_its_tensor_and_the_walk_is_the_references(seed):
    rng = np.random.default_rng(seed)
    for _ in range(60):
        n_tokens, raw_cap = int(rng.integers(1, 300)), int(rng.integers(1, 400))
        shape = dict(pos0=int(rng.choice([0, 1, int(rng.integers(0, 5000)), 2 ** 31 - 1 - n_tokens])), n_tokens=n_tokens,
                     raw_cap=raw_cap, raw_start=int(rng.integers(0, raw_cap)), window=int(rng.choice([0, 1, 128, 600])),
                     ratio=int(rng.choice([0, 1, 4, 128])), n_pool=int(rng.integers(1, 3000)))
        n_idx = int(rng.choice([0, 1, 31, 32, 33, 512, MAX_IDS]))
        ids = rng.integers(-2, shape["n_pool"] + 40, n_idx).tolist()
        if rng.random() < 0.5:
            ids = [i for i in sorted(ids)]
        for t in range(0, n_tokens, max(1, n_tokens // 5)):
            tiles, ring, visible, stop, wt = tiles_of(t, ids, **shape)
            want = []
            for i in ids:                                   # the walk: skip negatives, end at the first invisible id
                if i >= 0 and i >= visible:
                    break
                want += [i] if i >= 0 else []
            got_ring = [r for base, rows in tiles if base == "ring" for r in rows if r is not None]
            got_pool = [r for base, rows in tiles if base == "pool" for r in rows if r is not None]
            assert got_ring == ring and all(0 <= r < raw_cap for r in got_ring)
            assert got_pool == want and all(0 <= r < shape["n_pool"] for r in got_pool)


def test_no_token_visits_more_ring_rows_than_the_host_counts():
    """The host sizes ranges and scratch by host_n_win(); the kernel's own arithmetic stays within it, without a clamp."""
    for pos0 in (*range(9), 2 ** 31 - 8):
        for n_tokens in range(1, 6):
            for raw_cap in range(1, 14):
                for window in (0, 1, 2, 5, 9, 14):
                    most = host_n_win(pos0, n_tokens, raw_cap, window)
                    for t in range(n_tokens):
                        _, _, n_win = unit_rows(t, pos0=pos0, n_tokens=n_tokens, raw_cap=raw_cap, raw_start=0, window=window, ratio=4,
                                                n_pool=1, host_n_win=1 << 31)
                        assert n_win <= most, (pos0, n_tokens, raw_cap, window, t)


def test_division_by_reciprocal_is_division():
    """mspr_div(x, n, mspr_inverse(n)) of common.h for every x below 2^31: the high half of x * floor(2^32 / n), corrected by one."""
    rng = np.random.default_rng(2)
    text = open(os.path.join(build.CSRC, "common.h")).read()
    assert "int q = (int)__umulhi((uint32_t)x, inv);" in text and "if (x - q * n >= n) q++;" in text
    for n in [*range(2, 700), *(2 ** k + d for k in range(10, 31) for d in (-1, 0, 1)), *rng.integers(2, 2 ** 31, 300).tolist()]:
        inv = np.uint64(2 ** 32 // n)
        top = 2 ** 31 // n * n
        x = np.unique(np.clip(np.concatenate([rng.integers(0, 2 ** 31, 200), [0, 1, n - 1, n, n + 1, top - 1, top, 2 ** 31 - 1]]), 0, 2 ** 31 - 1))
        x = x.astype(np.uint64)
        q = x * inv >> np.uint64(32)
        q += (x - q * np.uint64(n) >= np.uint64(n)).astype(np.uint64)
        assert np.array_equal(q, x // np.uint64(n)), n


# ------------------------------------------------------------------------------------------------ key ranges

def test_key_ranges_of_a_cut_unit_hold_every_tile_once():
    rng = np.random.default_rng(1)
    for _ in range(4000):
        wt, n_idx = int(rng.integers(0, 20)), int(rng.integers(0, MAX_IDS + 1))
        ranges = int(rng.integers(2, 9))
        stop = int(rng.integers(0, n_idx + 1))
        total = wt + -(-stop // TILE)
        share = (wt + -(-n_idx // TILE) + ranges - 1) // ranges
        seen = []
        for r in range(ranges):
            begin = r * share
            end = min(total, begin + share) if total - begin > share else total
            seen += range(begin, end)
            if begin < wt:                                  # its first copy is issued before the ids are known: it is awaited
                assert end > begin
        assert seen == list(range(total))


def test_a_last_round_is_cut_only_where_the_partials_pay():
    """Scratch is asked for the partials of cut units alone: 64 heads, a window of 128."""
    if not _lib.library_available():
        pytest.skip("the library is not built")

    def parts(tokens, n_idx, heads=64):
        n = _lib.lib().mspr_indexed_mixed_attention_prefill_workspace_bytes(1, 1, heads, tokens, 128, n_idx)
        assert n % (64 * 514 * 4) == 0
        return n // (64 * 514 * 4)

    for n_idx in (0, 64, 127):
        assert all(parts(t, n_idx) == 0 for t in range(1, 600, 7))
    assert parts(8, 128) == 16 and parts(24, 128) == 0 and parts(64, 128) == 0     # 24: 16.9 us whole, 18.0 in two ranges
    assert parts(24, 256) == 96 and parts(48, 256) == 0
    assert parts(1, 512) == 8 and parts(64, 512) == 192
    assert parts(80, 512) == 240 and parts(85, 512) == 255 and parts(86, 512) == 0  # in two ranges 80 take longer than whole
    assert parts(512, 512) == 0 and parts(512 + 64, 512) == 192 and parts(512 + 48, 128) == 0
    assert all(parts(t, n) <= 256 for t in range(1, 1100, 3) for n in (128, 256, 512, 1024, 3000))
    assert parts(3, 512, heads=72) == parts(6, 512)


# ------------------------------------------------------------------------------------------------ schedule

def program(t_begin, n_tiles, wt, barrier=True, copy_behind_barrier=True):
    """(epoch, action, tile or None) of one wave in program order."""
    events, epoch = [], 0
    if t_begin < wt:
        events.append((epoch, "copy", t_begin))
    epoch += 1                                              # __syncthreads: the stop position is set
    events.append((epoch, "ids_write", None))
    epoch += 1                                              # __syncthreads
    events.append((epoch, "ids_read", None))
    if wt <= t_begin < n_tiles:
        events.append((epoch, "copy", t_begin))
    for tile in range(t_begin, n_tiles):
        if not copy_behind_barrier and tile + 1 < n_tiles:
            events.append((epoch, "copy", tile + 1))
        events.append((epoch, "await_all", tile))           # s_waitcnt vmcnt(0) lgkmcnt(0)
        epoch += barrier
        if copy_behind_barrier and tile + 1 < n_tiles:
            events += [(epoch, "ids_read", None), (epoch, "copy", tile + 1)]
        events.append((epoch, "read", tile))
    epoch += 1                                              # __syncthreads in front of the output staging
    events.append((epoch, "stage", None))
    return events


def check(events):
    at = {}
    for i, (epoch, kind, tile) in enumerate(events):
        at.setdefault((kind, tile), (epoch, i))
    tiles = sorted(t for k, t in at if k == "read")
    waits = [i for i, e in enumerate(events) if e[1] == "await_all"]
    for t in tiles:
        (copied, i_copy), (read, _) = at["copy", t], at["read", t]
        i_wait = next(i for i in waits if i > i_copy)       # the first full wait behind the copies of the tile
        assert events[i_wait][0] < read, "a tile is read before every wave has waited for its rows"
        if ("read", t - 2) in at:
            assert at["read", t - 2][0] < copied, "a buffer is overwritten while it may still be read"
    assert sum(k == "copy" for _, k, _ in events) == len(tiles), "every copy is of a tile that is awaited"
    assert at["ids_write", None][0] < min(e for e, k, _ in events if k == "ids_read")
    assert all(e < at["stage", None][0] for e, k, _ in events if k == "read")


def test_two_buffers_and_one_barrier_a_tile_keep_copies_and_reads_apart():
    for wt in (0, 1, 4):
        for n_tiles in range(wt, wt + 9):
            for t_begin in range(0, n_tiles + 1):
                check(program(t_begin, n_tiles, wt))


def test_the_model_sees_a_missing_barrier_and_a_copy_in_front_of_it():
    with pytest.raises(AssertionError):
        check(program(0, 6, 2, barrier=False))
    with pytest.raises(AssertionError, match="overwritten"):
        check(program(0, 6, 2, copy_behind_barrier=False))


# ------------------------------------------------------------------------------------------------ generated code

@pytest.fixture(scope="module")
def assembly():
    if not (os.path.exists(build.HIPCC) or shutil.which(build.HIPCC)):
        pytest.skip("hipcc not installed")
    return build.device_assembly(SOURCE)


def test_two_workgroups_fit_a_cu_without_scratch(assembly):
    kernels = {k: v for k, v in build.kernel_resources(SOURCE, assembly).items() if "indexed_prefill_kernel" in k}
    assert len(kernels) == 4, sorted(kernels)               # query type x cut
    for name, res in kernels.items():
        assert res["scratch_bytes"] == 0 and res["vgpr_spills"] == 0 and res["sgpr_spills"] == 0, (name, res)
        assert res["vgprs"] <= 256, (name, res)             # eight waves on the four SIMDs of a CU


def instructions(lines):
    code = [l.split(";")[0].strip() for l in lines]
    return [l for l in code if l and not l.startswith(".") and not l.endswith(":")]


def tile_loop(code):
    """(start, end) of the tile loop: from the barrier behind the full wait to the branch behind the 64 matrix instructions."""
    first = next(i for i, l in enumerate(code) if "v_mfma" in l)
    start = max(i for i in range(first) if code[i] == "s_barrier")
    assert code[start - 1] == "s_waitcnt vmcnt(0) lgkmcnt(0)", code[start - 1]
    end = next(i for i in range(start, len(code)) if re.match(r"s_c?branch", code[i]) and
               sum("v_mfma" in l for l in code[start:i]) == 64)
    return start, end


def memory_operations(code):
    return [l for l in code if re.match(r"(global|flat|buffer|scratch)_", l)]


def test_copies_and_waits_of_the_tile_loop_are_as_written(assembly):
    bodies = {k: v for k, v in build.kernel_bodies(assembly).items() if "indexed_prefill_kernel" in k}
    assert len(bodies) == 4
    for name, lines in bodies.items():
        assert build.inline_asm_register_loads(lines) == [], name
        code = instructions(lines)
        # the first tile's rows from the ring, from the pool, and the next tile's: eight rows a wave each
        assert sum("global_load_lds_dwordx4" in l for l in code) == 24, name
        # the loop's only vector-memory operations are the next tile's copies, so its full wait is for nothing else
        start, end = tile_loop(code)
        ops = memory_operations(code[start:end])
        assert len(ops) == 8 and all("global_load_lds_dwordx4" in l for l in ops), (name, ops)
        planted = code[:start + 1] + ["global_load_dwordx4 v[0:3], v4, s[0:1]"] + code[start + 1:]
        start, end = tile_loop(planted)
        assert len(memory_operations(planted[start:end])) == 9
