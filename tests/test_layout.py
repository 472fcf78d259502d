"""The many-row layout search (host code, CPU): the same choice as the plain search over every height and split length
it states, in a host time that every layer of a batched step can pay."""

from __future__ import annotations

import ctypes
import random
import time

import dkv_hip

FAKE = ctypes.c_void_p(256)  # never dereferenced: sizes come from the host arguments


def _args(lengths, q_heads, kv_heads, dim, rank, q_len):
    cu = [0]
    for n in lengths:
        cu.append(cu[-1] + n)
    host = (ctypes.c_int32 * len(cu))(*cu)
    order = dkv_hip.Order(rank // 64, rank // 8, FAKE, FAKE, FAKE, FAKE)
    a = dkv_hip.AttendArgs()
    a.batch, a.q_len, a.layers, a.layer = len(lengths), q_len, 2, 0
    a.kv_heads, a.head_dim, a.q_heads, a.rank = kv_heads, dim, q_heads, rank
    a.key = a.value = dkv_hip.Stream(FAKE, FAKE, FAKE, order, dkv_hip.DKV_FMT_PLANES, dkv_hip.Ladder())
    a.cu_seqlens = a.positions = a.key_basis = a.value_basis = a.mean_k = a.mean_v = 256
    a.rope_cos = a.rope_sin = a.query = a.out = 256
    a.rope_rows = max(lengths) + 1
    a.cu_seqlens_host = ctypes.cast(host, ctypes.c_void_p).value
    return a, host


def _bytes(lengths, *shape) -> int:
    a, keep = _args(lengths, *shape)
    return dkv_hip.lib().dkv_attend_workspace_bytes(ctypes.byref(a))


def _searched(lengths, q_heads, kv_heads, dim, rank, q_len) -> int:
    """Workspace bytes with the height and split length of least cost over all of them."""
    rows = q_heads * q_len
    tiles = [-(-n // 256) for n in lengths]
    splits = lambda st: sum(-(-t // st) for t in tiles)  # noqa: E731
    least, mw_best, st_best = 1e300, 0, 0
    for mw, tile_us in ((1, 2.4), (2, 3.2), (4, 6.0)):
        per_split = -(-rows // (64 * mw)) * (rank // 256)
        for st in range(2, max(2, sum(tiles)) + 1):
            n = splits(st)
            cost = -(-per_split * n // 256) * (st * tile_us + 8.0) + 0.1 * 4e-6 * n * rows * rank
            if cost < least * 0.999:
                least, mw_best, st_best = cost, mw, st
    slots, n = sum(tiles) * 256 + 1024, splits(st_best)
    stats = -(-rows // 8) * 8 * sum(tiles) * 4 * 4
    blocks = rank // 64 * (slots // 64) * 4
    areas = [slots * rank * 2, slots * rank, slots * (rank // 64) * 8, 256, blocks, slots * rank * 2, blocks,
             -(-rows // (64 * mw_best)) * 64 * mw_best * slots * 2, stats, stats, n * rows * rank * 4, n * rows * 4,
             rank // 128 * len(lengths) * rows * dim * 4, len(lengths) * rows * 4 * (dim + 2) * 4]
    return sum(-(-x // 256) * 256 for x in areas)


def _fixed(lengths, q_heads, kv_heads, dim, rank, q_len) -> int:
    """Bytes of the layout by which dkv_attend_layer_noalloc takes a many-row context: no lines, one statistics entry
    per tile, rows as they are, splits of 1,024 tokens (512 where those are fewer workgroups than CUs)."""
    rows, tiles = q_heads * q_len, sum(-(-n // 256) for n in lengths)
    splits = lambda tok: sum(-(-n // tok) for n in lengths)  # noqa: E731
    n = splits(1024) if splits(1024) * (rank // 64) * -(-rows // 32) >= 256 else splits(512)
    slots = tiles * 256 + 1024
    areas = [slots * rank * 2, slots * rank, slots * (rank // 64) * 8, rows * slots * 2, rows * tiles * 4, rows * tiles * 4,
             n * rows * rank * 4, rank // 128 * len(lengths) * rows * dim * 4, len(lengths) * rows * 4 * (dim + 2) * 4]
    return sum(-(-x // 256) * 256 for x in areas)


def _random_many_rows(rng, most_tokens):
    batch = rng.choice([1, 1, 1, 2, 5, 20])
    lengths = [rng.randint(1, int(10 ** rng.uniform(0, most_tokens))) for _ in range(batch)]
    dim = rng.choice([64, 128])
    kv_heads = 256 // dim * rng.randint(1, 8)
    heads = kv_heads * rng.randint(1, 8)
    q_len = rng.randint(4 * kv_heads // heads + 1, rng.choice([8, 80, 400]))
    return lengths, (heads, kv_heads, dim, 256 * rng.randint(1, 8), q_len)


def test_noalloc_takes_contexts_by_its_own_size():
    """Refused exactly above the documented maximum (elsewhere the call goes on to look for a GPU), and every context
    it takes fits the static array."""
    rng, most = random.Random(9), dkv_hip.NOALLOC_MAX_BYTES
    near = 0
    for _ in range(3000):
        lengths, shape = _random_many_rows(rng, 4.2)
        need = _fixed(lengths, *shape)
        if need < 4096 * 256:
            continue
        near += most // 2 < need < 2 * most
        a, keep = _args(lengths, *shape)
        a.value_basis = 256
        if need > most:
            assert dkv_hip.lib().dkv_attend_layer_noalloc(ctypes.byref(a), None) == -3
            assert f"needs {need} B of scratch; the static maximum is {most} B" in dkv_hip.lib().dkv_last_error().decode()
        else:
            assert _bytes(lengths, *shape) <= 2 * most, (lengths, shape)
    assert near > 200


def test_choice_is_the_plain_search():
    rng = random.Random(4)
    for _ in range(150):
        batch = rng.choice([1, 1, 2, 5, 20])
        lengths = [rng.randint(0, int(10 ** rng.uniform(1, 4.3))) for _ in range(batch)]
        kv_heads = rng.choice([4, 8])
        shape = (kv_heads * rng.choice([5, 8, 16]), kv_heads, rng.choice([64, 128]), 256 * rng.randint(1, 8), rng.choice([1, 3, 70]))
        assert _bytes(lengths, *shape) == _searched(lengths, *shape), (lengths, shape)


def test_host_time_of_batched_layouts():
    """One query token of a model with 8 query heads per KV head: every layer of the step asks for the layout."""
    for lengths in ([16384] * 64, [137 * i + 1 for i in range(1, 65)], [131072] * 8):
        a, keep = _args(lengths, 64, 8, 128, 2048, 1)
        call = dkv_hip.lib().dkv_attend_workspace_bytes
        best = 1.0
        for _ in range(20):
            t = time.perf_counter()
            call(ctypes.byref(a))
            best = min(best, time.perf_counter() - t)
        assert best < 60e-6, (len(lengths), max(lengths), best)
