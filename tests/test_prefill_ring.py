"""The prefill kernel's LDS ring (csrc/prefill.hip), replayed on the CPU.

Its waves share four stages of 64 keys and meet at one barrier a tile; a wave
whose rows end at earlier keys than its neighbours' runs out of blocks some
tiles early (G = 1: up to four, G = 2: two, G >= 4: one). The replay lists,
between two barriers, which wave uses which stage for which tile, and checks
that nobody writes what another wave still reads and that every read finds its
tile.
"""

import numpy as np
import pytest

from hayate_amd import _native

TILE, STAGES, WAVES, ROWS = 64, 4, 8, 256


def replay(item, group, late_pv):
    """Faults of one item {seq, q0, q1, kv0, kv1, slot, q_row, cache}: (phase,
    what, wave). late_pv: each block's V is read in the next block's body, the
    last one's after the loop; otherwise in the block's own. A quarter of a stage
    is (stage, 0..1) for K blocks and 2..3 for V blocks."""
    _, q0, q1, kv0, kv1, slot, _, cache = (int(v) for v in item)
    n_tiles = -(-(kv1 - kv0) // TILE)
    last = kv1 - 1
    phases = [[] for _ in range(n_tiles + 1)]  # (wave, "r" or "w", quarter, tile)

    def quarter(block, v):
        return (block // 2 % STAGES, 2 * v + block % 2)

    for wave in range(WAVES):
        t0 = q0 + 32 * wave // group
        t1 = min(q1 - 1, q0 + (32 * wave + 31) // group)
        hi = min(cache + t1, last)
        nb = (hi - kv0) // 32 + 1 if t0 < q1 and hi >= kv0 else 0
        for t in range(n_tiles):
            p = phases[t + 1]
            if t + 2 < n_tiles:
                for block in (2 * t + 4, 2 * t + 5):
                    p += [(wave, "w", quarter(block, 0), t + 2), (wave, "w", quarter(block, 1), t + 2)]
            for j in (2 * t, 2 * t + 1):
                if j >= nb:
                    continue
                if not late_pv or j > 0:
                    v = j - 1 if late_pv else j
                    p.append((wave, "r", quarter(v, 1), v // 2))
                if j + 2 < nb:  # past the last block the values are dropped
                    p.append((wave, "r", quarter(j + 2, 0), (j + 2) // 2))
        p = phases[n_tiles]
        if nb and late_pv:
            p.append((wave, "r", quarter(nb - 1, 1), (nb - 1) // 2))
        if slot < 0:  # output rows on their way to memory
            p.append((wave, "w", ((n_tiles + wave // 4) % STAGES, wave % 4), None))
    # the prologue brings tiles 0 and 1; loads land before the barrier that ends their phase
    holds = {q: b // 2 for b in range(4) for q in (quarter(b, 0), quarter(b, 1))}
    faults = []
    for i, p in enumerate(phases):
        written = {}
        for wave, kind, q, tile in p:
            if kind == "w":
                written.setdefault(q, {}).setdefault(tile, set()).add(wave)
        for wave, kind, q, tile in p:
            if kind == "r" and holds.get(q) != tile:
                faults.append((i, "stale", wave))
            if kind == "r" and any(w - {wave} for w in written.get(q, {}).values()):
                faults.append((i, "overwritten", wave))
        for q, tiles in written.items():
            holds[q] = next(iter(tiles))
    return faults


def items(group, cache, q_len):
    plan = _native.plan_tick(np.array(q_len), np.array(cache) + np.array(q_len), 8 * group, 8, 128,
                             256, 0)
    return plan.prefill


# (group, cached tokens, chunks): a wave's last tile lies three tiles or more
# before the item's
FAR = [(1, [0], [200]), (1, [32, 32], [256, 256]), (1, [4000], [480]), (2, [48], [81]),
       (2, [16], [128]), (2, [48], [200])]


def ticks(group):
    yield from ((c, q) for g, c, q in FAR if g == group)
    rng = np.random.default_rng(group)
    for _ in range(60):
        n = int(rng.integers(1, 5))
        yield rng.integers(0, 4097, n), rng.integers(2, 513, n)


@pytest.mark.parametrize("group", [1, 2, 4, 8, 16])
def test_no_wave_overwrites_what_another_reads(group):
    for cache, q in ticks(group):
        for it in items(group, cache, q):
            assert replay(it, group, late_pv=group >= 4) == [], (cache, q, it)


@pytest.mark.parametrize("group,cache,q", FAR)
def test_the_late_order_is_not_for_these(group, cache, q):
    """Why G < 4 multiplies each block's V in the block's own body."""
    assert any(replay(it, group, late_pv=True) for it in items(group, cache, q))
